"""Both LM heads at hidden widths other than the model's 896 (GPU).

The GEMMs' block loops treat the first blocks and the last ones apart: the
first block starts the running totals, loads run one or two blocks ahead
by kernel and format, and an odd or short block count ends outside the loop.  The
model's width (28 blocks) exercises none of the short or odd cases, so each
head runs here at 1, 2, 3, 5 and 29 blocks, through the narrow kernel with
its own quantisation (1 and 3 rows), the narrow kernel after lm_quant_kernel
(9 rows) and the wide kernel (66 rows).  Logits must be bit-identical to the
oracle's restatement of inference_q4_matvec_rows_prepared /
inference_q8_matvec_rows_prepared (fp32_sse2.rs:1217-1248, 1251-1280), and the
draws identical to the oracle sampler's on those logits.  At the odd widths
one Q4_0 tile carries an infinite weight scale (the subtract-then-multiply
epilogue); every row then ends in the same error record as the oracle's.
"""
import numpy as np
import pytest

from oracle import oracle as o
from promptboot_amd import sampler as s
from tests.conftest import to_dev

pytestmark = pytest.mark.gpu

V = s.VOCAB
WIDTHS = [32, 64, 96, 160, 928]
ROWS = [1, 3, 9, 66]


@pytest.fixture(scope="module")
def smp():
    b = s.BatchSampler(0)
    yield b
    b.close()


def make_head(cols: int, q8: bool, seed: int) -> np.ndarray:
    """A random head in promptboot's layout (vocab rows of 18- or 34-byte
    blocks with an fp16 scale first); a Q4_0 head of an odd block count gets
    one +inf scale in tile 7."""
    rng = np.random.default_rng(seed)
    blocks = cols // 32
    width = 34 if q8 else 18
    h = rng.integers(0, 256, (V, blocks, width), dtype=np.uint8)
    lo, hi = (0.0005, 0.004) if q8 else (0.001, 0.02)
    sc = rng.uniform(lo, hi, (V, blocks)).astype(np.float16).view(np.uint16)
    if not q8 and blocks % 2 == 1 and blocks > 1:
        sc[64 * 7 + 5, blocks - 1] = 0x7C00
    h[:, :, 0] = sc & 0xFF
    h[:, :, 1] = sc >> 8
    return h.reshape(-1)


@pytest.mark.parametrize("q8", [False, True], ids=["q4_0", "q8_0"])
@pytest.mark.parametrize("cols", WIDTHS)
def test_logits_and_draws_at_each_width(smp, q8, cols):
    import torch

    head = make_head(cols, q8, seed=cols + (1000 if q8 else 0))
    packed = smp.pack_lmhead(torch.from_numpy(head).to("cuda:0"), q8=q8, cols=cols)
    rng = np.random.default_rng(cols)
    for rows in ROWS:
        hidden = rng.standard_normal((rows, cols)).astype(np.float32)
        r24 = (np.arange(rows, dtype=np.uint32) * 7919 + 3) & 0xFFFFFF
        token = torch.empty(rows, dtype=torch.int32, device="cuda:0")
        logits = torch.empty((rows, V), dtype=torch.int32, device="cuda:0")
        smp.lmhead_sample(packed, to_dev(hidden), to_dev(r24), token=token, logits=logits,
                          cols=cols, q8=q8)
        torch.cuda.synchronize()
        glog = logits.cpu().numpy().view(np.uint32)
        rlog = o.lmhead_logits(hidden, head, V, cols, threads=16, q8=q8)
        gnan = np.isnan(glog.view(np.float32))
        rnan = np.isnan(rlog.view(np.float32))
        assert (gnan == rnan).all(), (cols, rows)
        bad = np.argwhere((glog != rlog) & ~rnan)
        assert bad.size == 0, (cols, rows, bad[:5])
        rtok, _, _, _ = o.sample_batch(rlog, np.zeros((rows, 1), np.uint32),
                                       np.zeros(rows, np.uint32), r24, threads=4)
        gtok = token.cpu().numpy().view(np.uint32)
        assert (gtok == rtok).all(), (cols, rows)


@pytest.mark.parametrize("q8", [False, True], ids=["q4_0", "q8_0"])
@pytest.mark.parametrize("cols", [32, 96, 128])
def test_narrow_head_either_side_of_every_row_count_it_branches_on(smp, q8, cols):
    """One row to 65: the narrow kernel keeps 1, 2, 4, 8, 12 or 16 result
    registers by the rows, in one row group or two, and 65 rows take the wide
    kernel.  Odd block counts carry an infinite scale in one Q4_0 tile, which
    is computed again.  Every value is defined bit for bit, so it must agree."""
    import torch

    head = make_head(cols, q8, seed=cols + (2000 if q8 else 0))
    packed = smp.pack_lmhead(torch.from_numpy(head).to("cuda:0"), q8=q8, cols=cols)
    rng = np.random.default_rng(cols + 7)
    hidden = rng.standard_normal((65, cols)).astype(np.float32)
    rlog = o.lmhead_logits(hidden, head, V, cols, threads=16, q8=q8)
    rnan = np.isnan(rlog.view(np.float32))
    for rows in (1, 2, 3, 4, 5, 8, 9, 16, 17, 24, 25, 32, 33, 64, 65):
        r24 = (np.arange(rows, dtype=np.uint32) * 7919 + 3) & 0xFFFFFF
        token = torch.empty(rows, dtype=torch.int32, device="cuda:0")
        logits = torch.full((rows + 1, V), -1, dtype=torch.int32, device="cuda:0")
        smp.lmhead_sample(packed, to_dev(hidden[:rows]), to_dev(r24), token=token,
                          logits=logits, cols=cols, q8=q8)
        torch.cuda.synchronize()
        glog = logits.cpu().numpy().view(np.uint32)
        assert (glog[rows] == 0xFFFFFFFF).all(), (cols, rows)  # nothing past the last row
        gnan = np.isnan(glog[:rows].view(np.float32))
        assert (gnan == rnan[:rows]).all(), (cols, rows)
        bad = np.argwhere((glog[:rows] != rlog[:rows]) & ~rnan[:rows])
        assert bad.size == 0, (cols, rows, bad[:5])
        rtok, _, _, _ = o.sample_batch(rlog[:rows], np.zeros((rows, 1), np.uint32),
                                       np.zeros(rows, np.uint32), r24, threads=4)
        assert (token.cpu().numpy().view(np.uint32) == rtok).all(), (cols, rows)


@pytest.mark.parametrize("q8", [False, True], ids=["q4_0", "q8_0"])
@pytest.mark.parametrize("rows", [33, 40, 47, 48, 49])
def test_two_row_groups_of_24_rows(smp, q8, rows):
    """33 to 48 rows take two groups of 24 rows, 49 two of 32: logits and draws
    of every row, the first group's last rows and the second's first among
    them, at an odd number of blocks.  Defined bit for bit, so they must agree."""
    import torch

    cols = 160
    head = make_head(cols, q8, seed=rows + (2000 if q8 else 0))
    packed = smp.pack_lmhead(torch.from_numpy(head).to("cuda:0"), q8=q8, cols=cols)
    hidden = np.random.default_rng(rows).standard_normal((rows, cols)).astype(np.float32)
    rlog = o.lmhead_logits(hidden, head, V, cols, threads=16, q8=q8)
    rnan = np.isnan(rlog.view(np.float32))
    r24 = (np.arange(rows, dtype=np.uint32) * 104729 + 11) & 0xFFFFFF
    token = torch.empty(rows, dtype=torch.int32, device="cuda:0")
    logits = torch.full((rows + 1, V), -1, dtype=torch.int32, device="cuda:0")
    smp.lmhead_sample(packed, to_dev(hidden), to_dev(r24), token=token, logits=logits, cols=cols, q8=q8)
    torch.cuda.synchronize()
    glog = logits.cpu().numpy().view(np.uint32)
    assert (glog[rows] == 0xFFFFFFFF).all()  # nothing past the last row
    assert (np.isnan(glog[:rows].view(np.float32)) == rnan).all()
    assert ((glog[:rows] == rlog) | rnan).all()
    rtok, _, _, _ = o.sample_batch(rlog, np.zeros((rows, 1), np.uint32), np.zeros(rows, np.uint32), r24,
                                   threads=4)
    assert (token.cpu().numpy().view(np.uint32) == rtok).all()


@pytest.mark.parametrize("q8", [False, True], ids=["q4_0", "q8_0"])
@pytest.mark.parametrize("rows", [3, 9, 10, 11, 17, 18, 19, 25, 26, 27, 33, 41, 49, 63])
def test_padding_rows_store_nothing(smp, q8, rows):
    """A row group's padding rows are computed with the real ones and must
    leave the 32 rows after the last real one alone.  At 9, 10, 17, 18, 25 and
    26 rows some result registers hold rows of which the first lies past the
    whole batch."""
    import torch

    cols = 64
    head = make_head(cols, q8, seed=rows + (2000 if q8 else 0))
    packed = smp.pack_lmhead(torch.from_numpy(head).to("cuda:0"), q8=q8, cols=cols)
    hidden = np.random.default_rng(rows + 50).standard_normal((rows, cols)).astype(np.float32)
    r24 = (np.arange(rows, dtype=np.uint32) * 7919 + 3) & 0xFFFFFF
    token = torch.empty(rows, dtype=torch.int32, device="cuda:0")
    logits = torch.full((rows + 32, V), -1, dtype=torch.int32, device="cuda:0")
    smp.lmhead_sample(packed, to_dev(hidden), to_dev(r24), token=token, logits=logits[:rows], cols=cols, q8=q8)
    torch.cuda.synchronize()
    got = logits.cpu().numpy().view(np.uint32)
    assert (got[rows:] == 0xFFFFFFFF).all()
    assert (got[:rows] == o.lmhead_logits(hidden, head, V, cols, threads=16, q8=q8)).all()
