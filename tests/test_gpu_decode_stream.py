"""Decode steps on a stream that does not wait for the null stream (GPU).

A step's uniforms go up, and its tokens and row states come back, by copies on
the caller's stream through one pinned buffer: each step is right only because
copy, launches and copy are on that stream.  Several steps of both entry points
run in lockstep with the oracle's loop, with a row that ends, one at its limit
and one that fails, and every copy is on the stream that the caller gave.
"""
import numpy as np
import pytest

from oracle import oracle as o
from promptboot_amd import hip
from promptboot_amd import sampler as s
from promptboot_amd import workloads
from tests.test_gpu_decode import stand_in_logits

pytestmark = pytest.mark.gpu

V = s.VOCAB
STEPS = 8
PROMPT_LENS = [30, 5, 300, 17, 64, 9]
LIMITS = [20, 3, 20, 20, 20, 20]


@pytest.mark.parametrize("head", [None, "q4_0", "q8_0"])
def test_decode_steps_on_a_non_blocking_stream(monkeypatch, head):
    import torch

    rng = np.random.default_rng(3)
    prompts = [workloads.zipf_ids(rng, n) for n in PROMPT_LENS]
    prompts[5] = np.append(prompts[5], np.uint32(V + 3))  # a bad id: the first step fails, no draw
    seeds = [11, 12, 13, 14, 15, 16]
    rows = len(prompts)
    oracle_rows = [o.DecodeRow(p, sd, lim) for p, sd, lim in zip(prompts, seeds, LIMITS)]
    smp = s.BatchSampler(0)
    dec = s.DecodeBatch(prompts, seeds, LIMITS, sampler=smp)
    stream = torch.cuda.Stream()
    cols = 160
    if head is not None:
        q8 = head == "q8_0"
        blocks = rng.integers(0, 256, (V, cols // 32, 34 if q8 else 18), dtype=np.uint8)
        scale = rng.uniform(0.001, 0.01, (V, cols // 32)).astype(np.float16).view(np.uint16)
        blocks[:, :, 0], blocks[:, :, 1] = scale & 0xFF, scale >> 8
        packed = smp.pack_lmhead(torch.from_numpy(blocks.reshape(-1)).to("cuda:0"), q8=q8, cols=cols)
        torch.cuda.synchronize()
    used = []
    copy_async = hip.copy_async

    def recorded(dst, src, nbytes, kind, stream=None):
        used.append((kind, hip.stream_handle(stream)))
        copy_async(dst, src, nbytes, kind, stream)

    monkeypatch.setattr(hip, "copy_async", recorded)
    try:
        for step in range(STEPS):
            if head is None:
                given = np.stack([stand_in_logits(r, step, d.working[-1], 4 if r == 2 else None)
                                  for r, d in enumerate(oracle_rows)])
                if step == 3:
                    given[3, 4321] = 0x7FC00000  # row 3 fails here
                logits = given
            else:
                given = np.stack([np.random.default_rng([r, step, d.working[-1]]).normal(0, 1, cols)
                                  for r, d in enumerate(oracle_rows)]).astype(np.float32).view(np.uint32)
                if step == 3:
                    given[3] = 0x7F800000  # infinite scales: row 3 fails
                logits = o.lmhead_logits(given.view(np.float32), blocks.reshape(-1), V, cols, threads=8, q8=q8)
            want = [d.step(logits[r]) for r, d in enumerate(oracle_rows)]
            used.clear()
            with torch.cuda.stream(stream):
                x = torch.from_numpy(given.view(np.int32)).to("cuda:0")
                got = dec.step(x, stream=stream) if head is None else \
                    dec.lmhead_step(packed, x, stream=stream, q8=q8)
            assert got.tolist() == [s.NO_TOKEN if t is None else t for t in want], step
            assert used == [(hip.H2D, stream.cuda_stream), (hip.D2H, stream.cuda_stream)]
        for r, d in enumerate(oracle_rows):
            assert dec.contexts()[r].tolist() == d.working, r
            st = dec.sampling_states()[r]
            assert (st.state(), st.draws()) == (d.state.state(), d.state.draws()), r
        reasons = [d.reason for d in oracle_rows]
        assert reasons[1] == "LIMIT" and reasons[3] == "ERROR" and reasons[5] == "ERROR"
        assert head is not None or reasons[2] == "EOS"
    finally:
        dec.close()
        smp.close()
    assert rows == len(dec.row_state_host)
