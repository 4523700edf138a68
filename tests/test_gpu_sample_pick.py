"""Every draw of the device's sampler against sample_token (sampler.cpp:9-79) on the logits it
drew from (GPU).

The logits are the call's own dump, so the pick is a function of them, the channel's history
and the call's xoshiro stream alone: it has to be the oracle's, whatever number of candidates
top_k leaves (one run of 64, its edges, several runs with a ragged end, all 1024).  Both the
one-launch local half and the kernel-per-operator sampler are held to it.  The one permitted
difference is expf's last bit, which moves a draw only when it lands within ~1e-7 of a
boundary; no draw of these seeds does.
"""
import numpy as np
import pytest

from mosship import HipLLM, SampleParams
from mosship import moss_format as mf
from oracle import SampleParams as OSP

pytestmark = pytest.mark.gpu

MODES = [(2, 1.0, 1.0), (63, 0.7, 0.9), (64, 1.0, 0.5), (65, 1.3, 1.0), (129, 0.9, 0.97), (1000, 1.0, 0.8),
         (1024, 1.5, 1.0), (0, 0.0, 0.999)]


@pytest.mark.parametrize("per_op", [False, True])
@pytest.mark.parametrize("top_k,temperature,top_p", MODES)
def test_every_draw_is_sample_tokens(torch_gpu, oracle, golden_model, top_k, temperature, top_p, per_op):
    blob, g = golden_model
    frames, seed, greedy_frames = 4, 77 + top_k, 1
    kw = dict(greedy=False, temperature=temperature, top_k=top_k, top_p=top_p, repetition_penalty=1.2,
              min_frames=2, end_greedy=False, greedy_frames=greedy_frames)
    print(f"top_k {top_k} per_op {per_op}", flush=True)
    m = HipLLM(blob, per_op=per_op)
    m.prefill(np.concatenate([g["rows"], mf.text_rows(np.arange(20) * 37 + 5)]))
    # the same codes again and again, so that the penalty acts on counts above one
    forced = np.full((frames, 17), mf.SLOT, np.int32)
    forced[:, 1:] = np.arange(16) * 61 % 1024
    out = m.generate(frames, SampleParams.make(**kw), seed=seed, forced=forced, logits=True)
    m.close()
    skip = 0
    for f in range(len(out["rows"])):
        if f >= 2:
            skip += 1  # the sampled end gate draws first
        for ch in range(16):
            p = OSP.make(**{**kw, "greedy": f < greedy_frames})
            want = oracle.sample_token(out["logits"][f, ch], p, prev=[int(forced[0, ch + 1])] * f, seed=seed, skip=skip)
            skip += f >= greedy_frames
            assert out["rows"][f, ch + 1] == want, (f, ch)
    assert len(out["rows"]) >= 2
