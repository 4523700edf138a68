"""Recovery of the fused decode kernels (GPU).

The fused global step and local half need every workgroup of their launch resident at
once; each wait between workgroups is bounded, and a launch whose wait runs out is redone
on the per-operator path from the last good state (llm_model.hip: Model::generate's
recover, Model::global_step).  The condition is forced from the host: MOSS_HIP_POLL_BUDGET
gives the waits a budget of a few poll rounds, so they run out while every kernel still
exits normally.  A recovered run must give what the per-operator model gives (bit for bit
when the first launch already fails: every kernel after that is the per-operator path's),
and agree with the oracle to the usual bars whatever frame the recovery hits.
"""
import numpy as np
import pytest
from conftest import max_rel

from mosship import HipLLM, SampleParams
from mosship import moss_format as mf
from oracle import SampleParams as OSP

pytestmark = pytest.mark.gpu
TOL = 1e-3


@pytest.fixture(scope="module")
def state(oracle, golden_model):
    blob, g = golden_model
    rng = np.random.default_rng(78)
    rows = np.concatenate([g["rows"], mf.text_rows(rng.integers(0, mf.VOCAB, 40))])
    m = oracle.model(blob)
    m.prefill(rows, a16=True)
    k, v = m.kv_export(len(rows))
    return blob, k, v, m.hidden()


def _model(blob, k, v, h, monkeypatch=None, budget=None, **kw):
    if budget is not None:
        monkeypatch.setenv("MOSS_HIP_POLL_BUDGET", str(budget))
    g = HipLLM(blob, kv_fp32=True, **kw)
    if budget is not None:
        monkeypatch.delenv("MOSS_HIP_POLL_BUDGET")
    g.kv_import(k, v, h)
    return g


def test_waits_that_run_out_fall_back_to_per_operator(torch_gpu, state, monkeypatch):
    """Budget of one poll round: the first fused launch of every call runs out; generate
    (greedy, repetition penalty) and global_step give the per-operator model's results."""
    blob, k, v, h = state
    frames = 6
    p = SampleParams.make(greedy=True, min_frames=frames, repetition_penalty=1.3)
    ref = _model(blob, k, v, h, per_op=True)
    g = _model(blob, k, v, h, monkeypatch, budget=1)
    print("generate with budget 1", flush=True)
    a = g.generate(frames, p)
    b = ref.generate(frames, p)
    assert g.fallbacks >= 1
    assert np.array_equal(a["rows"], b["rows"])
    assert np.array_equal(g.hidden(), ref.hidden()) and g.position == ref.position
    row = np.concatenate([[mf.SLOT], a["rows"][-1, 1:]]).astype(np.int32)
    before = g.fallbacks
    g.global_step(row)
    ref.global_step(row)
    assert g.fallbacks == before + 1
    assert np.array_equal(g.hidden(), ref.hidden()) and g.position == ref.position
    ka, va = g.kv_export(g.position)
    kb, vb = ref.kv_export(ref.position)
    assert np.array_equal(ka, kb) and np.array_equal(va, vb)
    g.close()
    ref.close()


@pytest.mark.parametrize("budget", ["1@0", "1@1", "1@2", "1@3", "1@5", "1@6", "3", "24"])
def test_recovery_at_any_frame_matches_oracle(torch_gpu, oracle, state, monkeypatch, budget):
    """Waits that run out in a chosen launch ("1@K": one poll round from the model's K-th
    fused launch on; generate alternates local half and global step, and nothing before it
    launches either: K = 0 hits L(0), 1 G(0) -- found at frame 1's readback --, 2 L(1), 3 G(1),
    5 G(2), 6 L(3)) or wherever a few poll rounds fall short
    ("3", "24").
    Teacher-forced codes and logits against the oracle, and the final hidden state and
    position, to the usual bars."""
    blob, k, v, h = state
    frames = 8
    m = oracle.model(blob)
    m.kv_import(k, v)
    m.set_hidden(h)
    ref = m.generate(frames, OSP.make(greedy=True, min_frames=frames), logits=True)
    forced = ref["rows"].copy()
    forced[:, 0] = mf.SLOT
    g = _model(blob, k, v, h, monkeypatch, budget=budget)
    print(f"teacher-forced generate with budget {budget}", flush=True)
    out = g.generate(frames, SampleParams.make(greedy=True, min_frames=frames), forced=forced, logits=True)
    print(f"budget {budget}: {g.fallbacks} fallbacks", flush=True)
    if "@" in budget:
        assert g.fallbacks == 1
    assert np.mean(out["rows"][:, 1:] == ref["rows"][:, 1:]) >= 0.99
    assert max_rel(out["logits"], ref["logits"]) <= TOL
    assert max_rel(g.hidden(), m.hidden()) <= TOL and g.position == m.position
    g.close()


SAMPLED = dict(greedy=False, temperature=0.9, top_p=0.95, repetition_penalty=1.3, end_greedy=False, min_frames=3)
SAMPLED_BUDGETS = ["1@0", "1@1", "1@2", "1@5", "1@6"]


@pytest.mark.parametrize("budget", SAMPLED_BUDGETS)
@pytest.mark.parametrize("top_k", [40, 200])
def test_recovery_of_a_sampled_call(torch_gpu, state, monkeypatch, budget, top_k):
    """The same for a call that draws its codes and, from frame 3 on, its end: the draws go on per
    operator from where the fused launches' stream stood, with the repetition counts of the frames
    before, so codes and length are those of the per-operator model with the same seed.  (The
    logits of the frames before the recovery differ in their last bits, which moves a draw only
    within ~1e-6 of a boundary; none of these does.  Not under W8A8: there a last bit can become a
    step of the int8 quantiser, 1 / 127 of a block's largest value, and the draws that land within
    ~1e-2 of a boundary are many.)"""
    blob, k, v, h = state
    p = SampleParams.make(top_k=top_k, **SAMPLED)
    ref = _model(blob, k, v, h, per_op=True)
    want = ref.generate(8, p, seed=11)["rows"]
    g = _model(blob, k, v, h, monkeypatch, budget=budget)
    print(f"sampled generate, top_k {top_k}, budget {budget}, {len(want)} frames", flush=True)
    got = g.generate(8, p, seed=11)["rows"]
    assert g.fallbacks == 1
    assert len(want) >= 3 and np.array_equal(got, want)
    assert max_rel(g.hidden(), ref.hidden()) <= TOL and g.position == ref.position
    g.close()
    ref.close()


@pytest.mark.parametrize("budget", SAMPLED_BUDGETS)
@pytest.mark.parametrize("a8", [False, True])
def test_recovered_draws_are_sample_tokens(torch_gpu, oracle, state, monkeypatch, budget, a8):
    """Every draw before and after a recovery is sample_token's (sampler.cpp:9-79) on the logits that
    it was made from (the call's own dump), the channel's history of forced codes and the call's
    stream, in which the end gate draws before the codes from frame 3 on."""
    blob, k, v, h = state
    frames, seed, top_k = 6, 12, 40
    forced = np.full((frames, 17), mf.SLOT, np.int32)
    forced[:, 1:] = np.arange(16) * 61 % 1024  # the same codes: counts above one
    g = _model(blob, k, v, h, monkeypatch, budget=budget, decode_a8=a8)
    print(f"sampled generate, a8 {a8}, budget {budget}", flush=True)
    out = g.generate(frames, SampleParams.make(top_k=top_k, **SAMPLED), seed=seed, forced=forced, logits=True)
    assert g.fallbacks == 1 and len(out["rows"]) >= 3
    g.close()
    skip = 0
    for f in range(len(out["rows"])):
        skip += f >= SAMPLED["min_frames"]
        for ch in range(16):
            want = oracle.sample_token(out["logits"][f, ch], OSP.make(top_k=top_k, **SAMPLED),
                                       prev=[int(forced[0, ch + 1])] * f, seed=seed, skip=skip)
            skip += 1
            assert out["rows"][f, ch + 1] == want, (f, ch)
