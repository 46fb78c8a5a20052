"""The grouped MoE products over many jobs (kq_moe_prefill.hip) on the GPU, at
shapes its rule takes below 96 tokens and at its groups' edges; oracle, bounds
and helpers as for the other MoE paths (test_gpu_moe.py, test_gpu_chain.py)."""
import numpy as np
import pytest

import aspida_amd as aa
import oracle
from aspida_amd import synth
from gpu_helpers import ncpu
from test_gpu_chain import FUSED_NORM_LAYERS, _chain_model, _close, _no_near_ties, _register
from test_gpu_moe import _assert_moe, _Dq, _layer, _moe_scale, _run_packed

pytestmark = pytest.mark.gpu

# dim, inter, n_exp, top_k, gate/up kind, down kind, gated, tokens, tokens that all
# choose expert 0.  Groups of up to 32 jobs (a shared expert of 17 and 50 jobs, one
# full and one partial group; expert 0 with exactly 32 and 33) and of up to 64
# (exactly 64, 65; short ones on the one-block form); tokens that fill no XCD round.
CASES = [
    (1024, 512, 8, 4, aa.Q4_K, aa.Q6_K, True, 17, 0),
    (1024, 512, 8, 4, aa.Q6_K, aa.Q4_K, False, 33, 33),
    (1024, 512, 16, 3, aa.Q5_K, aa.Q8_0, True, 32, 32),
    (2048, 256, 5, 2, aa.Q2_K, aa.Q3_K, True, 50, 7),
    (1024, 768, 6, 3, aa.Q8_0, aa.Q2_K, False, 65, 65),
    (2304, 256, 4, 2, aa.Q3_K, aa.Q5_K, True, 130, 64),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"d{c[0]}i{c[1]}e{c[2]}k{c[3]}g{c[4]}d{c[5]}T{c[7]}")
def test_moe_many_jobs(case):
    dim, inter, n_exp, top_k, gk, dk, gated, T, crowd = case
    gen = synth.rng(5100 + dim + inter + T)
    L = _layer(gen, dim, inter, n_exp, gk, gk, dk)
    X = synth.activations_np(T * dim, gen).reshape(T, dim)
    idx = np.zeros((T, top_k), np.int32)
    tw = np.zeros((T, top_k), np.float32)
    for t in range(T):
        logits = gen.standard_normal(n_exp).astype(np.float32)
        logits[0] = 20.0 if t < crowd else -20.0
        idx[t], tw[t] = oracle.route(logits, top_k)
    y1, y2 = _run_packed(aa.DeviceOps(), L, dim, inter, n_exp, top_k, gk, dk, gated, X, idx, tw)
    assert np.array_equal(y1.view(np.uint32), y2.view(np.uint32)), "not deterministic"
    sgi = L["sgi"] if gated else None
    dq = _Dq(L, dim, inter, n_exp)
    for t in sorted(set(np.linspace(0, T - 1, min(T, 24)).astype(int).tolist() + [T - 1, max(crowd - 1, 0)])):
        want = oracle.moe_experts(X[t], dim, top_k, inter, n_exp, idx[t], tw[t], L["gate"], L["up"], L["down"],
                                  L["shg"], L["shu"], L["shd"], shared_gate_inp=sgi, nthreads=ncpu())
        _assert_moe(y1[t], want, f"T={T} token {t}", _moe_scale(dq, X[t], top_k, idx[t], tw[t], sgi))


def test_moe_many_jobs_invalid_and_repeated_experts():
    """A token with an expert outside [0, n_exp) keeps its y unwritten; one that
    lists an expert twice gets both contributions."""
    dim, inter, n_exp, top_k, T = 1024, 512, 6, 3, 20
    gen = synth.rng(5200)
    L = _layer(gen, dim, inter, n_exp, aa.Q5_K, aa.Q5_K, aa.Q6_K)
    X = synth.activations_np(T * dim, gen).reshape(T, dim)
    idx = np.zeros((T, top_k), np.int32)
    tw = np.zeros((T, top_k), np.float32)
    for t in range(T):
        idx[t], tw[t] = oracle.route(gen.standard_normal(n_exp).astype(np.float32), top_k)
    idx[3], idx[9], idx[11] = [2, 2, 0], [1, n_exp, 0], [-1, 2, 3]
    y, _ = _run_packed(aa.DeviceOps(), L, dim, inter, n_exp, top_k, aa.Q5_K, aa.Q6_K, True, X, idx, tw)
    assert np.all(np.isnan(y[[9, 11]]))
    for t in (0, 3, 8, 10, 19):
        want = oracle.moe_experts(X[t], dim, top_k, inter, n_exp, idx[t], tw[t], L["gate"], L["up"], L["down"],
                                  L["shg"], L["shu"], L["shd"], shared_gate_inp=L["sgi"], nthreads=ncpu())
        _assert_moe(y[t], want, f"token {t}")


def test_model_chain_many_lanes():
    """Lane batches of the model chain whose experts take the grouped products:
    first run (eager) and two graph replays against the oracle, the next norm in
    the experts' combine included."""
    gen = synth.rng(5300)
    dim, inter, n_exp, top_k, B = 1024, 512, 16, 6, 16
    M = _chain_model(gen, dim, inter, n_exp, top_k, 300, 64, FUSED_NORM_LAYERS)
    ch = _register(M)
    try:
        rows = gen.integers(0, 64, B).astype(np.int32)
        first = ch.forward_batch(rows)
        for b, r in enumerate(rows):
            _, want, routes = oracle.chain_forward(M, int(r))
            _no_near_ties(routes, top_k, f"lane {b}")
            _close(first[b], want, f"lane {b} (row {r})")
        for _ in range(2):
            ch.forward(int(rows[0]))
            assert np.array_equal(ch.forward_batch(rows).view(np.uint32), first.view(np.uint32))
    finally:
        ch.reset()
