"""Batched assembly on device 0: the z-marching tilings give bit-identical results;
graph replays reproduce the eager results, with the coefficient changed and
eager work done between replays (each replay checked); a batched problem
matches the oracle."""
import numpy as np
import pytest

import oracle
from _helpers import STRUCT_KEYS, rel_err
from gridap_amd import AssemblyBatch, flux_operator_from_workload, problem_from_workload
from gridap_amd import workloads as W
from gridap_amd._lib import KERNEL_HBM_PATTERNS

pytestmark = pytest.mark.gpu


def make(ctx, p):
    assem, data = problem_from_workload(ctx, p)
    return assem, assem._problem_for(data)


def values(prob):
    prob.sync()
    return [(P["val"].copy(), P["b"].copy()) for P in (prob.export_part(k) for k in range(prob.nparts))]


@pytest.mark.parametrize("p", [W.poisson3d_q1(20, (2, 2, 2)), W.poisson3d_q2_fourier(10, (2, 1, 2)),
                               W.poisson3d_q1((9, 14, 40), (1, 2, 3))],
                         ids=["q1-20", "q2-10", "q1-aniso"])
def test_tilings_and_autotuned_kernel(gpu_ctx, p):
    """The z-marching kernel's column length splits the rows over workgroups and
    changes no value; the autotuner's kernel sums in another order."""
    assem, prob = make(gpu_ctx, p)
    got = []
    for rows_z in (16, 32, 64):
        prob.set_kernel(0, rows_z)
        prob.numeric()
        got.append(values(prob))
    for other in got[1:]:
        for (v0, b0), (v1, b1) in zip(got[0], other):
            assert np.array_equal(v0, v1) and np.array_equal(b0, b1)
    b = AssemblyBatch(gpu_ctx)
    b.add(prob)
    assert b.autotune(reps=2)[0] == -2 and prob.get_kernel()[0] == 2  # pair lattice
    prob.numeric()
    for (v0, b0), (v1, b1) in zip(got[0], values(prob)):
        assert rel_err(v1, v0) <= 1e-13 and rel_err(b1, b0) <= 1e-13
    b.close()
    prob.close()


def test_kernel_reported_where_there_is_a_choice(gpu_ctx):
    """Only 3D diffusion has kernels to choose from: the others report variant 0,
    and the autotuner a positive number."""
    diffusion = make(gpu_ctx, W.poisson3d_q1(6, (2, 1, 1)))[1]
    assert diffusion.get_kernel()[0] == 2
    op = flux_operator_from_workload(gpu_ctx, W.plaplacian3d_q1(6, (2, 1, 1)))
    others = [make(gpu_ctx, W.poisson2d_q1(8, (2, 1)))[1], op._problem(),
              make(gpu_ctx, W.elasticity3d_q2((3, 3, 2), (1, 1, 1)))[1]]
    assert [prob.get_kernel()[0] for prob in others] == [0, 0, 0]
    b = AssemblyBatch(gpu_ctx)
    for prob in [diffusion] + others:
        b.add(prob)
    chosen = b.autotune(reps=1)
    assert chosen[0] == -2 and all(c > 0 for c in chosen[1:])
    b.close()
    for prob in [diffusion] + others:
        prob.close()


@pytest.mark.parametrize("p", [W.poisson3d_q2_fourier(9, (2, 1, 3)), W.poisson3d_q2_fourier(6, (1, 2, 2), strategy="full"),
                               W.poisson3d_q1(11, (2, 2, 1)), dict(W.poisson3d_q2_fourier(7, (2, 2, 1)), qdeg=2)],
                         ids=["q2", "q2-full", "q1", "q2-qd2"])
@pytest.mark.parametrize("variant", [1, 2, 3], ids=["per-tile", "pair-lattice", "wave-slab"])
def test_tile_kernel_matches_oracle(gpu_ctx, p, variant):
    print("tile kernel variant", variant, p["order"], p["cells"], p["parts"], flush=True)
    if variant == 3 and p["order"] != 2:
        pytest.skip("the wave-slab kernel is built for Q2")
    r = oracle.run(p)
    assem, prob = make(gpu_ctx, p)
    prob.set_kernel(variant)
    assert prob.get_kernel()[0] == variant
    prob.numeric()
    prob.sync()
    for k, P in enumerate(r.parts):
        Q = prob.export_part(k)
        for key in STRUCT_KEYS:
            assert np.array_equal(P[key], Q[key]), (k, key)
        assert rel_err(Q["val"], P["val"]) <= 1e-12
        assert rel_err(Q["b"], P["b"]) <= 1e-12
        no = P["n_own"]
        assert np.all(Q["val"][Q["rowptr"][no]:] == 0.0) and np.all(Q["b"][no:] == 0.0)
    # back to z-marching with 16-row columns: same matrix to rounding
    prob.set_kernel(0, 16)
    prob.numeric()
    prob.sync()
    for k, P in enumerate(r.parts):
        Q = prob.export_part(k)
        assert rel_err(Q["val"], P["val"]) <= 1e-12
    prob.close()


@pytest.mark.parametrize("p", [W.poisson3d_q2_fourier(7, (2, 1, 2)), W.poisson3d_q1(9, (2, 2, 1)),
                               W.poisson3d_q2_fourier(6, (1, 2, 2), strategy="full")],
                         ids=["q2", "q1", "q2-full"])
@pytest.mark.parametrize("variant", [0, 1, 3], ids=["z-marching", "per-tile", "wave-slab"])
def test_hbm_pattern_instances_match_oracle(gpu_ctx, p, variant):
    """Tiles with more distinct position patterns than LDS holds run kernel
    instances that read the patterns from HBM; the flag sends every tile there.
    (The pair-lattice kernel has no such tiles and ignores the flag.)"""
    print("hbm-pattern instance, variant", variant, p["order"], p["cells"], p["parts"], flush=True)
    if variant == 3 and p["order"] != 2:
        pytest.skip("the wave-slab kernel is built for Q2")
    r = oracle.run(p)
    assem, prob = make(gpu_ctx, p)
    prob.set_kernel(variant | KERNEL_HBM_PATTERNS, 8)
    assert prob.get_kernel()[0] == variant | KERNEL_HBM_PATTERNS
    prob.numeric()
    prob.sync()
    for k, P in enumerate(r.parts):
        Q = prob.export_part(k)
        assert rel_err(Q["val"], P["val"]) <= 1e-12
        assert rel_err(Q["b"], P["b"]) <= 1e-12
        no = P["n_own"]
        assert np.all(Q["val"][Q["rowptr"][no]:] == 0.0) and np.all(Q["b"][no:] == 0.0)
    prob.close()


def test_graph_replays_match_eager(gpu_ctx):
    ws = W.batched_q1(seed=3, count=6, lo=6, hi=14)
    probs = [make(gpu_ctx, dict(q, modes=np.zeros((0, 5))))[1] for q in ws]
    rng = np.random.default_rng(0)
    kap = [[np.exp(rng.normal(size=int(np.prod(q["cells"])))) for q in ws] for _ in range(2)]
    eager = []
    for v in range(2):
        for prob, k in zip(probs, kap[v]):
            prob.set_cell_coefficient(k)
            prob.numeric()
        eager.append([values(prob) for prob in probs])
    b = AssemblyBatch(gpu_ctx)
    for prob in probs:
        b.add(prob)
    b.autotune(reps=1)
    b.capture()
    for rep in range(6):
        v = rep % 2
        for prob, k in zip(probs, kap[v]):
            prob.set_cell_coefficient(k)  # same device buffer, new contents
        b.launch()
        b.sync()
        for prob, ref in zip(probs, eager[v]):
            for (v0, b0), (v1, b1) in zip(ref, values(prob)):
                assert np.array_equal(v0, v1) and np.array_equal(b0, b1), rep
        probs[rep % len(probs)].numeric()  # eager work between replays
        probs[rep % len(probs)].sync()
    b.close()
    for prob in probs:
        prob.close()


def test_batched_problem_matches_oracle(gpu_ctx):
    q = W.batched_q1(seed=5, count=3, lo=7, hi=12)[2]
    r = oracle.run(q)
    assem, prob = make(gpu_ctx, q)
    b = AssemblyBatch(gpu_ctx)
    b.add(prob)
    b.autotune(reps=1)
    b.capture()
    b.launch()
    b.sync()
    for k, P in enumerate(r.parts):
        Q = prob.export_part(k)
        for key in STRUCT_KEYS:
            assert np.array_equal(P[key], Q[key]), (k, key)
        assert rel_err(Q["val"], P["val"]) <= 1e-12
        assert rel_err(Q["b"], P["b"]) <= 1e-12
    b.close()
    prob.close()
