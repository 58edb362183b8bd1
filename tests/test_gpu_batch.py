"""Many independent problems in one persistent launch (fc3d_hip_batch_*),
each checked against the oracle run in the same per-problem sweep order."""
import numpy as np
import pytest

from conftest import natural_residual
from siconos_amd import numerics as N

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def batch():
    probs = N.generate_batch(96, 8, 512, 0.1, 0.9, 11)
    return probs, N.Batch(probs)


def per_problem_order(B, order, k, nc):
    c0 = B.offsets[k]
    sel = order[(order >= c0) & (order < c0 + nc)]
    return sel - c0


@pytest.mark.parametrize("schedule", [1, 2])
def test_batch_fp64_bit_exact_per_problem(oracle, batch, schedule):
    probs, B = batch
    B.set_reaction(np.zeros(3 * B.ntotal))
    s, info, iters, res = B.solve(N.hip_params(tol=1e-6, max_iter=1000, schedule=schedule))
    assert s.schedule == schedule
    r, u, order = B.reaction(), B.velocity(), B.order()
    for k, (W, q, mu) in enumerate(probs):
        c0 = B.offsets[k]
        io, ro, uo, it, reso = oracle.nsgs(W, q, mu, tol=1e-6, max_iter=1000,
                                           order=per_problem_order(B, order, k, W.nc))
        assert info[k] == io and iters[k] == it, k
        np.testing.assert_array_equal(r[3 * c0:3 * (c0 + W.nc)], ro, err_msg=f"problem {k}")
        np.testing.assert_array_equal(u[3 * c0:3 * (c0 + W.nc)], uo, err_msg=f"problem {k}")
        np.testing.assert_allclose(res[k], reso, rtol=1e-12)
    assert s.converged == int(np.sum(res <= 1e-6))


def test_batch_mixed_precision_meets_tolerance(batch):
    probs, B = batch
    B.set_reaction(np.zeros(3 * B.ntotal))
    s, info, iters, res = B.solve(N.hip_params(tol=1e-6, max_iter=1000, precision=1))
    assert s.fp32_sweeps > 0
    r = B.reaction()
    for k, (W, q, mu) in enumerate(probs):
        if info[k] != 0:
            continue
        c0 = B.offsets[k]
        e, _ = natural_residual(W, q, mu, r[3 * c0:3 * (c0 + W.nc)])
        assert e <= 1e-6 * (1 + 1e-9), k
    assert s.converged >= 0.95 * len(probs)


def test_batch_autotuner_and_warm_start(batch):
    probs, B = batch
    B.set_reaction(np.zeros(3 * B.ntotal))
    s1, info1, it1, res1 = B.solve(N.hip_params(tol=1e-6, max_iter=1000, schedule=0))
    assert s1.schedule in (1, 2)
    r1 = B.reaction()
    # a converged start stays converged: one sweep at most per problem
    s2, info2, it2, res2 = B.solve(N.hip_params(tol=1e-6, max_iter=1000, schedule=0))
    assert np.all(it2[info1 == 0] <= 2)
    # warm_start = 1 restarts from zero and reproduces the first solve
    s3, info3, it3, res3 = B.solve(N.hip_params(tol=1e-6, max_iter=1000, warm_start=1))
    np.testing.assert_array_equal(B.reaction(), r1)


def test_batch_rejects_cross_problem_columns():
    probs = N.generate_batch(3, 8, 20, 0.1, 0.9, 12)
    W, q, mu = probs[1]
    ci = W.col_idx.copy()
    ci[0] = W.nc + 3  # points into the next problem
    bad = [probs[0], (N.SparseBlock3(W.row_ptr, ci, W.values), q, mu), probs[2]]
    with pytest.raises(RuntimeError, match="out of range"):
        N.Batch(bad)


@pytest.fixture(scope="module")
def batch4096():
    probs = N.generate_batch(4096, 8, 512, 0.1, 0.9, 3)
    return probs, N.Batch(probs)


@pytest.mark.parametrize("precision", [0, 1])
def test_full_4096_problem_launch_converges_everywhere(oracle, batch4096, precision):
    """The 4096-problem configuration in one persistent launch, every problem
    to its own FP64 residual <= 1e-6.  A few problems need far more sweeps
    than the rest (up to ~12k for one 29-contact problem, in the oracle's
    natural order too), so the sweep cap is 20000.  The oracle recomputes the
    residual of a sample of problems, the slowest ones included."""
    probs, B = batch4096
    nc = sum(W.nc for W, _, _ in probs)
    B.set_reaction(np.zeros(3 * nc))
    prm = N.hip_params(tol=1e-6, max_iter=20_000, precision=precision, fp32_tol=1e-6,
                       fp32_local_solver=550 if precision else 0, fp32_local_tol=1e-7)
    s, info, iters, res = B.solve(prm)
    print(f"\nprecision {precision}: {s.converged}/4096 converged, max sweeps {int(iters.max())}, "
          f"{s.solve_ms:.1f} ms", flush=True)
    assert s.converged == 4096 and np.all(info == 0) and np.all(res <= 1e-6)
    r = B.reaction()
    off = np.concatenate([[0], np.cumsum([W.nc for W, _, _ in probs])])
    slow = list(np.argsort(iters)[-16:])
    sample = sorted(set(slow) | set(range(0, 4096, 128)))
    for k in sample:
        W, q, mu = probs[k]
        e, _ = oracle.compute_error(W, q, mu, r[3 * off[k]:3 * off[k + 1]])
        assert e <= 1e-6, (k, e)
        assert e == pytest.approx(res[k], rel=1e-9)


@pytest.mark.parametrize("sizes", [(1, 2), (63, 64, 65), (513, 40), (2048, 8), (2049, 8)])
@pytest.mark.parametrize("mode", [1, 2])
def test_quads_at_their_edges(oracle, sizes, mode):
    """Four waves a problem at the edges of a slice, with rows longer than the 16
    planes a lane holds, and around the 2048 contacts that LDS holds (here in
    colours of three slices, so a wave a slice; test_four_waves_in_both_forms
    has 2048 contacts in LDS), bit for bit per problem."""
    probs = []
    for k, n in enumerate(sizes):
        nb = max(3, n // 6)  # ~24 blocks a row
        while n > nb * (nb - 1) // 2:
            nb += 1
        g = N.generate_random_pairs(nb, n, 0.1, 0.9, 70 + k)
        probs.append((g.W, g.q, g.mu))
    B = N.Batch(probs)
    s, info, it, res = B.solve(N.hip_params(tol=1e-4, max_iter=25, warm_start=1, schedule=2,
                                            error_evaluation=mode))
    order, r = B.order(), B.reaction()
    for (W, q, mu), a, b, n in zip(probs, B.offsets[:-1], B.offsets[1:], it):
        _, ro, _, _, _ = oracle.nsgs(W, q, mu, tol=1e-30, max_iter=int(n), order=order[a:b] - a)
        np.testing.assert_array_equal(r[3 * a:3 * b], ro)


@pytest.mark.parametrize("nc", [1, 64, 150, 400])
def test_small_problem_in_one_workgroup(oracle, nc):
    """A small problem's plain solve (one workgroup) against the oracle in the
    same order and against one launch per colour: the same bits and sweeps in
    every evaluation mode, from the resident reaction too."""
    nb = max(3, int(nc * 0.45))
    while nc > nb * (nb - 1) // 2:
        nb += 1
    g = N.generate_random_pairs(nb, nc, 0.2, 0.5, 5)
    P = N.HipProblem(g.W, g.q, g.mu)
    start = np.abs(np.random.default_rng(1).normal(size=3 * nc))
    for mode in (0, 1, 2, 3):
        out = []
        for schedule in (0, 1):
            P.set_reaction(start)
            s = P.solve(N.hip_params(tol=1e-5, max_iter=40, schedule=schedule,
                                     error_evaluation=mode, error_frequency=3))
            out.append((P.reaction(), s.iterations, s.info, s.residual, s.incr_error))
        np.testing.assert_array_equal(out[0][0], out[1][0])
        assert out[0][1:3] == out[1][1:3]
        for a, b in zip(out[0][3:], out[1][3:]):
            assert a == b or a == pytest.approx(b, rel=1e-12)
    _, ro, _, it, _ = oracle.nsgs(g.W, g.q, g.mu, tol=1e-5, max_iter=40, order=P.order(),
                                  reaction=start)
    P.set_reaction(start)
    s = P.solve(N.hip_params(tol=1e-5, max_iter=40))
    assert s.iterations == it
    np.testing.assert_array_equal(P.reaction(), ro)


@pytest.mark.parametrize("kind", ["narrow", "wide"])
@pytest.mark.parametrize("precision", [0, 1])
def test_four_waves_in_both_forms(oracle, kind, precision):
    """Colours of at most a slice up to the contacts that LDS holds (quads), and
    colours of ten slices (four waves beside each other): four waves a problem
    give the bits of one wave a problem, and in FP64 the oracle's."""
    if kind == "narrow":  # 102 bodies: at most 51 contacts a colour
        g = N.generate_random_pairs(102, 2048, 0.1, 0.9, 3)
        probs = [(g.W, g.q, g.mu), (g.W, -0.5 * g.q, g.mu)]
    else:  # a chain of contacts: two colours
        rng = np.random.default_rng(4)
        probs = []
        for n in (1200, 65):
            at = [[d for d in (c - 1, c, c + 1) if 0 <= d < n] for c in range(n)]
            rp = np.concatenate([[0], np.cumsum([len(a) for a in at])])
            blocks = [(3.0 if d == c else -0.4) * np.eye(3).reshape(-1)
                      for c in range(n) for d in at[c]]
            W = N.SparseBlock3(rp, np.concatenate(at), np.concatenate(blocks))
            probs.append((W, rng.normal(size=3 * n), rng.uniform(0.2, 0.7, n)))
    B = N.Batch(probs)
    out = []
    for schedule in (1, 2):
        s, info, it, res = B.solve(N.hip_params(tol=1e-6, max_iter=12, warm_start=1,
                                                schedule=schedule, precision=precision,
                                                fp32_tol=1e-3))
        out.append((B.reaction(), it))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    np.testing.assert_array_equal(out[0][1], out[1][1])
    if precision == 0:
        order = B.order()
        for (W, q, mu), a, b, n in zip(probs, B.offsets[:-1], B.offsets[1:], out[0][1]):
            _, ro, _, _, _ = oracle.nsgs(W, q, mu, tol=1e-30, max_iter=int(n),
                                         order=order[a:b] - a)
            np.testing.assert_array_equal(out[1][0][3 * a:3 * b], ro)
