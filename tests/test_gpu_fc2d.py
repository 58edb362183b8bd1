"""fc2d NSGS on the GPU (fc2d_driver with SICONOS_FRICTION_2D_NSGS_HIP, and
the fc2d_hip.h device layer) against the oracle.

The reference's own test (test_fc2d_1.c on data_collection_fc2d_1.c: tol
1e-5, 10000 iterations) is run through the drop-in driver; its CUDA
counterpart (test_fc2d_gpu.c) runs the same collection.  The GPU sweeps in
colour order; the oracle run in that order gives the same reactions bit for
bit and the same iteration count.
"""
import ctypes as C

import numpy as np
import pytest

from conftest import FC2D_COLLECTION, fixture_file
from oracle import pyoracle as O
from siconos_amd import capi
from siconos_amd import numerics as N

pytestmark = pytest.mark.gpu

FC2D_NSGS_HIP = 440


def _options(tol=1e-5, max_iter=10000):
    o = N.SolverOptions(FC2D_NSGS_HIP)
    o.dparam[N.SICONOS_DPARAM_TOL] = tol
    o.iparam[N.SICONOS_IPARAM_MAX_ITER] = max_iter
    return o


@pytest.mark.parametrize("name", FC2D_COLLECTION)
def test_driver_matches_the_oracle_in_colour_order(lib, name):
    path = fixture_file(name)
    p = N.FrictionContactProblem.from_file(path)
    nc = p.numberOfContacts
    r = np.zeros(2 * nc)
    u = np.zeros(2 * nc)
    o = _options()
    info = N.fc2d_driver(p, r, u, o)
    it = int(o.iparam[N.SICONOS_IPARAM_ITER_DONE])
    res = float(o.dparam[N.SICONOS_DPARAM_RESIDU])
    order = N.Fc2dHipProblem(p).order()
    info_o, r_o, u_o, it_o, res_o = O.Fc2dProblem(path).nsgs(tol=1e-5, max_iter=10000, mode=2,
                                                             order=order)
    print(f"\n[fc2d] {name}: {nc} contacts, {it} sweeps, residual {res:.3e}, "
          f"{int(o.iparam[25])} colours, {o.dparam[24]:.2f} ms")
    assert info == info_o == 0
    assert it == it_o
    np.testing.assert_array_equal(r, r_o)
    np.testing.assert_allclose(u, u_o, rtol=1e-13, atol=1e-13 * np.abs(u_o).max())
    assert abs(res - res_o) <= 1e-12 * max(res_o, 1e-300) + 1e-300
    assert res <= 1e-5


@pytest.mark.parametrize("name", FC2D_COLLECTION)
def test_both_schedules_give_the_same_solve(lib, name):
    """One workgroup for the whole solve and one launch per colour (replayed
    from a graph) run the same per-contact step and the same reductions:
    same reactions, velocities, sweep counts and residual, bit for bit."""
    p = N.FrictionContactProblem.from_file(fixture_file(name))
    H = N.Fc2dHipProblem(p)
    out = {}
    for sched in (1, 2):
        H.set_reaction(np.zeros(2 * p.numberOfContacts))
        s = H.solve(max_iter=10000, tol=1e-5, error_evaluation=2, schedule=sched)
        assert s.schedule == sched
        out[sched] = (s.info, s.iterations, s.residual, H.reaction(), H.velocity())
        print(f"\n[fc2d] {name}: schedule {sched}: {s.iterations} sweeps, {s.solve_ms:.2f} ms")
    a, b = out[1], out[2]
    assert a[:3] == b[:3] and a[0] == 0
    np.testing.assert_array_equal(a[3], b[3])
    np.testing.assert_array_equal(a[4], b[4])


def test_automatic_schedule_and_unknown_schedule(lib):
    """Colours wider than 2048 contacts take the per-colour schedule."""
    small = N.Fc2dHipProblem(N.FrictionContactProblem.from_file(
        fixture_file("FrictionContactProblem00237.dat")))
    assert small.solve(max_iter=10, schedule=0).schedule == 1
    with pytest.raises(RuntimeError):
        small.solve(max_iter=10, schedule=3)


@pytest.mark.parametrize("schedule", [1, 2])
def test_light_mode_max_iter_and_warm_start(lib, schedule):
    path = fixture_file("FrictionContactProblem00237.dat")
    p = N.FrictionContactProblem.from_file(path)
    H = N.Fc2dHipProblem(p)
    order = H.order()
    orc = O.Fc2dProblem(path)
    # no sweep at all: the final full error of the zero reaction
    s = H.solve(max_iter=0, tol=1e-5, error_evaluation=2, schedule=schedule)
    info_o, _, _, it_o, res_o = orc.nsgs(tol=1e-5, max_iter=0, mode=2, order=order)
    assert s.iterations == it_o == 0 and s.info == info_o
    assert abs(s.residual - res_o) <= 1e-12 * max(res_o, 1e-300)
    # LIGHT: stops on the light error, no velocity
    s = H.solve(max_iter=10000, tol=1e-5, error_evaluation=1, schedule=schedule)
    info_o, r_o, _, it_o, res_o = orc.nsgs(tol=1e-5, max_iter=10000, mode=1, order=order)
    assert s.info == info_o == 0 and s.iterations == it_o and not s.velocity_set
    np.testing.assert_array_equal(H.reaction(), r_o)
    # FULL is not evaluated by fc2d_nsgs: max_iter sweeps, info 1, residual inf
    H.set_reaction(np.zeros(2 * p.numberOfContacts))
    s = H.solve(max_iter=7, tol=1e-5, error_evaluation=0, schedule=schedule)
    assert s.info == 1 and s.iterations == 7 and s.residual == np.inf
    # max_iter bounds the sweeps: info 1
    H.set_reaction(np.zeros(2 * p.numberOfContacts))
    s = H.solve(max_iter=3, tol=1e-12, error_evaluation=2, schedule=schedule)
    info_o, r_o, u_o, it_o, res_o = orc.nsgs(tol=1e-12, max_iter=3, mode=2, order=order)
    assert s.info == info_o == 1 and s.iterations == 3
    np.testing.assert_array_equal(H.reaction(), r_o)
    # the resident reaction is the start of the next solve
    s = H.solve(max_iter=10000, tol=1e-5, schedule=schedule)
    info_o, r_o, _, it_o, _ = orc.nsgs(tol=1e-5, max_iter=10000, mode=2, order=order,
                                       reaction=r_o)
    assert s.info == 0 and s.iterations == it_o
    np.testing.assert_array_equal(H.reaction(), r_o)


@pytest.mark.parametrize("name", ["FrictionContactProblem00374.dat",
                                  "FrictionContactProblem00727.dat",
                                  "fc2d_granularflowonwall_02020_00213.dat"])
def test_compute_error_matches_the_oracle(lib, name):
    path = fixture_file(name)
    p = N.FrictionContactProblem.from_file(path)
    orc = O.Fc2dProblem(path)
    rng = np.random.default_rng(5)
    z = rng.normal(size=2 * p.numberOfContacts)
    w = np.zeros_like(z)
    e_o, w_o = orc.compute_error(z)
    norm = float(np.sqrt(np.sum(p.q * p.q)))
    info, e = N.fc2d_compute_error(p, z, w, 1e-5, norm)
    np.testing.assert_array_equal(w, w_o)
    assert abs(e - e_o) <= 1e-13 * e_o
    assert info == (1 if e > 1e-5 else 0)


def test_refusals(lib, tmp_path):
    p2 = N.FrictionContactProblem.from_file(fixture_file("FrictionContactProblem00031.dat"))
    r = np.zeros(2 * p2.numberOfContacts)
    u = np.zeros_like(r)
    o = _options()
    o.iparam[N.SICONOS_NSGS_FREEZING_CONTACT] = 20
    assert N.fc2d_driver(p2, r, u, o) == N.NUMERICS_ERR_NOT_IMPLEMENTED
    o3 = N.SolverOptions(540)  # an fc3d solver is not an fc2d solver
    assert N.fc2d_driver(p2, r, u, o3) == N.NUMERICS_ERR_INVALID_SOLVER
    p3 = N.FrictionContactProblem.from_file(fixture_file("FC3D_Example1_SBM.dat"))
    r3 = np.zeros(9)
    assert N.fc2d_driver(p3, r3, r3.copy(), _options()) == N.NUMERICS_ERR_INVALID_ARGUMENT
    # a singular diagonal block: info 1 before any sweep (fc2d_nsgs.c:318-334)
    path = tmp_path / "singular.dat"
    W = np.diag([1.0, 1.0, 0.0, 1.0])
    txt = "2\n2\n0\n4\n4\n4\t4\n" + "\n".join(" ".join(f"{v:.17g}" for v in W[:, j])
                                             for j in range(4))
    txt += "\n-1 0 -1 0\n0.5 0.5\n"
    path.write_text(txt)
    ps = N.FrictionContactProblem.from_file(str(path))
    r = np.zeros(4)
    o = _options()
    assert N.fc2d_driver(ps, r, np.zeros(4), o) == 1
    assert o.iparam[N.SICONOS_IPARAM_ITER_DONE] == 0
    assert o.dparam[N.SICONOS_DPARAM_RESIDU] == np.inf


def _write_dense_fc2d(path, W, q, mu):
    """A dimension-2 problem in the .dat layout of the dense fixtures
    (dimension, contacts, storage 0, sizes, the rows of W, q, mu)."""
    n = W.shape[0]
    with open(path, "w") as f:
        f.write(f"2\n{n // 2}\n0\n{n}\n{n}\n{n}\t{n}\n")
        for row in W:
            f.write(" ".join(f"{x:.17e}" for x in row) + "\n")
        f.write(" ".join(f"{x:.17e}" for x in q) + "\n")
        f.write(" ".join(f"{x:.17e}" for x in mu) + "\n")


def _edge_problem(case):
    rng = np.random.default_rng(7)
    nc = 1 if case == "one contact" else 40
    if case == "no shared body":
        W = np.zeros((2 * nc, 2 * nc))
        for k in range(nc):
            A = rng.normal(size=(2, 2))
            W[2 * k:2 * k + 2, 2 * k:2 * k + 2] = A @ A.T + 0.1 * np.eye(2)
    else:
        J = rng.normal(size=(2 * nc, 2 * nc + 4))
        W = J @ J.T
    q = rng.normal(size=2 * nc)
    q[0::2] = -np.abs(q[0::2]) - 0.1  # every contact approaching
    mu = np.zeros(nc) if case == "frictionless" else rng.uniform(0.1, 0.9, nc)
    return W, q, mu


@pytest.mark.parametrize("case", ["one contact", "no shared body", "frictionless"])
def test_edge_cases_through_the_driver(lib, tmp_path, case):
    """One contact; contacts whose W is block diagonal (one colour); a fully
    coupled frictionless problem (every contact a colour of its own, the
    tangential reactions stay 0): through fc2d_driver, against the oracle in
    colour order, bit for bit, with both schedules the same."""
    path = str(tmp_path / "edge.dat")
    _write_dense_fc2d(path, *_edge_problem(case))
    p = N.FrictionContactProblem.from_file(path)
    nc = p.numberOfContacts
    r, u = np.zeros(2 * nc), np.zeros(2 * nc)
    o = _options()
    info = N.fc2d_driver(p, r, u, o)
    it = int(o.iparam[N.SICONOS_IPARAM_ITER_DONE])
    H = N.Fc2dHipProblem(p)
    order = H.order()
    info_o, r_o, u_o, it_o, res_o = O.Fc2dProblem(path).nsgs(tol=1e-5, max_iter=10000, mode=2,
                                                             order=order)
    assert info == info_o == 0 and it == it_o
    np.testing.assert_array_equal(r, r_o)
    np.testing.assert_allclose(u, u_o, rtol=1e-13, atol=1e-13 * np.abs(u_o).max())
    assert H.num_colours == (1 if case != "frictionless" else nc)
    if case == "frictionless":
        assert np.all(r[1::2] == 0.0)
    for sched in (1, 2):
        H.set_reaction(np.zeros(2 * nc))
        s = H.solve(max_iter=10000, tol=1e-5, error_evaluation=2, schedule=sched)
        assert s.info == 0 and s.iterations == it
        np.testing.assert_array_equal(H.reaction(), r)


@pytest.mark.parametrize("nc", [1, 64, 65, 700, 9200, 9201])
@pytest.mark.parametrize("row_mode,own_zero", [(0, 0), (0, 1), (1, 0)])
def test_one_workgroup_at_the_edges_of_its_lds(lib, nc, row_mode, own_zero):
    """A chain of contacts (every third one also tied to the first, so that
    rows differ in length) up to and beyond the size whose reactions fit LDS:
    both schedules give the same bits, from a start that is not zero."""
    rng = np.random.default_rng(nc)
    rows = [[] for _ in range(nc)]
    for c in range(nc):
        for d in {c, c - 1, c + 1} | ({0} if c % 3 == 0 and c < 90 else set()):
            if 0 <= d < nc:
                rows[c].append(d)
    for c in range(3, min(nc, 90), 3):
        rows[0].append(c)
    rp, cols, vals, diag = [0], [], [], []
    for c in range(nc):
        blk = {d: rng.normal(size=(2, 2)) * 0.1 + (3.0 * np.eye(2) if d == c else 0.0)
               for d in sorted(set(rows[c]))}
        for i in range(2):
            for d, b in blk.items():
                for k in range(2):
                    cols.append(2 * d + k)
                    vals.append(b[i, k])
            rp.append(len(cols))
        diag.append(blk[c].reshape(-1, order="F"))
    rp, cols = np.array(rp, dtype=np.int64), np.array(cols, dtype=np.int64)
    vals, diag = np.array(vals), np.ascontiguousarray(np.concatenate(diag))
    q, mu = rng.normal(size=2 * nc), rng.uniform(0.1, 0.8, nc)
    h = C.c_void_p()
    assert lib.fc2d_hip_problem_create(nc, N.lptr(rp), N.lptr(cols), N.dptr(vals), row_mode,
                                       own_zero, N.dptr(diag), N.dptr(q), N.dptr(mu), 0,
                                       C.byref(h)) == 0, capi.last_error()
    P = N.Fc2dHipProblem.__new__(N.Fc2dHipProblem)
    P._lib, P.nc, P._h = lib, nc, h
    start = np.abs(rng.normal(size=2 * nc))
    out = []
    for schedule in (1, 2):
        P.set_reaction(start)
        s = P.solve(max_iter=30, tol=1e-9, schedule=schedule)
        out.append((P.reaction(), P.velocity(), s.iterations, s.residual, s.info))
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("nc", [200, 400])
def test_fully_coupled_contacts(lib, nc):
    """Contacts that are all coupled to each other, a colour each, on both
    sides of the size whose padded layout is built: a problem takes little more
    memory than its rows or the layout's bound, and both schedules give the
    same bits."""
    def free():  # (the HIP runtime that the library is linked to)
        a, b = C.c_size_t(), C.c_size_t()
        assert lib.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value
    rng = np.random.default_rng(nc)
    n2 = 2 * nc
    G = rng.normal(size=(n2, n2)) / np.sqrt(n2)
    W = G @ G.T + np.eye(n2)
    rp = np.arange(n2 + 1, dtype=np.int64) * n2
    cols = np.tile(np.arange(n2, dtype=np.int64), n2)
    vals = np.ascontiguousarray(W.reshape(-1))
    diag = np.concatenate([W[2 * c:2 * c + 2, 2 * c:2 * c + 2].reshape(-1, order="F")
                           for c in range(nc)])
    q, mu = rng.normal(size=n2), rng.uniform(0.1, 0.8, nc)
    before = free()
    h = C.c_void_p()
    assert lib.fc2d_hip_problem_create(nc, N.lptr(rp), N.lptr(cols), N.dptr(vals), 0, 0,
                                       N.dptr(diag), N.dptr(q), N.dptr(mu), 0,
                                       C.byref(h)) == 0, capi.last_error()
    P = N.Fc2dHipProblem.__new__(N.Fc2dHipProblem)
    P._lib, P.nc, P._h = lib, nc, h
    # 12 bytes an entry in the rows; the layout is kept up to 256 MB
    assert before - free() < (12 * n2 * n2 + (256 << 20) + (32 << 20))
    assert P.num_colours == nc
    out = []
    for schedule in (0, 2):
        P.set_reaction(np.zeros(n2))
        s = P.solve(max_iter=3, tol=1e-9, schedule=schedule)
        out.append((P.reaction(), P.velocity(), s.iterations, s.residual, s.info))
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
