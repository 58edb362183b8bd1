"""Device functions through the C-ABI, against the oracle (bit-exact in FP64:
both sides round every product before the sum it feeds)."""
import numpy as np
import pytest

from conftest import read_ac_inputs
from siconos_amd import capi
from siconos_amd import numerics as N

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("formulation,fn", [(0, "oracle_computeAlartCurnierSTD"),
                                            (1, "oracle_computeAlartCurnierJeanMoreau")])
def test_alart_curnier_kernel_on_acinputs(oracle, lib, formulation, fn):
    R, U, MU, RHO = read_ac_inputs()
    n = len(MU)
    F, A, B = np.zeros(3 * n), np.zeros(9 * n), np.zeros(9 * n)
    Rf, Uf, RHOf = (np.ascontiguousarray(x.reshape(-1)) for x in (R, U, RHO))
    rc = lib.fc3d_hip_alart_curnier(n, N.dptr(Rf), N.dptr(Uf), N.dptr(MU), N.dptr(RHOf),
                                    formulation, N.dptr(F), N.dptr(A), N.dptr(B))
    assert rc == 0, capi.last_error()
    L = oracle.load()
    for k in range(n):
        Fo, Ao, Bo = np.zeros(3), np.zeros(9), np.zeros(9)
        getattr(L, fn)(oracle.d(Rf[3 * k:3 * k + 3].copy()), oracle.d(Uf[3 * k:3 * k + 3].copy()),
                       MU[k], oracle.d(RHOf[3 * k:3 * k + 3].copy()), oracle.d(Fo), oracle.d(Ao),
                       oracle.d(Bo))
        np.testing.assert_array_equal(F[3 * k:3 * k + 3], Fo)
        np.testing.assert_array_equal(A[9 * k:9 * k + 9], Ao)
        np.testing.assert_array_equal(B[9 * k:9 * k + 9], Bo)


def test_projection_kernel(oracle, lib):
    rng = np.random.default_rng(21)
    n = 5000
    r = rng.normal(size=3 * n)
    mu = rng.uniform(0.05, 1.2, size=n)
    g = r.copy()
    assert lib.fc3d_hip_projection_on_cone(n, N.dptr(g), N.dptr(mu)) == 0
    L = oracle.load()
    for k in range(n):
        x = r[3 * k:3 * k + 3].copy()
        L.oracle_projectionOnCone(oracle.d(x), mu[k])
        np.testing.assert_array_equal(g[3 * k:3 * k + 3], x)


def local_params_from(o, sid):
    """C-ABI parameters equal to the oracle's local options (reference defaults)."""
    return N.hip_params(local_solver=sid, local_max_iter=int(o.iparam[0]),
                        local_tol=float(o.dparam[0]), local_formulation=int(o.iparam[10]),
                        rho_strategy=int(o.iparam[9]), rho_constant=float(o.dparam[3]),
                        ls_max_iter=int(o.iparam[12]), hybrid_strategy=int(o.iparam[14]),
                        hybrid_max_loop=int(o.iparam[15]), hybrid_max_iter=int(o.iparam[16]))


@pytest.mark.parametrize("sid", [565, 551, 550, 553, 552])
def test_local_solve_kernel(oracle, lib, sid):
    rng = np.random.default_rng(22 + sid)
    n = 2000
    Ws, qs, mus, r0 = [], [], [], []
    for k in range(n):
        M = rng.normal(size=(3, 3))
        W = M @ M.T + rng.uniform(0.1, 3) * np.eye(3)
        if k % 3 == 0:
            W = np.diag([2.0, 7.0, 7.0])
        Ws.append(W.reshape(-1, order="F"))
        qs.append(rng.normal(size=3))
        mus.append(rng.uniform(0.1, 0.9))
        r0.append(rng.normal(size=3) * (k % 2))
    W = np.ascontiguousarray(np.concatenate(Ws))
    q = np.ascontiguousarray(np.concatenate(qs))
    mu = np.array(mus)
    r = np.ascontiguousarray(np.concatenate(r0))
    o = oracle.Options.local(sid)
    p = local_params_from(o, sid)
    state = np.zeros(4 * n)
    info = np.zeros(n, dtype=np.int32)
    rg = r.copy()
    assert lib.fc3d_hip_local_solve(n, N.dptr(W), N.dptr(q), N.dptr(mu), N.dptr(rg), p,
                                    N.dptr(state), 1, N.iptr(info)) == 0, capi.last_error()
    L = oracle.load()
    for k in range(n):
        st = np.zeros(4)
        w = W[9 * k:9 * k + 9].copy()
        L.oracle_local_state_init(oracle.d(w), o.p, oracle.d(st))
        x = r[3 * k:3 * k + 3].copy()
        L.oracle_local_solve(oracle.d(w), oracle.d(q[3 * k:3 * k + 3].copy()), mu[k],
                             oracle.d(x), o.p, oracle.d(st))
        np.testing.assert_array_equal(rg[3 * k:3 * k + 3], x, err_msg=f"contact {k}")
        np.testing.assert_array_equal(state[4 * k:4 * k + 4], st)


def test_local_solve_kernel_spectral_norm_rho(oracle, lib):
    """Rho strategy SPECTRAL_NORM (onecontact...c:132-135, 1/eig_3x3[0]):
    the device's acos/cos may differ from the host libm's in the last bit,
    so rho is compared to 4 ulp and the local solution to 1e-12 relative."""
    rng = np.random.default_rng(41)
    n = 2000
    Ws, qs, mus = [], [], []
    for k in range(n):
        M = rng.normal(size=(3, 3))
        W = M @ M.T + rng.uniform(0.1, 3) * np.eye(3)
        if k % 4 == 0:
            W = np.diag([2.0, 7.0, 7.0])
        Ws.append(W.reshape(-1, order="F"))
        qs.append(rng.normal(size=3))
        mus.append(rng.uniform(0.1, 0.9))
    W = np.ascontiguousarray(np.concatenate(Ws))
    q = np.ascontiguousarray(np.concatenate(qs))
    mu = np.array(mus)
    o = oracle.Options.local(565)
    o.iparam[9] = 1
    p = local_params_from(o, 565)
    assert p.rho_strategy == 1
    state = np.zeros(4 * n)
    info = np.zeros(n, dtype=np.int32)
    rg = np.zeros(3 * n)
    assert lib.fc3d_hip_local_solve(n, N.dptr(W), N.dptr(q), N.dptr(mu), N.dptr(rg), p,
                                    N.dptr(state), 1, N.iptr(info)) == 0, capi.last_error()
    L = oracle.load()
    same = 0
    for k in range(n):
        st = np.zeros(4)
        w = W[9 * k:9 * k + 9].copy()
        assert L.oracle_local_state_init(oracle.d(w), o.p, oracle.d(st)) == 0
        rho0 = st.copy()
        x = np.zeros(3)
        L.oracle_local_solve(oracle.d(w), oracle.d(q[3 * k:3 * k + 3].copy()), mu[k],
                             oracle.d(x), o.p, oracle.d(st))
        np.testing.assert_allclose(state[4 * k + 1:4 * k + 4], rho0[1:], rtol=4 * 2.0 ** -52)
        np.testing.assert_allclose(rg[3 * k:3 * k + 3], x, rtol=1e-12, atol=1e-14)
        same += int(np.array_equal(state[4 * k + 1:4 * k + 4], rho0[1:]))
    # the diagonal blocks take the exact branch (no trigonometry)
    assert same >= n // 4


def test_fp32_local_solve_against_fp64(oracle, lib):
    """The FP32 sweeps' local solve (undamped AC Newton on float inputs, the
    hardware reciprocal and square root, the adjugate 3x3 solve with its FP64
    redo for near-singular systems) against the FP64 solve of the same
    contacts, to FP32 accuracy, and the local error of the FP32 solutions
    evaluated in FP64 by the oracle's unitary error.  The second group has a
    second tangent of stiffness 1e-9 and no load along it: those contacts
    stick, so the Newton matrix is -rho W with det ~ 1e-9, which the
    adjugate test hands to the FP64 factorisation; their solution stays
    bounded."""
    rng = np.random.default_rng(53)
    n_good, n_sing = 2000, 400
    Ws, qs, mus = [], [], []
    for k in range(n_good + n_sing):
        if k < n_good:
            M = rng.normal(size=(3, 3))
            W = M @ M.T + rng.uniform(0.1, 3) * np.eye(3)
        else:
            wn, a = rng.uniform(0.5, 2.0, size=2)
            c = rng.uniform(-0.3, 0.3)
            W = np.array([[wn, c, 0.0], [c, a, 0.0], [0.0, 0.0, 1e-9]])
        Ws.append(W.reshape(-1, order="F"))
        q = rng.normal(size=3)
        q[0] = -abs(q[0]) - 0.1  # in contact: the Newton branch, not the take-off
        if k >= n_good:
            q[1] *= 0.05  # within the friction cone: sticking
            q[2] = 0.0
        qs.append(q)
        mus.append(rng.uniform(0.1, 0.9))
    n = n_good + n_sing
    W = np.ascontiguousarray(np.concatenate(Ws))
    q = np.ascontiguousarray(np.concatenate(qs))
    mu = np.array(mus)

    def run(precision):
        p = N.hip_params(local_solver=550, local_tol=1e-14, local_max_iter=100,
                         precision=precision, fp32_local_solver=550, fp32_local_tol=1e-7)
        r = np.zeros(3 * n)
        state = np.zeros(4 * n)
        info = np.zeros(n, dtype=np.int32)
        assert lib.fc3d_hip_local_solve(n, N.dptr(W), N.dptr(q), N.dptr(mu), N.dptr(r), p,
                                        N.dptr(state), 1, N.iptr(info)) == 0, capi.last_error()
        return r, info

    r64, i64 = run(0)
    r32, i32 = run(1)
    L = oracle.load()

    def local_error(k, x):
        w = W[9 * k:9 * k + 9].reshape(3, 3, order="F")
        u = w @ x + q[3 * k:3 * k + 3]
        e = np.zeros(1)
        L.oracle_unitary_compute_and_add_error(oracle.d(x.copy()), oracle.d(u), mu[k],
                                               oracle.d(e))
        return np.sqrt(e[0]) / np.linalg.norm(q[3 * k:3 * k + 3])

    worst_good = 0.0
    worst_err = 0.0
    for k in range(n):
        x32 = r32[3 * k:3 * k + 3]
        x64 = r64[3 * k:3 * k + 3]
        if i64[k] == 0 and i32[k] == 0:
            worst_good = max(worst_good, np.linalg.norm(x32 - x64) /
                             max(np.linalg.norm(x64), 1e-30))
        if i64[k] == 0:
            # where the undamped Newton fails in FP64 too (a few contacts,
            # r_n < 0), FP32 follows the same iterates; judged where it converges
            worst_err = max(worst_err, local_error(k, x32))
    print(f"FP32 vs FP64 local solve: worst relative difference {worst_good:.2e}, "
          f"worst local error {worst_err:.2e}; converged FP32 {(i32 == 0).mean():.4f}, "
          f"FP64 {(i64 == 0).mean():.4f}", flush=True)
    assert worst_good < 1e-4  # measured 6.2e-6
    assert worst_err < 1e-5   # measured 6.9e-7; FP64's own is ~1e-16
    assert (i32 == 0).mean() > 0.99


@pytest.mark.parametrize("scale", [(1.0, 1e3, 1.0), (1.0, 1.0, 1e3), (1e3, 1.0, 1e-3),
                                   (1.0, 1.0, 0.0), (1.0, 1e-9, 1e-9)])
@pytest.mark.parametrize("sid", [565, 551, 550])
def test_local_solve_pivots_and_singular_blocks(oracle, lib, sid, scale):
    """Blocks D S D whose Newton matrices pivot on each of their rows, and
    singular or nearly singular ones (a zero or tiny scale), against the
    oracle bit for bit."""
    rng = np.random.default_rng(61)
    n = 400
    D = np.diag(scale)
    M = rng.normal(size=(n, 3, 3))
    S = D @ (M @ M.transpose(0, 2, 1) + 0.5 * np.eye(3)) @ D
    q = rng.normal(size=(n, 3))
    q[:, 0] = -abs(q[:, 0])
    W = np.ascontiguousarray(S.transpose(0, 2, 1)).reshape(-1)
    qf, mu, r = np.ascontiguousarray(q).reshape(-1), rng.uniform(0.1, 0.9, n), np.zeros(3 * n)
    r[::6] = rng.uniform(0.0, 1.0, n // 2)
    o = oracle.Options.local(sid)
    p = local_params_from(o, sid)
    rg, state, info = r.copy(), np.zeros(4 * n), np.zeros(n, dtype=np.int32)
    assert lib.fc3d_hip_local_solve(n, N.dptr(W), N.dptr(qf), N.dptr(mu), N.dptr(rg), p,
                                    N.dptr(state), 1, N.iptr(info)) == 0, capi.last_error()
    L = oracle.load()
    for k in range(n):
        st = np.zeros(4)
        w = W[9 * k:9 * k + 9].copy()
        L.oracle_local_state_init(oracle.d(w), o.p, oracle.d(st))
        x = r[3 * k:3 * k + 3].copy()
        L.oracle_local_solve(oracle.d(w), oracle.d(qf[3 * k:3 * k + 3].copy()), mu[k],
                             oracle.d(x), o.p, oracle.d(st))
        np.testing.assert_array_equal(rg[3 * k:3 * k + 3], x, err_msg=f"contact {k}")
        np.testing.assert_array_equal(state[4 * k:4 * k + 4], st)
