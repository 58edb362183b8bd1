"""fc3d_hip_compute_error_device (no allocation, caller-owned device arrays)
against fc3d_hip_compute_error on the same problems: velocities bit for bit
(both add each row's blocks in the stored order), the error to 1e-12 relative
(the partial sums are added in another order).  Two calls in a row, the second
on a smaller problem, as the static scratch array keeps the first call's
partials."""
import ctypes as C

import numpy as np
import pytest

from siconos_amd import capi
from siconos_amd import numerics as N

pytestmark = pytest.mark.gpu


class _Hip:
    """Device buffers through the HIP runtime (the test's own allocations)."""

    def __init__(self):
        self.lib = C.CDLL("libamdhip64.so")
        self.lib.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
        self.lib.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
        self.lib.hipFree.argtypes = [C.c_void_p]
        self.bufs = []

    def upload(self, a):
        a = np.ascontiguousarray(a)
        p = C.c_void_p()
        assert self.lib.hipMalloc(C.byref(p), max(a.nbytes, 8)) == 0
        assert self.lib.hipMemcpy(p, a.ctypes.data, a.nbytes, 1) == 0  # host to device
        self.bufs.append(p)
        return p.value

    def download(self, p, like):
        out = np.empty_like(like)
        assert self.lib.hipDeviceSynchronize() == 0
        assert self.lib.hipMemcpy(out.ctypes.data, C.c_void_p(p), out.nbytes, 2) == 0
        return out

    def free(self):
        for p in self.bufs:
            self.lib.hipFree(p)
        self.bufs = []


def _device_call(W, q, mu, r, norm, nnzb=None):
    d = _Hip()
    try:
        u0 = np.full(3 * W.nc, -1.0)
        e0 = np.full(1, -1.0)
        ptrs = [d.upload(np.asarray(W.row_ptr, dtype=np.int64)),
                d.upload(np.asarray(W.col_idx, dtype=np.int64)),
                d.upload(np.asarray(W.values, dtype=np.float64)),
                d.upload(np.asarray(q, dtype=np.float64)), d.upload(np.asarray(mu, dtype=np.float64)),
                d.upload(np.asarray(r, dtype=np.float64))]
        pu, pe = d.upload(u0), d.upload(e0)
        rc = capi.load().fc3d_hip_compute_error_device(
            W.nc, int(W.nnzb) if nnzb is None else nnzb, *ptrs, norm, pu, pe, 0, None)
        u = d.download(pu, u0)
        e = d.download(pe, e0)
        return rc, u, float(e[0])
    finally:
        d.free()


def test_no_alloc_residual_matches_the_resident_one_twice():
    for nb, nc, seed in ((20_000, 50_000, 3), (3_000, 7_000, 4)):
        g = N.generate_random_pairs(nb, nc, 0.2, 0.5, seed)
        H = N.HipProblem(g.W, g.q, g.mu)
        # a reaction after a few sweeps: inside the cone, not a solution
        H.set_reaction(np.zeros(3 * nc))
        H.solve(N.hip_params(tol=1e-12, max_iter=5))
        r = H.reaction()
        norm = float(np.linalg.norm(g.q))
        e_ref = H.compute_error(norm)
        u_ref = H.velocity()
        rc, u, e = _device_call(g.W, g.q, g.mu, r, norm)
        print(f"{nc} contacts: error {e:.17g} (resident {e_ref:.17g})", flush=True)
        assert rc == 0, capi.last_error()
        np.testing.assert_array_equal(u, u_ref)
        assert e == pytest.approx(e_ref, rel=1e-12)


def test_no_alloc_residual_refuses_sizes_beyond_its_scratch():
    g = N.generate_random_pairs(300, 1000, 0.2, 0.5, 1)
    d = _Hip()
    p = d.upload(np.zeros(16))
    lib = capi.load()
    rc = lib.fc3d_hip_compute_error_device((1 << 22) + 1, 0, p, p, p, p, p, p, 1.0, p, p, 0, None)
    assert rc == -2 and "scratch" in capi.last_error()
    rc = lib.fc3d_hip_compute_error_device(g.nc, 0, p, p, p, p, p, p, -1.0, p, p, 0, None)
    assert rc == -2
    d.free()


@pytest.mark.parametrize("nc", [1, 63, 64, 65, 130, 300])
def test_no_alloc_residual_rows_of_every_length(nc):
    """Rows of 0 to 300 blocks (several of the kernel's chunks, a wave's rows
    ending inside one), then one row with a column out of range and one with a
    range past the end: those rows are NaN and the others keep their bits."""
    rng = np.random.default_rng(nc)
    per = rng.integers(0, 8, nc)
    per[rng.integers(nc)] = 300
    rp = np.concatenate([[0], np.cumsum(per)])
    ci = rng.integers(0, nc, rp[-1])
    blocks = rng.normal(size=(rp[-1], 9))
    q, r = rng.normal(size=3 * nc), rng.normal(size=3 * nc)
    W = N.SparseBlock3(rp, ci, blocks.reshape(-1))
    rc, u, err = _device_call(W, q, np.full(nc, 0.4), r, 1.0)
    want = q.copy().reshape(-1, 3)
    for i in range(nc):
        for k in range(rp[i], rp[i + 1]):
            for j in range(3):  # column after column, as mvp3x3
                want[i] += blocks[k, 3 * j:3 * j + 3] * r[3 * ci[k] + j]
    assert rc == 0 and np.isfinite(err)
    np.testing.assert_array_equal(u, want.reshape(-1))
    row = int(np.argmax(per))
    bad = ci.copy()
    bad[rp[row] + 5] = nc
    rc, u, err = _device_call(N.SparseBlock3(rp, bad, blocks.reshape(-1)), q, np.full(nc, 0.4), r,
                              1.0)
    keep = np.repeat(np.arange(nc) != row, 3)
    assert rc == 0 and np.isnan(err) and np.isnan(u[~keep]).all()
    np.testing.assert_array_equal(u[keep], want.reshape(-1)[keep])
    past = W.row_ptr.copy()
    past[nc] += 1
    rc, u, err = _device_call(N.SparseBlock3(past, ci, blocks.reshape(-1)), q, np.full(nc, 0.4),
                              r, 1.0, nnzb=int(rp[-1]))
    assert rc == 0 and np.isnan(err) and np.isnan(u[-3:]).all()
    np.testing.assert_array_equal(u[:-3], want.reshape(-1)[:-3])


@pytest.mark.parametrize("nc", [262144, 262209])
def test_no_alloc_residual_on_both_sides_of_its_wide_form(nc):
    """The largest problem that takes four waves per 64 contacts and one that
    takes one wave, its last wave ragged: rows of 0 to 7 blocks and one of 300,
    then a column out of range, then row pointers that reach past the end and
    fall back, in a wave that has others after it in its workgroup: those two
    rows are NaN, and all others keep their bits, the wave's own too, which it
    walks from memory."""
    rng = np.random.default_rng(nc)
    per = rng.integers(0, 8, nc)
    per[nc - 70] = 300
    rp = np.concatenate([[0], np.cumsum(per)])
    ci = rng.integers(0, nc, rp[-1])
    blocks = rng.normal(size=(rp[-1], 9))
    q, r = rng.normal(size=3 * nc), rng.normal(size=3 * nc)
    want = q.copy().reshape(-1, 3)
    for k in range(300):
        rows = np.flatnonzero(per > k)
        b = blocks[rp[rows] + k]
        x = r.reshape(-1, 3)[ci[rp[rows] + k]]
        for j in range(3):  # column after column, as mvp3x3
            want[rows] += b[:, 3 * j:3 * j + 3] * x[:, j:j + 1]
    rc, u, err = _device_call(N.SparseBlock3(rp, ci, blocks.reshape(-1)), q, np.full(nc, 0.4), r,
                              1.0)
    assert rc == 0 and np.isfinite(err)
    np.testing.assert_array_equal(u, want.reshape(-1))
    ci[rp[nc - 70] + 200] = nc
    rc, u, err = _device_call(N.SparseBlock3(rp, ci, blocks.reshape(-1)), q, np.full(nc, 0.4), r,
                              1.0)
    assert rc == 0 and np.isnan(err) and np.isnan(u[3 * (nc - 70):3 * (nc - 69)]).all()
    keep = np.repeat(np.arange(nc) != nc - 70, 3)
    np.testing.assert_array_equal(u[keep], want.reshape(-1)[keep])
    ci[rp[nc - 70] + 200] = 0
    row = 64 * 4 * 17 + 64 + 20  # lane 20 of the second wave of a workgroup of four
    out = rp.copy()
    out[row + 1] = rp[-1] + 1
    rc, u, err = _device_call(N.SparseBlock3(out, ci, blocks.reshape(-1)), q, np.full(nc, 0.4), r,
                              1.0, nnzb=int(rp[-1]))
    keep = np.repeat(~np.isin(np.arange(nc), (row, row + 1, nc - 70)), 3)
    bad = slice(3 * row, 3 * (row + 2))
    assert rc == 0 and np.isnan(err) and np.isnan(u[bad]).all()
    np.testing.assert_array_equal(u[keep], want.reshape(-1)[keep])
