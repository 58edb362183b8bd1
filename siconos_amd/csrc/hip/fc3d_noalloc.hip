// fc3d_noalloc.hip — fc3d_compute_error on caller-owned device arrays, with
// no allocation (fc3d_hip_compute_error_device in fc3d_hip.h).
//
// The residual of fc3d_compute_error.c:70-122: u = q + W r with each row's
// blocks in their stored order (the order SBM_gemv_3x3 adds them in,
// SparseBlockMatrix.c:360-419), the unitary error of every contact, and the
// norms of r and u.  One thread per contact, one partial sum triple per wave
// of 64 contacts, then one workgroup adds the wave partials in a fixed order.
//
// The wave partials live in `scratch`, a file-scope device array of
// NOALLOC_MAX_WAVES triples (1.5 MiB per GPU, held until the process ends), so
// a call allocates nothing.  Host code never passes the array's name to a
// kernel: its device address is taken once per device with
// hipGetSymbolAddress, with that device current, and kept in g_scratch.  Every
// call on a GPU shares that GPU's array, so calls that overlap on one GPU
// (two host threads, or two streams) race; the array keeps the last call's
// partials, and every partial is rewritten before it is read.
#include <cmath>
#include <mutex>

#include "fc3d_internal.hpp"
#include "fc3d_sweep.hpp"

namespace fc3d {

constexpr int NOALLOC_MAX_CONTACTS = 1 << 22;
constexpr int NOALLOC_MAX_WAVES = NOALLOC_MAX_CONTACTS / 64;
constexpr int NOALLOC_MAX_DEVICES = 64;

static __device__ __align__(256) double scratch[3 * NOALLOC_MAX_WAVES];

static std::mutex g_scratch_lock;
static double* g_scratch[NOALLOC_MAX_DEVICES] = {};

// The scratch array's address on the current device, taken on first use.
static int scratch_on(int device, double** out) {
  std::lock_guard<std::mutex> lock(g_scratch_lock);
  if (!g_scratch[device]) {
    void* p = nullptr;
    FC3D_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch[device] = static_cast<double*>(p);
  }
  *out = g_scratch[device];
  return 0;
}

// The row sum of contact i, block by block in the stored order.  Row ranges
// and column indices are checked against nnzb and nc: a row with an entry
// outside them is bad, and gets a NaN velocity (and so a NaN error) instead of
// reading out of bounds.
__device__ __forceinline__ void add_block(const double* w, const double* __restrict__ r, int64_t j,
                                          double* u) {
  const double v[3] = {r[3 * j], r[3 * j + 1], r[3 * j + 2]};
  mvp3x3<double>(w, v, u);
}

// WPR waves per 64 contacts.  Their rows are one range of the CSR, which the
// waves walk CSR_CHUNK blocks a wave at a time: coalesced 512-byte loads of the
// blocks into LDS, a lane per block for its products with the neighbour's
// reaction (every gather of a chunk in flight), then a lane of the first wave
// per row adds its row's products in their order.  HBM bounds a large problem
// (0.85 GB for 1M contacts with 10.5M blocks): 1.8 TB/s when a lane walked its
// own row, 72 bytes in another 128-byte line than its neighbours at every step
// (480 us a call, both kernels), 4.1 TB/s so (207 us; a copy reaches 5.1).  A
// wave with a bad row walks its rows from memory: every form of row pointers
// that was accepted still is.
//
// A problem that leaves the GPU's wave slots empty is bound by the chain of a
// wave's chunks, and four waves per 64 contacts walk a quarter of it each; a
// larger one has the waves, and gains by not waiting for each other.  us a call
// (a lane per row / one wave / four waves): 1000 contacts 15.4 / 24.4 / 11.7,
// 16k 16.3 / 24.9 / 12.0, 64k 28.1 / 27.5 / 22.6, 256k 122 / 61.7 / 55.2, 512k
// 249 / 111 / 119, 1M 480 / 207 / 226.
constexpr int CSR_CHUNK = 128;
constexpr int CSR_WIDE_CONTACTS = 1 << 18;
template <int WPR>
__global__ __launch_bounds__(256) void k_csr_residual(int nc, int64_t nnzb,
                                                      const int64_t* __restrict__ rp,
                                                      const int64_t* __restrict__ ci,
                                                      const double* __restrict__ blocks,
                                                      const double* __restrict__ q,
                                                      const double* __restrict__ mu,
                                                      const double* __restrict__ r,
                                                      double* __restrict__ u_out,
                                                      double* __restrict__ part) {
  constexpr int T = 64 * WPR, CHUNK = CSR_CHUNK * WPR, G = 4 / WPR;
  __shared__ double sblk[G][CHUNK * 9];
  const int group = threadIdx.x / T, t = threadIdx.x % T, lane = threadIdx.x & 63;
  const int i = (blockIdx.x * G + group) * 64 + lane;
  auto sync = [] {
    if constexpr (WPR == 1) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    } else {
      __syncthreads();  // G = 1: the block's waves hold the same rows and walk the same chunks
    }
  };
  double e2 = 0.0, r2 = 0.0, u2 = 0.0;
  double u[3] = {0.0, 0.0, 0.0};
  int64_t k0 = 0, k1 = 0;
  bool bad = false;
  if (i < nc) {
#pragma unroll
    for (int e = 0; e < 3; e++) u[e] = q[3 * (size_t)i + e];
    k0 = rp[i];
    k1 = rp[i + 1];
    bad = k0 < 0 || k1 > nnzb || k1 < k0;
  }
  // the wave's range, when its rows follow each other inside [0, nnzb]
  const int last = min(63, nc - 1 - (i - lane));  // last lane with a row (< 0: none)
  const bool plain = __builtin_amdgcn_ballot_w64(bad) == 0;
  const int64_t kb = __shfl(k0, 0, 64), ke = last >= 0 ? __shfl(k1, last, 64) : 0;
  if (plain && last >= 0) {
    int64_t k = k0;
    for (int64_t c0 = kb; c0 < ke; c0 += CHUNK) {
      const int n = (int)min((int64_t)CHUNK, ke - c0);
      const double* __restrict__ src = blocks + 9 * c0;
      double b9[CSR_CHUNK * 9 / 64], v[CSR_CHUNK / 64][3];
      int64_t jc[CSR_CHUNK / 64];
#pragma unroll
      for (int x = 0; x < CSR_CHUNK / 64; x++)
        jc[x] = x * T + t < n ? ci[c0 + x * T + t] : 0;
#pragma unroll
      for (int x = 0; x < CSR_CHUNK * 9 / 64; x++)
        if (x * T + t < 9 * n) b9[x] = src[x * T + t];
#pragma unroll
      for (int x = 0; x < CSR_CHUNK / 64; x++) {
        const bool ok = jc[x] >= 0 && jc[x] < nc;
#pragma unroll
        for (int e = 0; e < 3; e++) {
          const double y = r[3 * (size_t)(ok ? jc[x] : 0) + e];
          v[x][e] = ok ? y : NAN;  // a column out of range: the row is NaN
        }
      }
#pragma unroll
      for (int x = 0; x < CSR_CHUNK * 9 / 64; x++)
        if (x * T + t < 9 * n) sblk[group][x * T + t] = b9[x];
      sync();
#pragma unroll
      for (int x = 0; x < CSR_CHUNK / 64; x++)
        if (x * T + t < n) {
          double* b = &sblk[group][9 * (x * T + t)];
#pragma unroll
          for (int e = 0; e < 9; e++) b[e] = b[e] * v[x][e / 3];
        }
      sync();
      // u += W r_j as mvp3x3 adds it: column after column
      for (const int64_t stop = WPR == 1 || t < 64 ? min(k1, c0 + n) : k; k < stop; k++) {
        const double* b = &sblk[group][9 * (int)(k - c0)];
#pragma unroll
        for (int e = 0; e < 9; e++) u[e % 3] += b[e];
      }
      sync();  // the chunk is read before the next one lands
    }
  } else if (i < nc && t < 64) {
    for (int64_t k = bad ? k1 : k0; k < k1; k++) {
      const int64_t j = ci[k];
      if (j < 0 || j >= nc) {
        bad = true;
        break;
      }
      double w[9];
#pragma unroll
      for (int e = 0; e < 9; e++) w[e] = blocks[9 * k + e];
      add_block(w, r, j, u);
    }
  }
  if (t >= 64) return;  // the first wave has the rows
  if (i < nc) {
    if (bad) u[0] = u[1] = u[2] = NAN;
#pragma unroll
    for (int e = 0; e < 3; e++) u_out[3 * (size_t)i + e] = u[e];
    const double rv[3] = {r[3 * (size_t)i], r[3 * (size_t)i + 1], r[3 * (size_t)i + 2]};
    e2 = unitary_error<double>(rv, u, mu[i]);
    r2 = rv[0] * rv[0] + rv[1] * rv[1] + rv[2] * rv[2];
    u2 = u[0] * u[0] + u[1] * u[1] + u[2] * u[2];
  }
  e2 = wave_sum(e2);
  r2 = wave_sum(r2);
  u2 = wave_sum(u2);
  if ((threadIdx.x & 63) == 0) {
    const size_t wv = (size_t)i >> 6;
    part[3 * wv] = e2;
    part[3 * wv + 1] = r2;
    part[3 * wv + 2] = u2;
  }
}

// fc3d_compute_error.c:100-115: the error relative to max(|q|, |r|, |u|).
__global__ __launch_bounds__(1024) void k_csr_residual_end(const double* __restrict__ part,
                                                           int nwaves, double norm,
                                                           double* __restrict__ error) {
  __shared__ double sh[3 * 16];
  double sums[3];
  block_sums<3>(part, nwaves, sh, sums);
  if (threadIdx.x != 0) return;
  double err = sqrt(sums[0]);
  const double scale = fmax(norm, fmax(sqrt(sums[1]), sqrt(sums[2])));
  if (fabs(scale) > DBL_EPSILON) err /= scale;
  *error = err;
}

}  // namespace fc3d

extern "C" {

int fc3d_hip_compute_error_device(int nc, int64_t nnzb, const int64_t* row_ptr,
                                  const int64_t* col_idx,
                                  const double* blocks, const double* q, const double* mu,
                                  const double* reaction, double norm, double* velocity,
                                  double* error, int device, void* stream) {
  using namespace fc3d;
  if (!row_ptr || !col_idx || !blocks || !q || !mu || !reaction || !velocity || !error)
    return NUMERICS_ERR_NULL_POINTER;
  if (nc < 1 || nc > NOALLOC_MAX_CONTACTS) {
    set_error("fc3d_hip_compute_error_device: %d contacts, outside [1, %d] (the size of the "
              "library's static scratch array)", nc, NOALLOC_MAX_CONTACTS);
    return NUMERICS_ERR_INVALID_ARGUMENT;
  }
  if (nnzb < 0) {
    set_error("fc3d_hip_compute_error_device: nnzb %lld < 0", (long long)nnzb);
    return NUMERICS_ERR_INVALID_ARGUMENT;
  }
  if (!(norm >= 0.0) || !std::isfinite(norm)) {
    set_error("fc3d_hip_compute_error_device: norm %g is not a finite value >= 0", norm);
    return NUMERICS_ERR_INVALID_ARGUMENT;
  }
  if (device < 0 || device >= NOALLOC_MAX_DEVICES) {
    set_error("fc3d_hip_compute_error_device: device %d outside [0, %d)", device,
              NOALLOC_MAX_DEVICES);
    return NUMERICS_ERR_INVALID_ARGUMENT;
  }
  int rc = use_device(device);
  if (rc) return rc;
  double* part = nullptr;
  if ((rc = scratch_on(device, &part))) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int nwaves = (nc + 63) / 64;
  const bool wide = nc <= CSR_WIDE_CONTACTS;
  hipLaunchKernelGGL(wide ? k_csr_residual<4> : k_csr_residual<1>,
                     dim3((unsigned)(wide ? nwaves : (nwaves + 3) / 4)), dim3(256), 0, s, nc, nnzb,
                     row_ptr, col_idx, blocks, q, mu, reaction, velocity, part);
  hipLaunchKernelGGL(k_csr_residual_end, dim3(1), dim3(1024), 0, s, (const double*)part, nwaves,
                     norm, error);
  FC3D_HIP_TRY(hipGetLastError());
  return 0;
}

}  // extern "C"
