// fc3d_transfer.hpp — reactions and velocities between the caller's arrays
// (three values a contact, in the caller's order) and the resident slots.
//
// The permutation runs on the device, so a transfer moves the 24 bytes a
// contact that the caller sees and the host touches them once, in order.  (As
// a host loop over a downloaded copy of the slots it took ~9 ms for each
// vector of 1M contacts, an eighth of the fast method's solve.)
#pragma once
#include <mutex>
#include <vector>

#include "fc3d_internal.hpp"

namespace fc3d {

// out[i] = slots[o2s[i]] for every contact: bound by the gather of one 32-byte
// vector a contact.
static __global__ void k_slots_to_contacts(int n, const int* __restrict__ o2s,
                                           const double4* __restrict__ slots,
                                           double* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double4 v = slots[o2s[i]];
  out[3 * (size_t)i] = v.x;
  out[3 * (size_t)i + 1] = v.y;
  out[3 * (size_t)i + 2] = v.z;
}

// slots[s] = in[s2o[s]], zero for padding slots.
static __global__ void k_contacts_to_slots(int nslots, const int* __restrict__ s2o,
                                           const double* __restrict__ in,
                                           double4* __restrict__ slots) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nslots) return;
  const int i = s2o[s];
  slots[s] = i < 0 ? make_double4(0.0, 0.0, 0.0, 0.0)
                   : make_double4(in[3 * (size_t)i], in[3 * (size_t)i + 1],
                                  in[3 * (size_t)i + 2], 0.0);
}

// Device side of a handle's transfers, allocated on first use.  Threads that
// read one handle at the same time take turns with its buffer.
struct Transfer {
  std::mutex turn;
  int *o2s = nullptr, *s2o = nullptr;
  double* buf = nullptr;  // three values a contact

  int ensure(const std::vector<int>& orig2slot, const std::vector<int>& slot2orig) {
    std::lock_guard<std::mutex> lock(turn);
    if (buf) return 0;
    const size_t n = orig2slot.size(), ns = slot2orig.size();
    if (!o2s) FC3D_HIP_TRY(hipMalloc(&o2s, sizeof(int) * n));
    if (!s2o) FC3D_HIP_TRY(hipMalloc(&s2o, sizeof(int) * ns));
    FC3D_HIP_TRY(hipMemcpy(o2s, orig2slot.data(), sizeof(int) * n, hipMemcpyHostToDevice));
    FC3D_HIP_TRY(hipMemcpy(s2o, slot2orig.data(), sizeof(int) * ns, hipMemcpyHostToDevice));
    FC3D_HIP_TRY(hipMalloc(&buf, sizeof(double) * 3 * n));
    return 0;
  }
  int to_host(int n, const double4* slots, double* out, hipStream_t s) {
    std::lock_guard<std::mutex> lock(turn);
    hipLaunchKernelGGL(k_slots_to_contacts, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n,
                       (const int*)o2s, slots, buf);
    FC3D_HIP_TRY(hipGetLastError());
    FC3D_HIP_TRY(hipMemcpyAsync(out, buf, sizeof(double) * 3 * (size_t)n, hipMemcpyDeviceToHost,
                                s));
    FC3D_HIP_TRY(hipStreamSynchronize(s));
    return 0;
  }
  int to_device(int n, int nslots, const double* in, double4* slots, hipStream_t s) {
    std::lock_guard<std::mutex> lock(turn);
    FC3D_HIP_TRY(hipMemcpyAsync(buf, in, sizeof(double) * 3 * (size_t)n, hipMemcpyHostToDevice,
                                s));
    hipLaunchKernelGGL(k_contacts_to_slots, dim3((unsigned)((nslots + 255) / 256)), dim3(256), 0,
                       s, nslots, (const int*)s2o, (const double*)buf, slots);
    FC3D_HIP_TRY(hipGetLastError());
    FC3D_HIP_TRY(hipStreamSynchronize(s));
    return 0;
  }
  void release() {
    void* p[] = {o2s, s2o, buf};
    for (void* q : p)
      if (q) hipFree(q);
  }
};

}  // namespace fc3d
