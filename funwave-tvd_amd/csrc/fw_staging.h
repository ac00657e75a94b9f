// fw_staging.h -- copies between the caller's (pageable) host arrays and the
// GPU, by kernels that read and write a ring of mapped pinned memory.
//
// What bounds them: the link (about 50 GB/s) and the CPU's own copy (80 GB/s
// in cache); the runtime's pageable copies take 50 to 80 us on top and its
// pitched ones go row by row (0.6 GB/s at 1024 x 768).  Here a kernel moves
// 512 KB between a pitched field and one slot of the ring and then publishes
// the slot's number, so the CPU copies one slot while the link carries the
// next; there is no call into the copy engine and no stream synchronisation.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstdint>
#include <cstring>

namespace fws {

// A launch that returns its own status: what hipGetLastError gives may be the
// error of an earlier, unrelated call of this thread, and asking clears it.
template <class T>
struct Same {
  using type = T;
};
template <class... P>
hipError_t start(void (*k)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t s, typename Same<P>::type... a) {
  void *args[] = {(void *)&a...};
  return hipLaunchKernel((const void *)k, grid, block, args, lds, s);
}

// Slots are read and written with system-scope accesses, which pass the caches
// by; once they have completed (the wait, in every wave), one counter and one
// store tell the host.  With a system-scope fence in every wave instead, which
// also writes caches back, a slot took 13.4 us down (16.6 with 128 workgroups).
__device__ __forceinline__ void slot_done(unsigned *count, uint64_t *flag, uint64_t seq) {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x == 0 && atomicAdd(count, 1u) == gridDim.x - 1) {
    *count = 0u;
    __hip_atomic_store(flag, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}
// n elements of rows of w from element off of row row0 on (dst, src: the row's
// start) := a slot, dense
template <class T>
__global__ void __launch_bounds__(256) k_slot_up(T *__restrict__ dst, size_t dp, const uint64_t *slot, uint32_t w,
                                                 uint32_t off, uint32_t n, unsigned *count, uint64_t *flag,
                                                 uint64_t seq) {
  constexpr uint32_t PER = 8 / sizeof(T);
  const uint32_t step = gridDim.x * 256u, nw = (n + PER - 1) / PER;
  for (uint32_t k0 = blockIdx.x * 256u + threadIdx.x; k0 < nw; k0 += 4 * step) {
    uint64_t v[4] = {};
#pragma unroll
    for (int q = 0; q < 4; q++)  // (not clamped: many loads of one host address take turns, 30 us a slot)
      if (k0 + q * step < nw)
        v[q] = __hip_atomic_load(slot + k0 + q * step, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (uint32_t p = 0; p < PER; p++) {
        const uint32_t k = (k0 + q * step) * PER + p, e = off + k;
        if (k < n) dst[(size_t)(e / w) * dp + e % w] = (T)(v[q] >> (32 * p));
      }
  }
  slot_done(count, flag, seq);
}
template <class T>
__global__ void __launch_bounds__(256) k_slot_down(uint64_t *slot, const T *__restrict__ src, size_t sp, uint32_t w,
                                                   uint32_t off, uint32_t n, unsigned *count, uint64_t *flag,
                                                   uint64_t seq) {
  constexpr uint32_t PER = 8 / sizeof(T);
  const uint32_t step = gridDim.x * 256u, nw = (n + PER - 1) / PER;
  for (uint32_t k0 = blockIdx.x * 256u + threadIdx.x; k0 < nw; k0 += 4 * step) {
    uint64_t v[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      v[q] = 0;
#pragma unroll
      for (uint32_t p = 0; p < PER; p++) {
        const uint32_t e = off + min((k0 + q * step) * PER + p, n - 1);
        v[q] |= (uint64_t)src[(size_t)(e / w) * sp + e % w] << (32 * p);
      }
    }
#pragma unroll
    for (int q = 0; q < 4; q++)
      if (k0 + q * step < nw)
        __hip_atomic_store(slot + k0 + q * step, v[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  slot_done(count, flag, seq);
}

// A ring of one context or network, freed with it.
class Staging {
 public:
  // the ring, unless it is there: 0.1 ms, which a network spends when it is
  // made and a context at its first copy
  hipError_t init() {
    if (ring) return hipSuccess;
    char *r = nullptr;
    unsigned *c = nullptr;
    const unsigned zero[kSlots] = {};
    hipError_t e = hipHostMalloc((void **)&r, kSlots * kSlot + 64, hipHostMallocMapped | hipHostMallocCoherent);
    if (e == hipSuccess) e = hipHostGetDevicePointer((void **)&ring_dev, r, 0);
    if (e == hipSuccess) e = hipMalloc((void **)&c, sizeof zero);
    if (e == hipSuccess) e = hipMemcpy(c, zero, sizeof zero, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
      if (r) (void)hipHostFree(r);
      if (c) (void)hipFree(c);
      return e;
    }
    memset(r + kSlots * kSlot, 0, 64);
    flag_dev = (uint64_t *)(ring_dev + kSlots * kSlot);
    ring = r;
    count = c;
    return hipSuccess;
  }
  // h rows of w elements: dst (device, pitch dp) := src (host, dense), queued
  // on s; src may be changed on return.  A slot's flag says that it has been
  // read, not that dst can be read from another stream: an XCD's cache is
  // written back when the kernel ends.
  template <class T>
  hipError_t up(T *dst, size_t dp, const T *src, uint32_t w, size_t h, hipStream_t s) {
    hipError_t e = init();
    const size_t n = (size_t)w * h, per = kSlot / sizeof(T);
    for (size_t k = 0; e == hipSuccess && k < n; k += per) {
      const size_t c = std::min(per, n - k);
      const int q = (int)(next % kSlots);
      if ((e = wait(q, s)) != hipSuccess) break;  // the slot's last copy
      memcpy(ring + q * kSlot, src + k, c * sizeof(T));
      ++next;
      e = start(k_slot_up<T>, dim3(kWg), dim3(256), 0, s, dst + k / w * dp, dp, slot(q), w, (uint32_t)(k % w),
                (uint32_t)c, count + q, flag_dev + q, next);
      if (e == hipSuccess) busy[q] = next;
    }
    return e;
  }
  // dst (host, dense) := src (device, pitch sp); complete on return, and with
  // it everything queued on s before
  template <class T>
  hipError_t down(T *dst, const T *src, size_t sp, uint32_t w, size_t h, hipStream_t s) {
    hipError_t e = init();
    const size_t n = (size_t)w * h, per = kSlot / sizeof(T), nc = (n + per - 1) / per;
    const uint64_t first = next;
    size_t issued = 0;
    for (size_t k = 0; e == hipSuccess && k < nc; k++) {
      for (; e == hipSuccess && issued < std::min(nc, k + kSlots); issued++) {
        const int q = (int)(next % kSlots);
        if ((e = wait(q, s)) != hipSuccess) break;
        const size_t k0 = issued * per;
        ++next;
        e = start(k_slot_down<T>, dim3(kWg), dim3(256), 0, s, slot(q), src + k0 / w * sp, sp, w, (uint32_t)(k0 % w),
                  (uint32_t)std::min(per, n - k0), count + q, flag_dev + q, next);
        if (e == hipSuccess) busy[q] = next;
      }
      if (e != hipSuccess) break;
      const int q = (int)((first + k) % kSlots);
      if ((e = wait(q, s)) != hipSuccess) break;
      memcpy(dst + k * per, ring + q * kSlot, std::min(per, n - k * per) * sizeof(T));
    }
    return e;
  }
  // (after the owner's stream has been synchronised)
  void release() {
    if (ring) (void)hipHostFree(ring);
    if (count) (void)hipFree(count);
    ring = nullptr;
    count = nullptr;
  }

 private:
  static constexpr int kSlots = 4;
  static constexpr size_t kSlot = 512u << 10;
  static constexpr unsigned kWg = 64;  // workgroups of a slot's copy
  char *ring = nullptr, *ring_dev = nullptr;  // kSlots slots, then a flag each
  uint64_t *flag_dev = nullptr;
  unsigned *count = nullptr;
  uint64_t next = 0;            // copies issued
  uint64_t busy[kSlots] = {};   // number of the slot's copy in flight, 0: none

  uint64_t *slot(int q) { return (uint64_t *)(ring_dev + q * kSlot); }
  // until the slot is free.  A wait longer than 20 ms goes to the stream,
  // whose error it then reports.
  hipError_t wait(int q, hipStream_t s) {
    if (!busy[q]) return hipSuccess;
    const uint64_t *f = (const uint64_t *)(ring + kSlots * kSlot) + q;
    const auto t0 = std::chrono::steady_clock::now();
    while (__atomic_load_n(f, __ATOMIC_ACQUIRE) != busy[q]) {
      for (int k = 0; k < 32; k++) __builtin_ia32_pause();
      if (std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(20)) {
        const hipError_t e = hipStreamSynchronize(s);
        if (e != hipSuccess) return e;
        if (__atomic_load_n(f, __ATOMIC_ACQUIRE) != busy[q]) return hipErrorUnknown;
      }
    }
    busy[q] = 0;
    return hipSuccess;
  }
};

}  // namespace fws
