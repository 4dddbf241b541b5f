// fdtd_stream_dev.h -- what the FP64 row-streaming kernels share (fdtd_stream.hip,
// fdtd_stream_split.hip): complex arithmetic, lane shifts, scalar loads, the LDS
// barrier and the covering of an axis with strips.
#ifndef FDTD_STREAM_DEV_H
#define FDTD_STREAM_DEV_H

#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

typedef double2 D2;

#ifdef __HIP_DEVICE_COMPILE__
#define CAS_(T) __attribute__((address_space(4))) T
#else
#define CAS_(T) T
#endif
#define CAS(T) const CAS_(T) *
// read-only data at a wavefront-uniform address: scalar loads
template <class T>
__device__ __forceinline__ T cload(const T *p)
{
  return *(CAS(T))p;
}

__device__ __forceinline__ D2 d2(double x, double y) { return make_double2(x, y); }
__device__ __forceinline__ D2 cload2(const D2 *p)
{
  CAS(double) q = (CAS(double))p;
  return d2(q[0], q[1]);
}
__device__ __forceinline__ D2 add(D2 a, D2 b) { return d2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ D2 sub(D2 a, D2 b) { return d2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ D2 mul(double s, D2 a) { return d2(s * a.x, s * a.y); }
__device__ __forceinline__ D2 mad(double s, D2 a, D2 b) { return d2(fma(s, a.x, b.x), fma(s, a.y, b.y)); }
__device__ __forceinline__ D2 cmulp(D2 a, D2 b) { return d2(fma(a.x, b.x, -(a.y * b.y)), fma(a.x, b.y, a.y * b.x)); }
// the value of the lane below (0x138 wave_shr:1) / above (0x130 wave_shl:1); 0 enters at the end
template <int CTRL>
__device__ __forceinline__ double dppd(double v)
{
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ D2 below(D2 v) { return d2(dppd<0x138>(v.x), dppd<0x138>(v.y)); }
__device__ __forceinline__ D2 above(D2 v) { return d2(dppd<0x130>(v.x), dppd<0x130>(v.y)); }

// conditions of the row loop's side paths: their code is laid out after the loop's, so
// that a row's turn runs through without taken branches
#define RARE(x) __builtin_expect(!!(x), 0)

// Workgroup barrier that orders LDS accesses only.  __syncthreads() also waits for
// every outstanding global load and store, so the rows fetched ahead would be
// waited for in each iteration (1.55 us an iteration instead of the rows' own work).
__device__ __forceinline__ void lds_barrier()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Cover the core [lo, hi) of an axis of n entries (ring at 0 and n - 1) with blocks of
// B entries: hl entries of halo below and hu above, none where the block reaches the ring.
struct Span {
  int c0, c1, b0;
};
static inline std::vector<Span> cover_cols(int lo, int hi, int n, int B, int hl, int hu)
{
  std::vector<Span> v;
  for (int c = lo; c < hi;) {
    const int b0 = c == 1 ? 0 : c - hl;
    const int e = std::min(hi, b0 + B >= n ? n - 1 : b0 + B - hu);
    v.push_back({c, e, b0});
    c = e;
  }
  return v;
}

#endif
