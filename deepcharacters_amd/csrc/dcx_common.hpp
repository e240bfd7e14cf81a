// Internal helpers shared by the dcx HIP translation units: status codes,
// the thread-local last-error message, launch checking and block reductions.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stddef.h>

#include "../../include/dcx.h"
#include "dcx_math.hpp"

namespace dcx {

// Records a formatted message as the calling thread's last error and
// returns `code`.  Never aborts the process.
dcx_status set_error(dcx_status code, const char* fmt, ...);

inline hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

// Checks the launch status of the kernel just enqueued on the stream.
dcx_status check_launch(const char* what);

#define DCX_REQUIRE(cond, ...)                                   \
  do {                                                           \
    if (!(cond)) return ::dcx::set_error(DCX_ERR_INVALID, __VA_ARGS__); \
  } while (0)

#define DCX_HIP(call)                                                          \
  do {                                                                         \
    hipError_t e_ = (call);                                                    \
    if (e_ != hipSuccess)                                                      \
      return ::dcx::set_error(DCX_ERR_HIP, "%s failed: %s", #call,             \
                              hipGetErrorString(e_));                          \
  } while (0)

inline unsigned int ceil_div(long long a, long long b) { return (unsigned int)((a + b - 1) / b); }

// Wave64 sum via cross-lane shuffles (result valid in every lane).
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Sums of eight values over a wavefront (all lanes active): lane l gets the sum
// of v[l & 7].  Each of the first three exchanges halves the values a lane
// carries, so this is 10 exchanges where eight separate sums take 48.
__device__ __forceinline__ float wave_sum8(const float* v) {
  const int lane = threadIdx.x & 63;
  float a[4], b[2];
#pragma unroll
  for (int i = 0; i < 4; ++i) {  // lanes 1 apart: keep v[2 i + bit 0]
    const float keep = lane & 1 ? v[2 * i + 1] : v[2 * i], give = lane & 1 ? v[2 * i] : v[2 * i + 1];
    a[i] = keep + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(give), 0xB1, 0xf, 0xf, false));
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {  // lanes 2 apart
    const float keep = lane & 2 ? a[2 * i + 1] : a[2 * i], give = lane & 2 ? a[2 * i] : a[2 * i + 1];
    b[i] = keep + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(give), 0x4E, 0xf, 0xf, false));
  }
  const float keep = lane & 4 ? b[1] : b[0], give = lane & 4 ? b[0] : b[1];
  float t = keep + __shfl_xor(give, 4, 64);
#pragma unroll
  for (int o = 8; o < 64; o <<= 1) t += __shfl_xor(t, o, 64);
  return t;
}

// s[0..n) += term(k) for k = k0, ..., k1 - 1, one after the other, for the lists
// that the lanes of a wavefront walk (a vertex's faces).  term(k, base, out)
// loads term k of the list whose owner passed `base`.  The terms of a short list
// are loaded kBatch at a time by its lane; a list longer than kLongList (a
// mesh's pole has a hundred faces and more) is loaded by the whole wavefront and
// added up in the same order, since a lane that walks it load by load is the
// last of its launch.  All lanes of the wavefront call it, those without a list
// with k0 == k1.
constexpr int kLongList = 16;
template <int n, int kBatch, class Term>
__device__ __forceinline__ void add_in_order(int k0, int k1, int base, float* s, Term term) {
  if (k1 - k0 <= kLongList)
    for (int k = k0; k < k1; k += kBatch) {
      float t[kBatch][n];
#pragma unroll
      for (int j = 0; j < kBatch; ++j) term(min(k + j, k1 - 1), base, t[j]);
#pragma unroll
      for (int j = 0; j < kBatch; ++j)
        if (k + j < k1) {
#pragma unroll
          for (int q = 0; q < n; ++q) s[q] += t[j][q];
        }
    }
  for (unsigned long long many = __ballot(k1 - k0 > kLongList); many; many &= many - 1) {
    const int src = __ffsll(many) - 1, lane = threadIdx.x & 63;
    const int c0 = __builtin_amdgcn_readlane(k0, src), c1 = __builtin_amdgcn_readlane(k1, src);
    const int cb = __builtin_amdgcn_readlane(base, src);
    float t[n], u[n];
#pragma unroll
    for (int q = 0; q < n; ++q) t[q] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s[q]), src));
    for (int k = c0; k < c1; k += 64) {
      term(min(k + lane, c1 - 1), cb, u);
      const int m = min(64, c1 - k);
      for (int j = 0; j < m; ++j) {
#pragma unroll
        for (int q = 0; q < n; ++q) t[q] += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(u[q]), j));
      }
    }
    if (lane == src) {
#pragma unroll
      for (int q = 0; q < n; ++q) s[q] = t[q];
    }
  }
}

// Smallest value of a group of 4, 16 or 64 lanes (all of them active), valid in
// every lane: DPP row operations, which need no LDS crossbar round trip, and
// for the whole wavefront the four rows' results through scalar registers.
template <int kLanes>
__device__ __forceinline__ unsigned group_min(unsigned v) {
  static_assert(kLanes == 4 || kLanes == 16 || kLanes == 64, "a quad, a DPP row or a wavefront");
  v = min(v, (unsigned)__builtin_amdgcn_update_dpp((int)v, (int)v, 0xB1, 0xf, 0xf, false));  // [1,0,3,2]
  v = min(v, (unsigned)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x4E, 0xf, 0xf, false));  // [2,3,0,1]
  if (kLanes >= 16) {
    v = min(v, (unsigned)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x141, 0xf, 0xf, false));  // half mirror
    v = min(v, (unsigned)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x140, 0xf, 0xf, false));  // mirror
  }
  if (kLanes == 64) {
    const unsigned a = (unsigned)__builtin_amdgcn_readlane((int)v, 15), b = (unsigned)__builtin_amdgcn_readlane((int)v, 31);
    const unsigned c = (unsigned)__builtin_amdgcn_readlane((int)v, 47), d = (unsigned)__builtin_amdgcn_readlane((int)v, 63);
    v = min(min(a, b), min(c, d));
  }
  return v;
}

}  // namespace dcx
