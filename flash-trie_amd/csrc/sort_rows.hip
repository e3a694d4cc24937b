// sort_rows.hip -- puts proposal rows that came in no token order (a model
// emits them by score) into ascending token order on the device, before the
// search that follows on the stream.
//
// One workgroup a row, its (token, index) pairs in registers, kE a thread:
// a bitonic sort whose exchanges at distances below 64 are lane shuffles and
// in-thread swaps, and go through LDS only from 64 to half the workgroup (10
// of the 55 exchanges of 1024 pairs).  Bound by the row's way over PCIe and
// the launch: three requests of nine rows of 777 take 604 -> 151 us a call
// with the sort here instead of std::sort on the packing thread (19 us a
// row, 27 rows one after another).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "tbs_kernel.h"

namespace ftk {
namespace {

__device__ __forceinline__ uint64_t shfl_xor64(uint64_t v, int m) {
  return ((uint64_t)(uint32_t)__shfl_xor((int)(uint32_t)(v >> 32), m, 64) << 32) |
         (uint32_t)__shfl_xor((int)(uint32_t)v, m, 64);
}

// Block (r, t): row t of request r, from its block at `src` to the same
// block at `dst`; block (r, 0) also copies what lies in front of the rows.  A
// token that a row holds twice withdraws the request (its ready word).
template <int kT, int kE>
__global__ void __launch_bounds__(kT) sort_rows_kernel(const DevReq* reqs, const uint8_t* src,
                                                       uint8_t* dst, uint64_t stage_bytes,
                                                       unsigned long long* ready,
                                                       unsigned long long tag) {
  __shared__ uint64_t keys[kT * kE];
  __shared__ float lps[kT * kE];
  const uint32_t r = blockIdx.x, t = blockIdx.y, tid = threadIdx.x;
  const DevReq d = reqs[r];
  // (the search reports a block that does not fit)
  if ((d.flags & kReqSkip) || t >= d.T || d.K > (uint32_t)(kT * kE) || !block_fits(stage_bytes, d))
    return;
  const uint32_t K = d.K;
  const uint64_t row = (uint64_t)t * K;
  if (t == 0)
    for (uint32_t i = tid; i < d.rid_off / 16u; i += kT)
      ((uint4*)(dst + d.in_off))[i] = ((const uint4*)(src + d.in_off))[i];
  const uint32_t* rid = (const uint32_t*)(src + d.in_off + d.rid_off) + row;
  const float* rlp = (const float*)(src + d.in_off + d.rlp_off) + row;
  uint64_t key[kE];
#pragma unroll
  for (int e = 0; e < kE; ++e) {
    const uint32_t i = (uint32_t)e * kT + tid;
    key[e] = ~0ull;  // (after every pair: an index is below 2^16)
    if (i < K) {
      key[e] = ((uint64_t)rid[i] << 32) | i;
      lps[i] = rlp[i];
    }
  }
  // pairs i and i ^ j in ascending order where bit k of i is clear; the pairs
  // past K stay where they are, so sorting up to the next power of two does
  for (uint32_t k = 2; (k >> 1) < K; k <<= 1) {
    for (uint32_t j = k >> 1; j > 0; j >>= 1) {
      if (j >= (uint32_t)kT) {
        const uint32_t je = j / kT;
#pragma unroll
        for (int e = 0; e < kE; ++e) {
#pragma unroll
          for (int f = e + 1; f < kE; ++f) {
            if ((uint32_t)(e ^ f) == je) {
              const bool up = (((uint32_t)e * kT) & k) == 0;
              const uint64_t a = min(key[e], key[f]), b = max(key[e], key[f]);
              key[e] = up ? a : b;
              key[f] = up ? b : a;
            }
          }
        }
        continue;
      }
      uint64_t other[kE];
      if (j < 64u) {
#pragma unroll
        for (int e = 0; e < kE; ++e) other[e] = shfl_xor64(key[e], (int)j);
      } else {
        __syncthreads();
#pragma unroll
        for (int e = 0; e < kE; ++e) keys[e * kT + tid] = key[e];
        __syncthreads();
#pragma unroll
        for (int e = 0; e < kE; ++e) other[e] = keys[e * kT + (tid ^ j)];
      }
#pragma unroll
      for (int e = 0; e < kE; ++e) {
        const uint32_t i = (uint32_t)e * kT + tid;
        const bool low = (i & j) == 0, up = (i & k) == 0;
        key[e] = low == up ? min(key[e], other[e]) : max(key[e], other[e]);
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < kE; ++e) keys[e * kT + tid] = key[e];
  __syncthreads();
  uint32_t* oid = (uint32_t*)(dst + d.in_off + d.rid_off) + row;
  float* olp = (float*)(dst + d.in_off + d.rlp_off) + row;
  uint16_t* ork = (uint16_t*)(dst + d.in_off + d.rk_off) + row;
  bool twice = false;
#pragma unroll
  for (int e = 0; e < kE; ++e) {
    const uint32_t i = (uint32_t)e * kT + tid;
    if (i < K) {
      const uint32_t tok = (uint32_t)(key[e] >> 32), at = (uint32_t)key[e];
      twice = twice || (i > 0 && (uint32_t)(keys[i - 1] >> 32) == tok);
      oid[i] = tok;
      olp[i] = lps[at];
      ork[i] = (uint16_t)at;
    }
  }
  if (twice)
    __hip_atomic_store(&ready[r], tag | kReadyWithdrawn, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace

hipError_t launch_sort_rows(const KArgs& a, hipStream_t stream) {
  const dim3 grid(a.batch, a.sort_steps);
  const unsigned long long tag = (unsigned long long)a.epoch << 32;
  unsigned long long* ready = const_cast<unsigned long long*>(a.ready);
  uint8_t* dst = const_cast<uint8_t*>(a.stage);
  // the smallest workgroup (and pairs a thread) that holds the longest row
  if (a.sort_topk <= 256u)
    hipLaunchKernelGGL((sort_rows_kernel<256, 1>), grid, dim3(256), 0, stream, a.reqs, a.sort_src,
                       dst, a.stage_bytes, ready, tag);
  else if (a.sort_topk <= 1024u)
    hipLaunchKernelGGL((sort_rows_kernel<1024, 1>), grid, dim3(1024), 0, stream, a.reqs,
                       a.sort_src, dst, a.stage_bytes, ready, tag);
  else if (a.sort_topk <= kMaxLdsTopk)
    hipLaunchKernelGGL((sort_rows_kernel<1024, 4>), grid, dim3(1024), 0, stream, a.reqs,
                       a.sort_src, dst, a.stage_bytes, ready, tag);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace ftk
