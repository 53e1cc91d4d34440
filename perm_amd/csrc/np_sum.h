// numpy's float64 summation of n values v(i), by one workgroup (np.add.reduce of a
// contiguous or strided vector). It reduces in chunks of 8192 values (its ufunc buffer size),
// adding the chunk sums left to right onto +0.0. Inside a chunk the sum is pairwise: fewer than
// 8 values one by one from +0.0; up to 128 with eight strided accumulators,
// ((r0+r1)+(r2+r3))+((r4+r5)+(r6+r7)), then the remainder one by one; longer runs split at n/2
// rounded down to a multiple of 8, the two halves summed recursively.
//
// The chunk's split tree is laid out as a heap (node i, halves 2i and 2i + 1; a run of m
// values splits into at most m/2 + 8, so 8192 end by level 7), its leaves are summed in
// parallel by 8 lanes each, and the halves added level by level, over as many levels as the
// chunk can reach (all seven for 32 values: 4.3 us, 2.0 so). Walked by one lane, the tree is a
// chain of dependent loads (objective totals of 29 tensors up to n = 3072: 167 us, 10 here; the
// damping shift of one n = 1024 matrix: 19 us, 7 here).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cp {

constexpr int kNpChunk = 8192, kTreeNodes = 256;

struct NpSumLds {
  int2 node[kTreeNodes];  // (first value, count) of each run; count 0: absent
  double val[kTreeNodes];
};

// Every thread of the workgroup (a multiple of 64, at least 128) calls this and gets the sum.
template <class V>
__device__ double np_sum_block(const V& v, int64_t n, NpSumLds& lds) {
  auto& node = lds.node;
  auto& val = lds.val;
  double s = 0.0;
  const int t = (int)threadIdx.x, groups = (int)blockDim.x / 8;
  for (int64_t c0 = 0; c0 < n; c0 += kNpChunk) {
    const int count = (int)(n - c0 < kNpChunk ? n - c0 : kNpChunk);
    int last = 1;  // first node of the last level
    for (int m = count; m > 128; m = m / 2 + 8) last *= 2;
    __syncthreads();
    if (t == 0) node[1] = make_int2(0, count);
    for (int first = 1; first < last; first *= 2) {
      __syncthreads();
      if (t < first) {
        const int2 p = node[first + t];
        const int h = p.y > 128 ? p.y / 2 / 8 * 8 : 0;  // 0: a leaf, or absent
        node[2 * (first + t)] = make_int2(p.x, h);
        node[2 * (first + t) + 1] = make_int2(p.x + h, h ? p.y - h : 0);
      }
    }
    __syncthreads();
    for (int i0 = 0; i0 < 2 * last; i0 += groups) {  // the same trips for every lane of a wave
      const int i = i0 + t / 8;
      const int2 p = i > 0 && i < 2 * last ? node[i] : make_int2(0, 0);
      const bool leaf = p.y > 0 && p.y <= 128;
      const int whole = p.y / 8 * 8;
      double r = 0.0;
      if (leaf && whole) {
        const int64_t o = c0 + p.x + t % 8;
        r = v(o);
        for (int k = 8; k < whole; k += 8) r = r + v(o + k);
      }
      r = r + __shfl_xor(r, 1);
      r = r + __shfl_xor(r, 2);
      r = r + __shfl_xor(r, 4);
      if (leaf && t % 8 == 0) {
        for (int k = whole; k < p.y; ++k) r = r + v(c0 + p.x + k);
        val[i] = r;
      }
    }
    for (int first = last / 2; first >= 1; first /= 2) {
      __syncthreads();
      if (t < first && node[first + t].y > 128) val[first + t] = val[2 * (first + t)] + val[2 * (first + t) + 1];
    }
    __syncthreads();
    s = s + val[1];
  }
  return s;
}

}  // namespace cp
