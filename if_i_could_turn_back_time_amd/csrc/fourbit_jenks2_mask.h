// The mask of the two-class Jenks split: which values sit at or past it in the stable ascending
// order.  Shared by fourbit_jenks2.hip and the tests, which place splits where a minimum of the
// within-class sums practically never is (inside a run of equal values).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace {

// Which of the values equal to the one at the split are kept: those at index >= first.
struct J2Ties {
  float t;        // the value at the split's sorted position
  int before;     // values equal to t at sorted positions before the split
  int first;
};
constexpr int kTieSeg = 16384;  // values one workgroup counts

int grid_of(int64_t items, int threads) { return (int)((items + threads - 1) / threads); }
int64_t tie_segments(int64_t n) { return (n + kTieSeg - 1) / kTieSeg; }

// keep[i] = 1 when w[i] sits at a position >= split of the stable ascending sort.  With t the
// value at that position: every value above t is kept and every value below is not; values
// equal to t (-0.0 == +0.0) sit in index order, so of those all but the first `before` are.  So
// the sort needs no indices: keys alone, and where the split falls inside a run of equal values
// (rare) a count finds the index of the first one kept.
__global__ void j2_ties(const float* __restrict__ skeys, const int64_t* __restrict__ split,
                        J2Ties* __restrict__ out) {
  const int64_t sp = *split;
  const float t = skeys[sp];
  int64_t lo = sp;
  if (sp > 0 && !(skeys[sp - 1] < t)) {  // first position not below t
    lo = 0;
    int64_t hi = sp - 1;
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (skeys[mid] < t)
        lo = mid + 1;
      else
        hi = mid;
    }
  }
  out->t = t;
  out->before = (int)(sp - lo);
  out->first = 0;
}

// How many values of each segment equal t (only where the split is inside a run of them).
__global__ __launch_bounds__(256) void j2_tie_count(const float* __restrict__ w, int n,
                                                    const J2Ties* __restrict__ ties,
                                                    int* __restrict__ cnt) {
  if (ties->before == 0) return;
  __shared__ int part[4];
  const float t = ties->t;
  const int64_t i0 = (int64_t)blockIdx.x * kTieSeg;
  const int64_t i1 = i0 + kTieSeg < n ? i0 + kTieSeg : n;
  int c = 0;
  for (int64_t i = i0 + threadIdx.x; i < i1; i += 256) c += w[i] == t ? 1 : 0;
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) c += __shfl_xor(c, m, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) cnt[blockIdx.x] = part[0] + part[1] + part[2] + part[3];
}

// The index of the value equal to t that has `before` others ahead of it: one wave walks the
// segments' counts, then the segment.
__global__ __launch_bounds__(64) void j2_tie_find(const float* __restrict__ w, int n, int nseg,
                                                  const int* __restrict__ cnt,
                                                  J2Ties* __restrict__ ties) {
  int left = ties->before;
  if (left == 0) return;
  const float t = ties->t;
  int seg = 0;
  for (; seg < nseg - 1; ++seg) {
    const int c = cnt[seg];
    if (left < c) break;
    left -= c;
  }
  const int64_t i0 = (int64_t)seg * kTieSeg;
  const int64_t i1 = i0 + kTieSeg < n ? i0 + kTieSeg : n;
  for (int64_t i = i0; i < i1; i += 64) {
    const int64_t at = i + threadIdx.x;
    const uint64_t b = __ballot(at < i1 && w[at] == t);
    const int c = __popcll(b);
    if (left < c) {
      const uint64_t below = threadIdx.x == 0 ? 0ull : (~0ull >> (64 - threadIdx.x));
      if ((b >> threadIdx.x & 1) && __popcll(b & below) == left) ties->first = (int)at;
      return;
    }
    left -= c;
  }
}

// The streaming pass over w that writes the mask, 4 values a thread where w and keep allow it.
__global__ void j2_mask(const float* __restrict__ w, int n, const J2Ties* __restrict__ ties,
                        uint8_t* __restrict__ keep, int vec) {
  const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (i >= n) return;
  const float t = ties->t;
  const int it = ties->first;
  auto kept = [&](float v, int64_t at) -> unsigned { return v > t || (v == t && at >= it); };
  if (vec && i + 4 <= n) {
    const float4 v = *reinterpret_cast<const float4*>(w + i);
    *reinterpret_cast<unsigned*>(keep + i) = kept(v.x, i) | (kept(v.y, i + 1) << 8) |
                                             (kept(v.z, i + 2) << 16) | (kept(v.w, i + 3) << 24);
  } else {
    for (int64_t j = i; j < n && j < i + 4; ++j) keep[j] = (uint8_t)kept(w[j], j);
  }
}

// keep [n] from w [n], its ascending sort skeys and *split, all on the device; ties and cnt
// (tie_segments(n) values) are scratch.
void launch_mask(const float* w, int n, const float* skeys, const int64_t* split, J2Ties* ties,
                 int* cnt, uint8_t* keep, hipStream_t hs) {
  const int nseg = (int)tie_segments(n);
  hipLaunchKernelGGL(j2_ties, dim3(1), dim3(1), 0, hs, skeys, split, ties);
  hipLaunchKernelGGL(j2_tie_count, dim3(nseg), dim3(256), 0, hs, w, n, ties, cnt);
  hipLaunchKernelGGL(j2_tie_find, dim3(1), dim3(64), 0, hs, w, n, nseg, cnt, ties);
  const int vec = (reinterpret_cast<uintptr_t>(w) & 15u) == 0 &&
                  (reinterpret_cast<uintptr_t>(keep) & 3u) == 0;
  hipLaunchKernelGGL(j2_mask, dim3(grid_of(n, 1024)), dim3(256), 0, hs, w, n, ties, keep, vec);
}

}  // namespace
