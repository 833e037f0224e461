// Packers on the GPU, producing the same bytes as the host packers of fourbit_host.cpp:
// GF4 (the Jenks-16 and masked Jenks quantizer, one wavefront per (row, 128-group), fp64)
// and E2M1 (32 lanes per 32-group).
//
// Every fp64 expression is the host's, evaluated in the host's order, and this file is
// compiled with -ffp-contract=off (no fused multiply-adds), so each operation rounds
// exactly as on the CPU.  IEEE fp64 add/mul/div are correctly rounded on gfx950 and the
// conversions fp64 -> fp32 -> fp16 round to nearest even, so the outputs are bit-identical
// to fb_quantize_gf4 / fb_quantize_gf4_masked (and to the CPU oracle).
//
// Per group (one wave, LDS region of its own):
//   1. load 128 fp32 values (2 per lane) and the keep flags; compact the kept values in
//      index order with ballots (m of them);
//   2. stable rank by (value, index): rank = #{u : v_u < v} + #{u < t : v_u == v};
//   3. sequential fp64 prefix sums S1, S2 (one running sum, as the host);
//   4. the DP D[c][j] = min_{i >= c-1} D[c-1][i] + SSD(i, j) over classes c = 2..k, lane L
//      owning j = L+1 and j = L+65 for all classes at once, in registers.  The i loop is
//      outermost: SSD(i, j) does not depend on c, so it is computed once instead of 15 times,
//      and column i is final when the loop reaches i (every i' < i has been offered), so its
//      15 values go to all lanes by readlane.  For every (c, j) the candidates still come in
//      ascending i and only a strictly smaller one replaces: ties keep the smallest break, as
//      on the host;
//   5. no back pointers are kept (a third of the loop's instructions): the walk back finds each
//      break as the first i whose candidate equals D[c][j]; lanes 0..k-1 form the centroids;
//      the codes are scattered back to index order, nibble-packed, and written with the
//      codebook.
//
// The division of SSD(i, j) by j - i <= 128 is a product with the correctly rounded reciprocal
// and one correction, q + (x - q d) r: x - q d is exact (a small multiple of q's last place),
// so q1 before its rounding is within 2^-50 last places of x / d, while x / d is at least
// 1 / 256 of a last place away from every rounding boundary (or exact: 2 x = (2 n + 1) d has
// no 53-bit solution x for a 54-bit odd 2 n + 1 unless d is a power of two, and then x / d is
// exact).  So it rounds as the division does.  x = s^2 is 0 or at least 2^-298 (s is a
// multiple of the smallest fp32), so nothing underflows.
//
// Bound by the VALU (fp64 adds, minima and readlanes: about 95 instructions per i, 14,300 per
// group in all).  4096^2 (131,072 groups): 17.9 ms with the class loop outermost (SSD with a
// division in it, back pointers kept), 4.0 ms now, the VALU busy 97% of the time.
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

#include <cstdint>

#include "fourbit.h"
#include "fourbit_layout.h"

namespace {

constexpr int kGroup = 128;
constexpr int kMaxClasses = 16;

struct PackLds {
  double vs[kGroup];              // kept values, sorted
  double S1[kGroup + 1];          // prefix sums of vs
  double S2[kGroup + 1];          // prefix sums of vs^2
  double inv[kGroup + 1];         // 1 / d
  float sub[kGroup];              // kept values in index order
  uint8_t pos[kGroup];            // original index of sub[t]
  uint8_t order[kGroup];          // original index of vs[p]
  uint8_t code[kGroup];           // final code by original index
  int bounds[kMaxClasses + 1];
  uint16_t cb[kMaxClasses];
};

// SSD(i, j) from column j's prefix sums, with d = j - i and r = 1 / d (see above).
__device__ __forceinline__ double ssd(double S1i, double S2i, double S1j, double S2j, double d,
                                      double r) {
  const double s = S1j - S1i;
  const double q = S2j - S2i;
  const double x = s * s;
  const double t = x * r;
  return q - __builtin_fma(__builtin_fma(-t, d, x), r, t);
}

// the smaller of two values, neither of them NaN (fmin would first canonicalise both operands,
// one more instruction per candidate)
__device__ __forceinline__ double min_f64(double a, double b) {
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

__device__ __forceinline__ double lane_value(double v, int lane) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const unsigned lo = __builtin_amdgcn_readlane((int)(unsigned)b, lane);
  const unsigned hi = __builtin_amdgcn_readlane((int)(unsigned)(b >> 32), lane);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

__global__ __launch_bounds__(64) void gf4_pack_kernel(const float* __restrict__ w,
                                                      const uint8_t* __restrict__ keep,
                                                      int K, int64_t groups,
                                                      uint8_t* __restrict__ codes,
                                                      uint16_t* __restrict__ book) {
  __shared__ PackLds L;
  const int lane = threadIdx.x;
  const int G = K / kGroup;
  for (int d = lane; d <= kGroup; d += 64) L.inv[d] = 1.0 / (double)d;  // [0] is not read
  for (int64_t it = blockIdx.x; it < groups; it += gridDim.x) {
    const int64_t n = it / G, g = it - n * G;
    const int64_t off = n * K + g * kGroup;

    // 1. load and compact the kept values (index order)
    const float v0 = w[off + lane], v1 = w[off + lane + 64];
    const bool k0 = keep ? keep[off + lane] != 0 : true;
    const bool k1 = keep ? keep[off + lane + 64] != 0 : true;
    const uint64_t b0 = __ballot(k0), b1 = __ballot(k1);
    const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const int c0 = __popcll(b0);
    const int m = c0 + __popcll(b1);
    const bool full = m == kGroup;
    const int k = full ? kMaxClasses : (m < kMaxClasses - 1 ? m : kMaxClasses - 1);
    if (k0) {
      const int t = __popcll(b0 & below);
      L.sub[t] = v0;
      L.pos[t] = (uint8_t)lane;
    }
    if (k1) {
      const int t = c0 + __popcll(b1 & below);
      L.sub[t] = v1;
      L.pos[t] = (uint8_t)(lane + 64);
    }
    __syncthreads();

    // 2. stable rank by (value, index) -- the host's std::stable_sort on (double)value
    {
      const int t0 = lane, t1 = lane + 64;
      const float a0 = t0 < m ? L.sub[t0] : 0.0f, a1 = t1 < m ? L.sub[t1] : 0.0f;
      int r0 = 0, r1 = 0;
      for (int u = 0; u < m; ++u) {
        const float vu = L.sub[u];
        r0 += (vu < a0) || (vu == a0 && u < t0);
        r1 += (vu < a1) || (vu == a1 && u < t1);
      }
      if (t0 < m) {
        L.vs[r0] = (double)a0;
        L.order[r0] = L.pos[t0];
      }
      if (t1 < m) {
        L.vs[r1] = (double)a1;
        L.order[r1] = L.pos[t1];
      }
    }
    __syncthreads();

    // 3. sequential prefix sums (every lane runs the same chain; lane 0 stores it)
    {
      double a = 0.0, b = 0.0;
      if (lane == 0) {
        L.S1[0] = 0.0;
        L.S2[0] = 0.0;
      }
      for (int t = 0; t < m; ++t) {
        const double x = L.vs[t];
        a = a + x;
        b = b + x * x;
        if (lane == 0) {
          L.S1[t + 1] = a;
          L.S2[t + 1] = b;
        }
      }
    }
    __syncthreads();

    // 4. DP over classes; lane owns columns j0 = lane+1 and j1 = lane+65 (valid if <= m)
    const double inf = __builtin_huge_val();
    const int j0 = lane + 1, j1 = lane + 65;
    const bool ok0 = j0 <= m, ok1 = j1 <= m;
    const double S1j0 = ok0 ? L.S1[j0] : 0.0, S2j0 = ok0 ? L.S2[j0] : 0.0;
    const double S1j1 = ok1 ? L.S1[j1] : 0.0, S2j1 = ok1 ? L.S2[j1] : 0.0;
    double D0[kMaxClasses], D1[kMaxClasses];  // D[c][j0], D[c][j1] for c = 1..15
    // one class: [0, j)
    D0[1] = ok0 ? ssd(0.0, 0.0, S1j0, S2j0, (double)j0, L.inv[j0]) : inf;
    D1[1] = ok1 ? ssd(0.0, 0.0, S1j1, S2j1, (double)j1, L.inv[j1]) : inf;
#pragma unroll
    for (int c = 2; c < kMaxClasses; ++c) D0[c] = D1[c] = inf;
    // breaks i whose column is a j0 (both of a lane's columns may use them)
    for (int i = 1; i < m && i <= 64; ++i) {
      const double S1i = L.S1[i], S2i = L.S2[i];
      const int d0 = j0 - i, d1 = j1 - i;  // d1 >= 1
      const bool use0 = d0 > 0 && ok0;
      double w0 = ssd(S1i, S2i, S1j0, S2j0, (double)d0, L.inv[use0 ? d0 : 1]);
      double w1 = ssd(S1i, S2i, S1j1, S2j1, (double)d1, L.inv[d1]);
      w0 = use0 ? w0 : inf;
      w1 = ok1 ? w1 : inf;
#pragma unroll
      for (int c = 2; c < kMaxClasses; ++c) {
        const double d = lane_value(D0[c - 1], i - 1);
        D0[c] = min_f64(D0[c], d + w0);
        D1[c] = min_f64(D1[c], d + w1);
      }
    }
    // breaks whose column is a j1
    for (int i = 65; i < m; ++i) {
      const int d1 = j1 - i;
      const bool use1 = d1 > 0 && ok1;
      double w1 = ssd(L.S1[i], L.S2[i], S1j1, S2j1, (double)d1, L.inv[use1 ? d1 : 1]);
      w1 = use1 ? w1 : inf;
#pragma unroll
      for (int c = 2; c < kMaxClasses; ++c)
        D1[c] = min_f64(D1[c], lane_value(D1[c - 1], i - 65) + w1);
    }

    // 5. breaks, centroids, codes.  The last break of (c, j) is the first i whose candidate is
    // D[c][j]: the lanes form the candidates of their own columns again, the same bits.
    {
      int j = m;
      if (lane == 0) L.bounds[k] = m;
#pragma unroll
      for (int c = kMaxClasses; c >= 2; --c) {
        if (c > k) continue;
        const double S1j = L.S1[j], S2j = L.S2[j];
        const int d0 = j - j0, d1 = j - j1;
        double e0 = D0[c - 1] + ssd(S1j0, S2j0, S1j, S2j, (double)d0, L.inv[d0 > 0 ? d0 : 1]);
        double e1 = D1[c - 1] + ssd(S1j1, S2j1, S1j, S2j, (double)d1, L.inv[d1 > 0 ? d1 : 1]);
        e0 = d0 > 0 ? e0 : inf;
        e1 = d1 > 0 ? e1 : inf;
        double best;
        if (c == kMaxClasses) {  // the row that the loops above leave out: only j = m is needed
          best = min_f64(e0, e1);
#pragma unroll
          for (int x = 32; x >= 1; x >>= 1) best = min_f64(best, __shfl_xor(best, x, 64));
        } else {
          best = j > 64 ? lane_value(D1[c], (j - 1) & 63) : lane_value(D0[c], (j - 1) & 63);
        }
        const uint64_t m0 = __ballot(d0 > 0 && e0 == best), m1 = __ballot(d1 > 0 && e1 == best);
        j = m0 ? __builtin_ctzll(m0) + 1 : m1 ? __builtin_ctzll(m1) + 65 : 0;
        if (lane == 0) L.bounds[c - 1] = j;
      }
      if (lane == 0) L.bounds[0] = 0;
    }
    __syncthreads();
    if (lane < k) {
      const int lo = L.bounds[lane], hi = L.bounds[lane + 1];
      const double mean = (L.S1[hi] - L.S1[lo]) / (double)(hi - lo);
      L.cb[lane] = __half_as_ushort(__float2half_rn((float)mean));
    }
    __syncthreads();
    // the zero entry of a masked group goes after the strictly negative centroids
    int z = 0;
    if (!full)
      for (int t = 0; t < k; ++t) z += ((L.cb[t] & 0x8000u) && (L.cb[t] & 0x7fffu)) ? 1 : 0;
    for (int h = 0; h < 2; ++h) {
      const int p = lane + 64 * h;
      L.code[p] = (uint8_t)z;  // masked entries
    }
    __syncthreads();
    for (int h = 0; h < 2; ++h) {
      const int p = lane + 64 * h;
      if (p < m) {
        int cls = 0;
        for (int c = 1; c < k; ++c) cls += (L.bounds[c] <= p) ? 1 : 0;
        L.code[L.order[p]] = (uint8_t)(full ? cls : cls + (cls >= z ? 1 : 0));
      }
    }
    __syncthreads();
    codes[n * (K / 2) + g * 64 + lane] = (uint8_t)(L.code[2 * lane] | (L.code[2 * lane + 1] << 4));
    if (lane < kMaxClasses) {
      uint16_t e;
      if (full) {
        e = L.cb[lane];
      } else {
        const int t = lane < k ? lane : k;  // entries past the last used one repeat it
        e = t < z ? L.cb[t] : (t == z ? (uint16_t)0 : L.cb[t - 1]);
      }
      book[it * kMaxClasses + lane] = e;
    }
    __syncthreads();
  }
}

// E2M1 + E8M0 per 32-group, 32 lanes per group (a wave packs two groups): the host
// packer's rule (fb_quantize_e2m1) in fp32, which is exact here: amax's exponent comes from
// frexp, q = v * 2^-e is a power-of-two scaling, and the rounding midpoints are fp32 values.
__device__ __forceinline__ int e2m1_index(float a) {
  const float mids[7] = {0.25f, 0.75f, 1.25f, 1.75f, 2.5f, 3.5f, 5.0f};
  int idx = 0;
  bool tie = false;
#pragma unroll
  for (int t = 0; t < 7; ++t) {
    idx += a > mids[t] ? 1 : 0;
    tie = tie || a == mids[t];
  }
  if (tie && (idx & 1)) ++idx;
  return idx < 7 ? idx : 7;
}

__global__ __launch_bounds__(256) void e2m1_pack_kernel(const float* __restrict__ w,
                                                        int64_t groups,
                                                        uint8_t* __restrict__ codes,
                                                        uint8_t* __restrict__ scales) {
  const int lane = threadIdx.x & 63;
  const int t = lane & 31;                        // value index in the group
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> 6;
  for (int64_t it0 = wave * 2; it0 < groups; it0 += nwaves * 2) {  // uniform per wave
    const int64_t it = it0 + (lane >> 5);
    const bool live = it < groups;
    const float v = live ? w[it * 32 + t] : 0.0f;
    float amax = __builtin_fabsf(v);
#pragma unroll
    for (int m = 16; m >= 1; m >>= 1) amax = fmaxf(amax, __shfl_xor(amax, m, 32));
    int ex = 0;
    if (amax > 0.0f) {
      int e2;
      (void)frexpf(amax, &e2);  // amax = m * 2^e2, m in [0.5, 1)
      ex = e2 - 1 - 2;
      ex = ex < -127 ? -127 : (ex > 127 ? 127 : ex);
    }
    const float q = ldexpf(v, -ex);
    const int code = (__builtin_signbit(v) ? 8 : 0) | e2m1_index(__builtin_fabsf(q));
    const int hi = __shfl_xor(code, 1, 32);
    if (live && !(t & 1)) codes[it * 16 + (t >> 1)] = (uint8_t)(code | (hi << 4));
    if (live && t == 0) scales[it] = (uint8_t)(ex + 127);
  }
}

// ---------------------------------------------------------------------------------
// Canonical codes and codebooks (or scales) -> the kernels' weight stream: fb_to_device on the
// GPU, the same bytes.  One wave per block, lane L its item (row 16t + L % 16, group 4sp + L /
// 16): it reads the item's 64 bytes of codes and its codebook or scales, and writes the block's
// chunks, each 1 KiB over the wave.  Items past N or K are zero bytes.  Bound by memory.
// ---------------------------------------------------------------------------------
__device__ __forceinline__ unsigned spread4(unsigned x) {  // nibble k of 4 -> byte k
  x = (x | (x << 8)) & 0x00FF00FFu;
  return (x | (x << 4)) & 0x0F0F0F0Fu;
}

template <int FMT>
__global__ __launch_bounds__(256) void layout_kernel(const uint8_t* __restrict__ codes,
                                                     const uint8_t* __restrict__ meta,
                                                     uint8_t* __restrict__ wdev, int N, int K,
                                                     int GS, int64_t blocks) {
  constexpr int BB = FMT == FB_FMT_GF4 ? fb::kGf4BlockBytes : fb::kE2m1BlockBytes;
  const int lane = threadIdx.x & 63;
  const int64_t b = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (b >= blocks) return;
  const int64_t t = b / GS;
  const int sp = (int)(b - t * GS);
  const int64_t n = t * 16 + (lane & 15);
  const int G = K / 128, g = sp * 4 + (lane >> 4);
  const bool live = n < N && g < G;
  uint4 q[4] = {};
  if (live) {
    const uint4* src = reinterpret_cast<const uint4*>(codes + n * (K / 2) + g * 64);
#pragma unroll
    for (int c = 0; c < 4; ++c) q[c] = src[c];
  }
  uint8_t* const dst = wdev + b * BB;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    if (FMT == FB_FMT_GF4) {
      unsigned* w = reinterpret_cast<unsigned*>(&q[c]);
#pragma unroll
      for (int d = 0; d < 4; ++d) w[d] = spread4(w[d] & 0xFFFFu) | (spread4(w[d] >> 16) << 4);
    }
    *reinterpret_cast<uint4*>(dst + c * 1024 + lane * 16) = q[c];
  }
  if (FMT == FB_FMT_GF4) {
    uint8_t lo[16], hi[16], tl[16] = {}, th[16] = {};
    if (live) {
      const uint16_t* book = reinterpret_cast<const uint16_t*>(meta) + (n * G + g) * 16;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        lo[i] = (uint8_t)(book[i] & 0xFF);
        hi[i] = (uint8_t)(book[i] >> 8);
      }
      fb::gf4_xor_tables(lo, tl, tl + 8);
      fb::gf4_xor_tables(hi, th, th + 8);
    }
    unsigned wl[4], wh[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      wl[i] = tl[4 * i] | (tl[4 * i + 1] << 8) | (tl[4 * i + 2] << 16) | ((unsigned)tl[4 * i + 3] << 24);
      wh[i] = th[4 * i] | (th[4 * i + 1] << 8) | (th[4 * i + 2] << 16) | ((unsigned)th[4 * i + 3] << 24);
    }
    *reinterpret_cast<uint4*>(dst + 4096 + lane * 16) = make_uint4(wl[0], wl[1], wl[2], wl[3]);
    *reinterpret_cast<uint4*>(dst + 5120 + lane * 16) = make_uint4(wh[0], wh[1], wh[2], wh[3]);
  } else {
    unsigned sc = 0;
    if (live) sc = *reinterpret_cast<const unsigned*>(meta + (n * G + g) * 4);
    *reinterpret_cast<unsigned*>(dst + 4096 + lane * 4) = sc;
  }
}

}  // namespace

extern "C" {

int fb_to_device_gpu(const uint8_t* codes, const void* meta, void* wdev, const fb_shape_t* s,
                     void* stream) {
  if (!s || !codes || !meta || !wdev) return FB_ERR_NULL;
  const int st = fb_validate(s);
  if (st != FB_OK) return st;
  if ((reinterpret_cast<uintptr_t>(codes) & 15u) || (reinterpret_cast<uintptr_t>(wdev) & 15u) ||
      (reinterpret_cast<uintptr_t>(meta) & 3u))
    return FB_ERR_ALIGN;
  const int GS = (int)fb::spans_per_row(s->K);
  const int64_t blocks = fb::row_tiles(s->N) * GS;  // < 2^31 (fb_validate)
  const dim3 grid((unsigned)((blocks + 3) / 4));
  hipStream_t hs = static_cast<hipStream_t>(stream);
  const uint8_t* m = static_cast<const uint8_t*>(meta);
  uint8_t* w = static_cast<uint8_t*>(wdev);
  if (s->fmt == FB_FMT_GF4)
    hipLaunchKernelGGL(layout_kernel<FB_FMT_GF4>, grid, dim3(256), 0, hs, codes, m, w, s->N, s->K,
                       GS, blocks);
  else
    hipLaunchKernelGGL(layout_kernel<FB_FMT_E2M1>, grid, dim3(256), 0, hs, codes, m, w, s->N, s->K,
                       GS, blocks);
  return hipGetLastError() == hipSuccess ? FB_OK : FB_ERR_HIP;
}

int fb_quantize_gf4_gpu(const float* w, const uint8_t* keep, int32_t N, int32_t K,
                        uint8_t* codes, uint16_t* codebook, void* stream) {
  if (!w || !codes || !codebook) return FB_ERR_NULL;
  if (N < 1 || K < 128 || K % 128) return FB_ERR_SHAPE;
  const int64_t groups = (int64_t)N * (K / kGroup);
  const int grid = (int)(groups < (1 << 14) ? groups : (1 << 14));  // 64 waves per CU, in turn
  hipLaunchKernelGGL(gf4_pack_kernel, dim3(grid), dim3(64), 0,
                     static_cast<hipStream_t>(stream), w, keep, K, groups, codes, codebook);
  return hipGetLastError() == hipSuccess ? FB_OK : FB_ERR_HIP;
}

}  // extern "C"

extern "C" int fb_quantize_e2m1_gpu(const float* w, int32_t N, int32_t K, uint8_t* codes,
                                    uint8_t* scales, void* stream) {
  if (!w || !codes || !scales) return FB_ERR_NULL;
  if (N < 1 || K < 128 || K % 128) return FB_ERR_SHAPE;
  const int64_t groups = (int64_t)N * (K / 32);
  const int64_t blocks = (groups + 7) / 8;  // 8 groups per 256-thread block
  const int grid = (int)(blocks < (1 << 20) ? blocks : (1 << 20));
  hipLaunchKernelGGL(e2m1_pack_kernel, dim3(grid), dim3(256), 0,
                     static_cast<hipStream_t>(stream), w, groups, codes, scales);
  return hipGetLastError() == hipSuccess ? FB_OK : FB_ERR_HIP;
}
