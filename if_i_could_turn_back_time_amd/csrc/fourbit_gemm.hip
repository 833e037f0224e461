// The 4-bit linear layer on many rows of x (prompts, training batches): y[M, N] = x[M, K] .
// W^T, one launch over all of x, where 16-row GEMV calls would read and decode the whole
// weight once per 16 rows.
//
// Workgroup tile: (64 RT rows of W) x (16 CT rows of x), 4 waves, one per SIMD, two workgroups
// per CU; each wave owns
// RT 16-row weight tiles and all CT column tiles, RT * CT * 4 fp32 accumulators per lane.
//  - W goes from the device stream straight into MFMA A operands, as in the GEMV: lane L's 16
//    bytes of a block are row L % 16, item L / 16, so no weight passes through LDS.  Every
//    weight is decoded once per workgroup.
//  - x goes through LDS in chunks of 128 K-values: the 32 values of each of a span's four
//    128-value items that the four k-steps of one 16-byte nibble chunk multiply.  The loads
//    write LDS directly (no VGPRs, no ds_write); the 16-byte units of an x row are permuted on
//    the load's source side (unit_mask), which leaves the MFMA B reads (16 rows, 256 bytes
//    apart) without a bank conflict.
//  - Nibbles and x are requested kBufs - 1 (1 or 3) chunks ahead, with one barrier per chunk.
//  - Each k-step's decode (21 VALU instructions per GF4 row tile, 8 codes per lane) is written
//    between the MFMAs of the step before it, a half decode per column tile, and the column
//    tiles are separate scheduling regions, so that the instruction stream alternates the two
//    (left to itself the compiler groups them, and a wave then waits for its own MFMAs).
// What bounds it: E2M1 runs at the matrix cores' power-limited rate (8192 -> 28672, M = 2048:
// 621 to 635 us, 1,515 to 1,549 TFLOP/s; the library's bf16 GEMM of 8192^3 reaches 1418 on the same card; one
// workgroup of wider staging per CU: 737 us); GF4 issues nearly as many cycles of decode and MFMA
// instructions as its MFMAs take (964 us, 998 TFLOP/s; 16-row GEMV calls: 4840 us; one workgroup
// per CU: 1006).  Small M is bound by latency and the x fill of each CU; the K range is then
// cut into P parts whose fp32 sums gemm_sum adds in part order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>

#include "fourbit.h"
#include "fourbit_decode.h"
#include "fourbit_layout.h"

// Host helpers shared by the GPU units.  Not part of the library's ABI.
namespace fb_gpu {
__attribute__((visibility("hidden"))) int cu_count();
__attribute__((visibility("hidden"))) int rotate_rows(const void* x, void* xo, int rows, int K,
                                                      int block, hipStream_t hs);
__attribute__((visibility("hidden"))) int sum_parts(const float* part, int P, int64_t n, void* y,
                                                    int ydt, int vec, const void* bias, int bdt,
                                                    int N, hipStream_t hs);
}  // namespace fb_gpu

namespace {

constexpr int kGemmWaves = 4;
constexpr int kRowBytes = 256;  // one x row of a chunk: 128 K-values, 32 of each item of a span

// What the 16-byte units of an x row n (mod 16) in LDS are permuted by (unit u sits at place u ^
// unit_mask(n)).  A 16-byte LDS read serves 16 lanes at a time over all 64 banks: lanes 0-3,
// 12-15, 20-23 and 24-27 together, and so on.  In the B read lane L takes row L % 16, unit
// 4 (L / 16) + s, so such a set holds 16 different rows, of two neighbouring items, and n itself
// as the mask would put half of them on the same places (4 of 12 cycles per read, counted).
__device__ __forceinline__ int unit_mask(int n) { return n ^ ((((n >> 2) ^ (n >> 3)) & 1) << 2); }

struct GemmArgs {
  const uint8_t* w;
  const void* x;
  void* y;
  float* part;  // P > 1: the parts' fp32 sums [P, M, N]; else null
  const void* bias;  // [N] of dtype bdt, or null; added in fp32 before y's one rounding
  int M, N, K;
  int GS;       // spans per row
  int tiles_n, tiles_m;
  int spp;      // spans per K-part
  int ydt, bdt;
  int vec;      // y (and part) rows take 4-value stores: N % 4 == 0, 16-byte aligned y
};

template <int RT, int CT>
struct GemmTile {
  static constexpr int kRows = RT * 16 * kGemmWaves;  // rows of W
  static constexpr int kCols = CT * 16;               // rows of x
  static constexpr int kBuf = kCols * kRowBytes;      // one staged chunk
  // Two workgroups share a CU (two waves per SIMD: one's decode issues while the other's
  // MFMAs run), so two chunks of the wide tiles are staged at a time; four of the small ones,
  // whose chunks are too short to cover a request's latency.
  static constexpr int kBufs = kBuf * 4 <= 64 * 1024 && RT * CT <= 12 ? 4 : 2;
  static_assert(kBuf * kBufs <= 80 * 1024, "two workgroups per CU");
};

template <int FMT, int XDT, int RT, int CT>
__global__ __launch_bounds__(kGemmWaves * 64, 2) void gemm_kernel(GemmArgs a) {
  using T = GemmTile<RT, CT>;
  constexpr int BB = FMT == FB_FMT_GF4 ? fb::kGf4BlockBytes : fb::kE2m1BlockBytes;
  constexpr int NB = T::kBufs, D = NB - 1;
  // The barrier in the middle of the chunk before, where a chunk is long enough for the shorter
  // time that leaves its requests: 1 to 6% over 13 shapes with CT = 3 and 4 (8192 -> 28672, M = 64,
  // GF4: 55.1 -> 52.2 us), 0 to 3% slower with CT = 2.
  constexpr bool kEarly = NB == 4 && CT >= 3;
  constexpr int XD = T::kBuf / (kGemmWaves * 1024);  // 1 KiB x requests of one wave per chunk
  __shared__ __align__(1024) uint8_t xb0[T::kBuf], xb1[T::kBuf];
  __shared__ __align__(1024) uint8_t xb2[NB == 4 ? T::kBuf : 16], xb3[NB == 4 ? T::kBuf : 16];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // Tile of this workgroup.  Workgroups go round-robin over the 8 XCDs: each XCD takes a
  // contiguous run of tiles, 4 x-tiles by many weight tiles at a time, so that the tiles in
  // flight on an XCD share x and weights in its L2.
  const int per = a.tiles_n * a.tiles_m;
  const int total = gridDim.x;
  int id = blockIdx.x;
  {
    const int q = total >> 3, r = total & 7, xcd = id & 7, k = id >> 3;
    id = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + k;
  }
  const int p = id / per;
  id -= p * per;
  const int gsz = 4 * a.tiles_n;
  const int g = id / gsz, gm = min(4, a.tiles_m - g * 4);
  const int rem = id - g * gsz;
  const int tn = rem / gm, tm = g * 4 + (rem - tn * gm);

  const int sp0 = p * a.spp, sp1 = min(a.GS, sp0 + a.spp);
  const int nsp = sp1 - sp0;
  const int m0 = tm * T::kCols;
  const int rows = min(T::kCols, a.M - m0);
  const int row_tiles = (a.N + 15) >> 4;
  const int t0 = tn * (RT * kGemmWaves) + wave * RT;

  const rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(static_cast<const uint8_t*>(a.x)) + (int64_t)m0 * a.K * 2, (short)0,
      rows * a.K * 2, kRsrcWord3);
  rsrc_t wrs[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int t = min(t0 + r, row_tiles - 1);
    wrs[r] = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(a.w) + (int64_t)t * a.GS * BB, (short)0, a.GS * BB, kRsrcWord3);
  }

  // Request j of a wave fills 4 x rows of a chunk (1 KiB, lane order): this lane's row and the
  // 16-byte unit whose place in that row it fills.  Rows past M are out of the resource's
  // range and read zeros; so do K-values past K (the weight stream is zero there).
  unsigned xoff[4];
  int xk[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int row = (wave * XD + j) * 4 + (lane >> 4);
    const int u = (lane & 15) ^ unit_mask(row & 15);
    xoff[j] = (unsigned)row * (unsigned)a.K * 2u + (u >> 2) * 256 + (u & 3) * 16;
    xk[j] = (u >> 2) * 128;
  }
  auto stage = [&](int sp, int c, uint8_t* buf) {
    const int kleft = a.K - sp * 512;
    const unsigned so = (unsigned)sp * 1024u + (unsigned)c * 64u;
#pragma unroll
    for (int j = 0; j < XD; ++j) {
      const unsigned off = xk[j & 3] < kleft
                               ? xoff[j & 3] + (unsigned)((j >> 2) * 16) * (unsigned)a.K * 2u + so
                               : kXOutOfRange;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          xrs, (lds_byte*)(buf + (wave * XD + j) * 1024), 16, off, 0, 0, 0);
    }
  };

  u32x4 nib[NB][RT];
  u32x4 tb[RT][2], tbn[RT][2];
  auto load_nib = [&](int sp, int c, u32x4 (&d)[RT]) {
#pragma unroll
    for (int r = 0; r < RT; ++r)
      d[r] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                           wrs[r], lane * 16 + c * 1024, sp * BB, 0));
  };
  auto load_tab = [&](int sp, u32x4 (&d)[RT][2]) {
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      if constexpr (FMT == FB_FMT_GF4) {
        d[r][0] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                wrs[r], lane * 16 + 4096, sp * BB, 0));
        d[r][1] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                wrs[r], lane * 16 + 5120, sp * BB, 0));
      } else {
        d[r][0].x = __builtin_amdgcn_raw_buffer_load_b32(wrs[r], lane * 4 + 4096, sp * BB, 0);
      }
    }
  };

  f32x4 acc[RT][CT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int c = 0; c < CT; ++c) acc[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};

  // B operand of column tile ct, k-step s: x row lane % 16, unit 4 (lane / 16) + s
  const unsigned rbase =
      (lane & 15) * kRowBytes + ((((lane >> 4) * 4) ^ unit_mask(lane & 15)) << 4);

  // Half h of the A operand of k-step s of chunk c (words 2h, 2h + 1 of 4), from nibbles nb
  // and tables tt.
  auto decode_half = [&](u32x4& A, const u32x4& nb, const u32x4 (&tt)[2], int c, int s, int h) {
    if constexpr (FMT == FB_FMT_GF4) {
      const unsigned sel = (h ? nb[s] >> 4 : nb[s]) & 0x0F0F0F0Fu;
      const unsigned sel8 = sel ^ 0x08080808u;
      const unsigned lo = perm(tt[0].y, tt[0].x, sel) ^ perm(tt[0].w, tt[0].z, sel8);
      const unsigned hi = perm(tt[1].y, tt[1].x, sel) ^ perm(tt[1].w, tt[1].z, sel8);
      A[2 * h] = perm(hi, lo, 0x05010400u);
      A[2 * h + 1] = perm(hi, lo, 0x07030602u);
    } else {
      const float sc = __builtin_bit_cast(float, ((tt[0].x >> (8 * c)) & 0xFFu) << 23);
      const u32x4 v = e2m1_decode8<XDT>(nb[s], sc);
      A[2 * h] = v[2 * h];
      A[2 * h + 1] = v[2 * h + 1];
    }
  };
  u32x4 A[2][RT];  // this k-step's operands and the next one's
  // k-steps [s0, s1) of a chunk: RT x CT MFMAs each, B operands read kAhead column tiles ahead
  // (with four chunks staged, from the next chunk too).
  constexpr int kAhead = kEarly ? 3 : 2, kRing = kAhead + 1;
  u32x4 B[kRing];
  auto readb = [&](const uint8_t* buf, int i) {
    return *reinterpret_cast<const u32x4*>(buf + (rbase ^ ((i / CT) * 16)) +
                                           (i % CT) * 16 * kRowBytes);
  };
  auto compute = [&](const uint8_t* buf, const uint8_t* bufn, const u32x4 (&nb)[RT],
                     const u32x4 (&nbn)[RT], int c, int s0, int s1) {
    const int ring0 = kEarly ? c * 4 * CT : 0;  // 16 CT is a multiple of the early ring's 4
#pragma unroll
    for (int s = s0; s < s1; ++s) {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        const int i = s * CT + ct, ia = i + kAhead;
        if (ia < 4 * CT)
          B[(ring0 + ia) % kRing] = readb(buf, ia);
        else if (kEarly)
          B[(ring0 + ia) % kRing] = readb(bufn, ia - 4 * CT);
        // this step's share of the next k-step's 2 RT half decodes
#pragma unroll
        for (int q = ct * 2 * RT / CT; q < (ct + 1) * 2 * RT / CT; ++q) {
          const int r = q >> 1, h = q & 1;
          if (s < 3)
            decode_half(A[(s + 1) & 1][r], nb[r], tb[r], c, s + 1, h);
          else if (c < 3)
            decode_half(A[0][r], nbn[r], tb[r], c + 1, 0, h);
          else
            decode_half(A[0][r], nbn[r], tbn[r], 0, 0, h);
        }
#pragma unroll
        for (int r = 0; r < RT; ++r)
          acc[r][ct] = mfma<XDT>(A[s & 1][r], B[(ring0 + i) % kRing], acc[r][ct]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  uint8_t* const bufs[4] = {xb0, xb1, NB == 4 ? xb2 : xb0, NB == 4 ? xb3 : xb1};
  if (nsp > 0) {
    load_tab(sp0, tb);
#pragma unroll
    for (int c = 0; c < D; ++c) {
      load_nib(sp0, c, nib[c]);
      stage(sp0, c, bufs[c]);
      request_group_end();
    }
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      decode_half(A[0][r], nib[0][r], tb[r], 0, 0, 0);
      decode_half(A[0][r], nib[0][r], tb[r], 0, 0, 1);
    }
    if constexpr (kEarly) {  // the first chunk: D - 1 chunks' requests are younger
      wait_barrier<(D - 1) * (XD + RT)>();
#pragma unroll
      for (int i = 0; i < kAhead; ++i) B[i] = readb(bufs[0], i);
    }
    for (int sp = sp0; sp < sp1; ++sp) {
      const int spn = min(sp + 1, sp1 - 1);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int cn = (c + D) & 3;
        const int spx = c + D >= 4 ? spn : sp;
        // Every chunk requests XD pieces of x and RT nibble chunks (and sometimes tables), so at
        // most k chunks' worth of requests in flight means that all older ones have arrived.
        // Past the barrier every wave's part of them has.
        if constexpr (kEarly) {
          // In the middle of chunk c: the next one must be there (the one after it is still on
          // its way), and every wave is done with the one before, whose place the request
          // takes.  So B operands can be read ahead across the chunk's end.
          compute(bufs[c], bufs[(c + 1) & 3], nib[c], nib[(c + 1) & 3], c, 0, 2);
          wait_barrier<XD + RT>();
        } else {
          // chunk c is there (D - 1 younger ones may not be), and every wave is done with the
          // one before
          wait_barrier<(D - 1) * (XD + RT)>();
        }
        load_nib(spx, cn, nib[cn % NB]);
        if (cn == 0) load_tab(spx, tbn);
        stage(spx, cn, bufs[cn]);
        if constexpr (kEarly) {
          compute(bufs[c], bufs[(c + 1) & 3], nib[c], nib[(c + 1) & 3], c, 2, 4);
        } else {
#pragma unroll
          for (int i = 0; i < kAhead; ++i) B[i] = readb(bufs[c], i);
          compute(bufs[c], nullptr, nib[c % NB], nib[(c + 1) % NB], c, 0, 4);
        }
      }
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        tb[r][0] = tbn[r][0];
        tb[r][1] = tbn[r][1];
      }
    }
  }

  // lane: x row 16 ct + lane % 16, weight rows 4 (lane / 16) .. + 3 of each row tile
  if (a.bias && !a.part) {
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      f32x4 b;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        b[e] = load_as_float(a.bias, min((t0 + r) * 16 + (lane >> 4) * 4 + e, a.N - 1), a.bdt);
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) acc[r][ct] += b;
    }
  }
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const int m = ct * 16 + (lane & 15);
    if (m >= rows) continue;
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const int n = (t0 + r) * 16 + (lane >> 4) * 4;
      const f32x4 v = acc[r][ct];
      const int64_t o = (int64_t)(m0 + m) * a.N + n;
      if (a.part) {
        float* dst = a.part + (int64_t)p * a.M * a.N + o;
        if (a.vec && n + 4 <= a.N) {
          *reinterpret_cast<f32x4*>(dst) = v;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < a.N) dst[e] = v[e];
        }
      } else if (a.vec && n + 4 <= a.N) {
        store4(a.y, o, v, a.ydt);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < a.N) store_y(a.y, o + e, v[e], a.ydt);
      }
    }
  }
}

// y = the P parts' sums added in part order (deterministic) plus the bias of column i % N, four
// outputs per thread.
__global__ __launch_bounds__(256) void gemm_sum(const float* __restrict__ part, int P, int64_t n,
                                                void* __restrict__ y, int ydt, int vec,
                                                const void* __restrict__ bias, int bdt, int N) {
  const int64_t i0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i0 >= n) return;
  if (vec) {
    f32x4 a = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(part + i0));
#pragma unroll 4
    for (int p = 1; p < P; ++p)
      a += __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(part + (int64_t)p * n + i0));
    if (bias) {  // vec: N % 4 == 0, so the four columns are consecutive
      const int c = (int)(i0 % N);
#pragma unroll
      for (int e = 0; e < 4; ++e) a[e] += load_as_float(bias, c + e, bdt);
    }
    store4(y, i0, a, ydt);
  } else {
    for (int64_t i = i0; i < min(n, i0 + 4); ++i) {
      float a = part[i];
      for (int p = 1; p < P; ++p) a += part[(int64_t)p * n + i];
      if (bias) a += load_as_float(bias, i % N, bdt);
      store_y(y, i, a, ydt);
    }
  }
}

// y[m, n] += bias[n] for the GEMV's 1 to 16 rows, rounded as torch's y.add_(bias.to(y.dtype)):
// the bias to y's dtype, then the sum.
template <typename T>
__global__ __launch_bounds__(256) void add_bias_kernel(T* __restrict__ y, int64_t n, int N,
                                                       const void* __restrict__ bias, int bdt) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  y[i] = (T)((float)y[i] + (float)(T)load_as_float(bias, i % N, bdt));
}

// x [M, K] of one dtype -> [M, ld] of another (round to nearest even), zeros past K: the
// conversion and the padding to whole groups in one pass.  8 outputs per thread.
__global__ __launch_bounds__(256) void cast_rows_kernel(const void* __restrict__ x, int xdt,
                                                        int64_t M, int K,
                                                        uint16_t* __restrict__ out, int odt,
                                                        int ld) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;
  if (i >= M * ld) return;
  const int64_t m = i / ld;
  const int k = (int)(i - m * ld);
  const int64_t at = m * K + k;
  unsigned h[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float v = 0.f;
    if (k + e < K) v = load_as_float(x, at + e, xdt);
    h[e] = odt == FB_DT_F16 ? __builtin_bit_cast(unsigned short, (_Float16)v)
                            : __builtin_bit_cast(unsigned short, (__bf16)v);
  }
  *reinterpret_cast<u32x4*>(out + i) = u32x4{h[0] | (h[1] << 16), h[2] | (h[3] << 16),
                                             h[4] | (h[5] << 16), h[6] | (h[7] << 16)};
}

// ---------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------
// Tile shapes the plan chooses from, with the time in us that a span (512 K-values) of one
// tile takes on a CU when one workgroup runs there and when two do (both done).  Fitted to
// timings of every shape and part count over M = 17..2048 on 4096^2, 8192^2, 4096 -> 11008,
// 11008 -> 4096 and 8192 -> 28672.  Timed again with every shape and part count on those and on
// 1024^2 and 896 -> 300 (126 cases, profiles/gemm_plan_vs_all_tiles.md): the plan it picks is
// 0.6% (geometric mean; 9.4% at worst) from the best.  A table rather than a formula because the costs follow no
// simple one: small tiles are bound by latency and the x fill, GF4's wide ones by instruction
// issue (RT = 4 does not fit two workgroups' registers there), E2M1's by the MFMAs.
struct GemmShape {
  int rt, ct;
  float one, two;
};
constexpr GemmShape kGf4Shapes[] = {{3, 8, 5.65f, 9.84f}, {3, 6, 4.52f, 8.04f},
                                    {2, 8, 4.08f, 7.35f}, {2, 6, 3.26f, 5.82f},
                                    {2, 4, 2.69f, 4.82f}, {2, 3, 2.36f, 3.93f},
                                    {2, 2, 1.94f, 3.34f}};
constexpr GemmShape kE2m1Shapes[] = {{4, 8, 5.32f, 8.83f}, {4, 6, 3.89f, 6.70f},
                                     {4, 4, 2.74f, 4.85f}, {3, 6, 3.04f, 5.44f},
                                     {4, 3, 2.23f, 4.12f}, {2, 4, 1.55f, 3.15f},
                                     {2, 3, 1.28f, 2.39f}, {2, 2, 1.08f, 1.86f}};
// the same fits' cost of a part-sum launch and of its traffic per million fp32 sums
constexpr float kSumCost[] = {2.32f, 2.68f}, kSumPerMillion[] = {1.27f, 1.25f};
constexpr int kMaxParts = 8;
constexpr int64_t kMaxPartBytes = 256ll << 20;

struct GemmPlan {
  int rt = 0, ct = 0, P = 1;
};

template <size_t NS>
GemmPlan gemm_plan(const fb_shape_t* s, int cus, const GemmShape (&shapes)[NS], double sum_cost,
                   double sum_per_million) {
  const int GS = (s->K / 128 + 3) / 4;
  GemmPlan best;
  double bt = 0;
  for (const GemmShape& c : shapes) {
    const int64_t T = (int64_t)((s->N + c.rt * 64 - 1) / (c.rt * 64)) *
                      ((s->B + c.ct * 16 - 1) / (c.ct * 16));
    for (int P = 1; P <= kMaxParts && P <= GS; ++P) {
      const int S = (GS + P - 1) / P;
      if (S * (P - 1) >= GS) continue;  // an empty part
      if (P > 1 && 4 * (int64_t)P * s->B * s->N > kMaxPartBytes) break;
      const int64_t slots = 2 * (int64_t)cus, full = T * P / slots, rem = T * P % slots;
      double t = S * (full * c.two + (rem == 0 ? 0.0 : rem <= cus ? c.one : c.two));
      if (P > 1) t += sum_cost + sum_per_million * 1e-6 * s->B * (double)s->N * P;
      if (!best.rt || t < bt) {
        bt = t;
        best.rt = c.rt;
        best.ct = c.ct;
        best.P = P;
      }
    }
  }
  return best;
}

GemmPlan gemm_plan(const fb_shape_t* s, int cus) {
  return s->fmt == FB_FMT_GF4 ? gemm_plan(s, cus, kGf4Shapes, kSumCost[0], kSumPerMillion[0])
                              : gemm_plan(s, cus, kE2m1Shapes, kSumCost[1], kSumPerMillion[1]);
}

template <int FMT, int XDT, int RT, int CT>
int launch_gemm(GemmArgs a, int P, hipStream_t hs) {
  using T = GemmTile<RT, CT>;
  a.tiles_n = (a.N + T::kRows - 1) / T::kRows;
  a.tiles_m = (a.M + T::kCols - 1) / T::kCols;
  a.spp = (a.GS + P - 1) / P;
  const int64_t grid = (int64_t)a.tiles_n * a.tiles_m * P;
  if (grid > INT32_MAX) return FB_ERR_SHAPE;
  hipLaunchKernelGGL((gemm_kernel<FMT, XDT, RT, CT>), dim3((unsigned)grid),
                     dim3(kGemmWaves * 64), 0, hs, a);
  return hipGetLastError() == hipSuccess ? FB_OK : FB_ERR_HIP;
}

template <int FMT, int XDT>
int launch_gemm_tile(const GemmArgs& a, const GemmPlan& pl, hipStream_t hs) {
  const int shape = pl.rt * 100 + pl.ct;
  if constexpr (FMT == FB_FMT_GF4) {
    if (shape == 308) return launch_gemm<FMT, XDT, 3, 8>(a, pl.P, hs);
    if (shape == 208) return launch_gemm<FMT, XDT, 2, 8>(a, pl.P, hs);
    if (shape == 206) return launch_gemm<FMT, XDT, 2, 6>(a, pl.P, hs);
  } else {
    if (shape == 408) return launch_gemm<FMT, XDT, 4, 8>(a, pl.P, hs);
    if (shape == 406) return launch_gemm<FMT, XDT, 4, 6>(a, pl.P, hs);
    if (shape == 404) return launch_gemm<FMT, XDT, 4, 4>(a, pl.P, hs);
    if (shape == 403) return launch_gemm<FMT, XDT, 4, 3>(a, pl.P, hs);
  }
  switch (shape) {
    case 306: return launch_gemm<FMT, XDT, 3, 6>(a, pl.P, hs);
    case 204: return launch_gemm<FMT, XDT, 2, 4>(a, pl.P, hs);
    case 203: return launch_gemm<FMT, XDT, 2, 3>(a, pl.P, hs);
    default: return launch_gemm<FMT, XDT, 2, 2>(a, pl.P, hs);
  }
}

// x (rotated already where the layer is) times W^T with the parts' sums in ws (pl.P > 1).
int gemm_run(const void* wdev, const void* x, void* y, const fb_shape_t* s, const GemmPlan& pl,
             const void* bias, int bdt, void* ws, hipStream_t hs) {
  GemmArgs a{};
  a.w = static_cast<const uint8_t*>(wdev);
  a.x = x;
  a.y = y;
  a.part = pl.P > 1 ? static_cast<float*>(ws) : nullptr;
  a.M = s->B;
  a.N = s->N;
  a.K = s->K;
  a.GS = (s->K / 128 + 3) / 4;
  a.ydt = s->y_dtype;
  a.bias = bias;
  a.bdt = bdt;
  a.vec = (s->N & 3) == 0 && (reinterpret_cast<uintptr_t>(y) & 15u) == 0;
  int st;
  if (s->fmt == FB_FMT_GF4)
    st = launch_gemm_tile<FB_FMT_GF4, FB_DT_F16>(a, pl, hs);
  else if (s->x_dtype == FB_DT_BF16)
    st = launch_gemm_tile<FB_FMT_E2M1, FB_DT_BF16>(a, pl, hs);
  else
    st = launch_gemm_tile<FB_FMT_E2M1, FB_DT_F16>(a, pl, hs);
  if (st != FB_OK || pl.P == 1) return st;
  return fb_gpu::sum_parts(a.part, pl.P, (int64_t)s->B * s->N, y, s->y_dtype, a.vec, bias, bdt,
                           s->N, hs);
}

size_t rot_bytes(const fb_shape_t* s) {
  return s->fwht_block ? ((size_t)s->B * s->K * 2 + 255) & ~size_t(255) : 0;
}

// A tile's x rows and a weight tile's stream are addressed with 32-bit byte offsets.
int gemm_check(const fb_shape_t* s) {
  const int st = fb_validate(s);
  if (st != FB_OK) return st;
  if (s->K > (1 << 22) || s->B > (1 << 24)) return FB_ERR_SHAPE;
  if (s->fwht_block && s->x_dtype != FB_DT_F16) return FB_ERR_DTYPE;
  return FB_OK;
}

}  // namespace

// y[i] = part 0's + part 1's + ... sum i, plus bias[i % N] where there is one, for n sums (vec:
// n % 4 == 0, N % 4 == 0 with a bias, and y 16-byte aligned)
int fb_gpu::sum_parts(const float* part, int P, int64_t n, void* y, int ydt, int vec,
                      const void* bias, int bdt, int N, hipStream_t hs) {
  if ((n + 1023) / 1024 > INT32_MAX) return FB_ERR_SHAPE;
  hipLaunchKernelGGL(gemm_sum, dim3((unsigned)((n + 1023) / 1024)), dim3(256), 0, hs, part, P, n,
                     y, ydt, vec, bias, bdt, N);
  return hipGetLastError() == hipSuccess ? FB_OK : FB_ERR_HIP;
}

extern "C" {

int fb_add_bias(void* y, int32_t y_dtype, int32_t M, int32_t N, const void* bias,
                int32_t bias_dtype, void* stream) {
  if (!y || !bias) return FB_ERR_NULL;
  if (M < 1 || N < 1) return FB_ERR_SHAPE;
  if (bias_dtype != FB_DT_F16 && bias_dtype != FB_DT_BF16 && bias_dtype != FB_DT_F32)
    return FB_ERR_DTYPE;
  if ((reinterpret_cast<uintptr_t>(bias) & (bias_dtype == FB_DT_F32 ? 3u : 1u)) ||
      (reinterpret_cast<uintptr_t>(y) & (y_dtype == FB_DT_F32 ? 3u : 1u)))
    return FB_ERR_ALIGN;
  const int64_t n = (int64_t)M * N;
  if ((n + 255) / 256 > INT32_MAX) return FB_ERR_SHAPE;
  const dim3 grid((unsigned)((n + 255) / 256)), block(256);
  hipStream_t hs = static_cast<hipStream_t>(stream);
  if (y_dtype == FB_DT_F32)
    hipLaunchKernelGGL(add_bias_kernel<float>, grid, block, 0, hs, static_cast<float*>(y), n, N,
                       bias, bias_dtype);
  else if (y_dtype == FB_DT_F16)
    hipLaunchKernelGGL(add_bias_kernel<_Float16>, grid, block, 0, hs, static_cast<_Float16*>(y), n,
                       N, bias, bias_dtype);
  else if (y_dtype == FB_DT_BF16)
    hipLaunchKernelGGL(add_bias_kernel<__bf16>, grid, block, 0, hs, static_cast<__bf16*>(y), n, N,
                       bias, bias_dtype);
  else
    return FB_ERR_DTYPE;
  return hipGetLastError() == hipSuccess ? FB_OK : FB_ERR_HIP;
}

int fb_cast_rows(const void* x, int32_t x_dtype, int32_t M, int32_t K, void* out,
                 int32_t out_dtype, int32_t ld, void* stream) {
  if (!x || !out) return FB_ERR_NULL;
  if (M < 1 || K < 1 || ld < K || ld % 128) return FB_ERR_SHAPE;
  if ((x_dtype != FB_DT_F16 && x_dtype != FB_DT_BF16 && x_dtype != FB_DT_F32) ||
      (out_dtype != FB_DT_F16 && out_dtype != FB_DT_BF16))
    return FB_ERR_DTYPE;
  if ((reinterpret_cast<uintptr_t>(out) & 15u) ||
      (reinterpret_cast<uintptr_t>(x) & (x_dtype == FB_DT_F32 ? 3u : 1u)))
    return FB_ERR_ALIGN;
  const int64_t blocks = ((int64_t)M * ld / 8 + 255) / 256;
  if (blocks > INT32_MAX) return FB_ERR_SHAPE;
  hipLaunchKernelGGL(cast_rows_kernel, dim3((unsigned)blocks), dim3(256), 0,
                     static_cast<hipStream_t>(stream), x, x_dtype, (int64_t)M, K,
                     static_cast<uint16_t*>(out), out_dtype, ld);
  return hipGetLastError() == hipSuccess ? FB_OK : FB_ERR_HIP;
}

size_t fb_gemm_workspace_bytes(const fb_shape_t* s) {
  if (!s || gemm_check(s) != FB_OK) return 0;
  const GemmPlan pl = gemm_plan(s, fb_gpu::cu_count());
  return rot_bytes(s) + (pl.P > 1 ? ((size_t)pl.P * s->B * s->N * 4 + 255) & ~size_t(255) : 0);
}

int fb_gemm(const void* wdev, const void* x, void* y, const fb_shape_t* s, const void* bias,
            int32_t bias_dtype, void* ws, size_t ws_bytes, void* stream) {
  if (!s || !wdev || !x || !y) return FB_ERR_NULL;
  const int st = gemm_check(s);
  if (st != FB_OK) return st;
  if (bias) {
    if (bias_dtype != FB_DT_F16 && bias_dtype != FB_DT_BF16 && bias_dtype != FB_DT_F32)
      return FB_ERR_DTYPE;
    if (reinterpret_cast<uintptr_t>(bias) & (bias_dtype == FB_DT_F32 ? 3u : 1u))
      return FB_ERR_ALIGN;
  }
  if ((reinterpret_cast<uintptr_t>(wdev) & 15u) || (reinterpret_cast<uintptr_t>(x) & 15u) ||
      (reinterpret_cast<uintptr_t>(y) & 3u))
    return FB_ERR_ALIGN;
  hipStream_t hs = static_cast<hipStream_t>(stream);
  GemmPlan pl = gemm_plan(s, fb_gpu::cu_count());
  const size_t rot = rot_bytes(s);
  const size_t need = rot + (pl.P > 1 ? (size_t)pl.P * s->B * s->N * 4 : 0);
  if (need && !ws) return FB_ERR_NULL;
  if (need && (reinterpret_cast<uintptr_t>(ws) & 255u)) return FB_ERR_ALIGN;
  if (need > ws_bytes) return FB_ERR_WORKSPACE;
  if (rot) {
    const int rc = fb_gpu::rotate_rows(x, ws, s->B, s->K, s->fwht_block, hs);
    if (rc != FB_OK) return rc;
    x = ws;
  }
  return gemm_run(wdev, x, y, s, pl, bias, bias_dtype, static_cast<uint8_t*>(ws) + rot, hs);
}

}  // extern "C"
