// The activation gradient of the 4-bit linear layer: gx[M, K] = gy[M, N] . W[N, K].
//
// The contraction runs over the weight's rows, across the lanes of the device stream, so the
// stream cannot be an MFMA operand here.  Two passes instead of one fp32 decode and an fp32
// library GEMM:
//  1. grad_decode_kernel decodes W and transposes it through LDS into MFMA A operands of
//     16-bit values, 1 KiB per (16 k, 32 n), exact in every case: fp16 for GF4 (and E2M1 whose
//     scales allow it) against fp16 gy; else bf16, GF4's 11-bit values as two terms hi + lo.
//  2. grad_gemm_kernel multiplies them with gy, also held exactly in 16 bits: as it is, or a
//     wider gy as a sum of bf16 terms (fp16: 2, fp32: 3).  Every product of two terms is
//     exact in fp32, and all go into the same fp32 accumulators, so the result has the
//     precision of an fp32 GEMM of the exact weight.
// The matrix cores do 16-bit products 16 times as fast as fp32 ones, so even fp32 gy against
// GF4 (6 term pairs) is faster than an fp32 GEMM.  Measured (us; the fp32 decode and library
// GEMM of before): GF4 4096^2, M = 256, fp16 gy: 29 (about 190); GF4 8192^2, M = 1024: 163 fp16,
// 329 bf16, 819 fp32.  At M <= 64 it is bound by pass 1 (10 us + 0.35 us per million weights and
// plane: the 16-bit stores), beyond by the MFMAs (1,080 TFLOP/s at M = 1024).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "fourbit.h"
#include "fourbit_decode.h"
#include "fourbit_layout.h"

// Host helpers of fourbit_gemv.hip and fourbit_gemm.hip.  Not part of the library's ABI.
namespace fb_gpu {
__attribute__((visibility("hidden"))) int cu_count();
__attribute__((visibility("hidden"))) int sum_parts(const float* part, int P, int64_t n, void* y,
                                                    int ydt, int vec, const void* bias, int bdt,
                                                    int N, hipStream_t hs);
}  // namespace fb_gpu

namespace {

constexpr int kChunkN = 128;    // contraction values of one chunk: 4 k-steps of 32
constexpr int kTileBytes = 4096;  // one chunk of one 16-row A tile
constexpr int kGradWaves = 4;
constexpr int kRowBytes = 256;  // one gy row of a chunk

// ---------------------------------------------------------------------------------
// Pass 1.  Workgroup = (128 rows of W, one span): wave w holds the block of row tile 8q + w.
// For each 16-byte nibble chunk (128 k: 32 of each item) the 8 waves write their decoded
// values to LDS as [k][n] and read back 16-byte runs along n.  Memory-bound: the 16-bit
// stores are 2.7 (GF4) to 3.8 times the bytes read.
// LDS rows are 272 bytes and the items 32 bytes further apart, so that neither the 2-byte
// writes (16 n of 4 items per instruction) nor the 16-byte reads (16 k) meet in a bank.
// ---------------------------------------------------------------------------------
constexpr int kTRow = 272;
constexpr int kTItem = 32 * kTRow + 32;
constexpr int kTPlane = 4 * kTItem;

// MODE 0: fp16 values.  1: bf16 (E2M1, exact).  2: bf16 hi and lo terms (GF4).
template <int FMT, int MODE>
__global__ __launch_bounds__(512) void grad_decode_kernel(const uint8_t* __restrict__ w,
                                                          uint8_t* __restrict__ out, int T, int GS,
                                                          int sp0, int QN, int64_t plane) {
  constexpr int BB = FMT == FB_FMT_GF4 ? fb::kGf4BlockBytes : fb::kE2m1BlockBytes;
  constexpr int NP = MODE == 2 ? 2 : 1;
  __shared__ __align__(16) uint8_t lds[NP * kTPlane];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int q = blockIdx.x, spl = blockIdx.y;
  const int t = q * 8 + wave;
  Rec<FMT> r;
  if (t < T) {
    load_rec_global<FMT>(w + ((int64_t)t * GS + sp0 + spl) * BB, lane, r);
  } else {  // rows past the last tile: zeros
    r.t0 = r.t1 = u32x4{0, 0, 0, 0};
#pragma unroll
    for (int c = 0; c < 4; ++c) r.nib[c] = u32x4{0, 0, 0, 0};
  }
  uint8_t* const dst = lds + (lane >> 4) * kTItem + (wave * 16 + (lane & 15)) * 2;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int e = FMT == FB_FMT_GF4 ? 0 : (int)((r.t0.x >> (8 * c)) & 0xFFu) - 127;
    __syncthreads();
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      u32x4 pr;
      if constexpr (FMT == FB_FMT_GF4)
        pr = gf4_decode8(r.nib[c][d], r.t0, r.t1);
      else
        pr = e2m1_decode8<FB_DT_BF16>(r.nib[c][d], 1.0f);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const unsigned bits = (pr[j >> 1] >> (16 * (j & 1))) & 0xFFFFu;
        uint8_t* const p = dst + (d * 8 + j) * kTRow;
        if constexpr (FMT == FB_FMT_GF4 && MODE == 0) {
          *reinterpret_cast<unsigned short*>(p) = (unsigned short)bits;
        } else if constexpr (FMT == FB_FMT_GF4) {
          const float v = (float)__builtin_bit_cast(_Float16, (unsigned short)bits);
          const __bf16 hi = (__bf16)v;
          *reinterpret_cast<__bf16*>(p) = hi;
          *reinterpret_cast<__bf16*>(p + kTPlane) = (__bf16)(v - (float)hi);
        } else {
          const float v = __builtin_ldexpf(__builtin_bit_cast(float, bits << 16), e);
          if constexpr (MODE == 0)
            *reinterpret_cast<_Float16*>(p) = (_Float16)v;
          else
            *reinterpret_cast<__bf16*>(p) = (__bf16)v;
        }
      }
    }
    __syncthreads();
    // this wave's k-tile: item wave / 2, half wave % 2 of its 32 values
    const int i = wave >> 1, h = wave & 1;
    const int kt = spl * 32 + i * 8 + c * 2 + h;
    const uint8_t* src = lds + i * kTItem + (h * 16 + (lane & 15)) * kTRow + (lane >> 4) * 16;
    uint8_t* o = out + ((int64_t)kt * QN + q) * kTileBytes + lane * 16;
#pragma unroll
    for (int pl = 0; pl < NP; ++pl)
#pragma unroll
      for (int s = 0; s < 4; ++s)
        *reinterpret_cast<u32x4*>(o + pl * plane + s * 1024) =
            *reinterpret_cast<const u32x4*>(src + pl * kTPlane + s * 64);
  }
}

// gy [M, N] as planes of bf16 (fp16 copied to one fp16 plane) with rows of ld values, zeros
// past N.  The terms come from truncation, which cannot overflow: t0 = the upper 16 bits of the
// fp32 value, t1 those of what is left, t2 the rest; their sum is the value.  A non-finite
// value is its own t0 and has no other terms; `finite` (against W's lo terms, whose sign and
// zeros are not W's) holds t0 with non-finite values as 0.
struct GyPlanes {
  unsigned short* p[4];  // t0, finite t0, t1, t2 (null: not wanted)
};
__global__ __launch_bounds__(256) void grad_gy_kernel(const void* __restrict__ gy, int64_t M,
                                                      int N, int ld, int dt, GyPlanes g) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= M * ld) return;
  const int64_t m = i / ld;
  const int n = (int)(i - m * ld);
  const int64_t at = m * N + n;
  if (dt == FB_DT_F16 && !g.p[2]) {  // fp16 as it is
    g.p[0][i] = n < N ? static_cast<const unsigned short*>(gy)[at] : (unsigned short)0;
    return;
  }
  float v = 0.f;
  if (n < N)
    v = dt == FB_DT_F32   ? static_cast<const float*>(gy)[at]
        : dt == FB_DT_F16 ? (float)static_cast<const _Float16*>(gy)[at]
                          : __builtin_bit_cast(
                                float, (unsigned)static_cast<const unsigned short*>(gy)[at] << 16);
  const unsigned b = __builtin_bit_cast(unsigned, v);
  const bool fin = (b & 0x7F800000u) != 0x7F800000u;
  unsigned t0 = b & 0xFFFF0000u;
  if (!fin && (b & 0x007FFFFFu)) t0 |= 0x00400000u;  // NaN stays NaN when cut
  const float r1 = fin ? v - __builtin_bit_cast(float, t0) : 0.f;
  const unsigned t1 = __builtin_bit_cast(unsigned, r1) & 0xFFFF0000u;
  const float r2 = r1 - __builtin_bit_cast(float, t1);
  g.p[0][i] = (unsigned short)(t0 >> 16);
  if (g.p[1]) g.p[1][i] = fin ? (unsigned short)(t0 >> 16) : (unsigned short)0;
  if (g.p[2]) g.p[2][i] = (unsigned short)(t1 >> 16);
  if (g.p[3]) g.p[3][i] = (unsigned short)(__builtin_bit_cast(unsigned, r2) >> 16);
}

// ---------------------------------------------------------------------------------
// Pass 2.  The forward GEMM's structure (tile of 64 RT rows of W^T by 16 CT rows of gy, gy
// through LDS with direct loads and the same unit permutation, one barrier per chunk), with A
// operands read as they are, one chunk ahead, instead of decoded.  The chunks of all term
// pairs form one contraction.
// ---------------------------------------------------------------------------------
struct GradArgs {
  const uint8_t* a;     // A operands [plane][k-tile][QN][4 KiB]
  const uint8_t* b;     // gy planes
  void* gx;
  float* part;          // P > 1: fp32 sums [P, M, K]
  int64_t plane_a, plane_b;
  int M, Nb;            // rows of gy, values of a gy row that may be read
  int ldb;              // row stride of b in values
  int KT;               // k-tiles of this call
  int64_t ldx;          // gx row stride in values
  int k0, K;            // first column of gx, columns in all
  int QN, total, cpp;   // chunks per term pair, in all, per part
  int pa, pb;           // pair p: A plane (pa >> 4 p) & 15, gy plane (pb >> 4 p) & 15 (bits)
  int tiles_k, tiles_m;
  int dt, vec;
};

template <int RT, int CT>
struct GradTile {
  static constexpr int kRows = RT * 16 * kGradWaves;
  static constexpr int kCols = CT * 16;
  static constexpr int kBuf = kCols * kRowBytes;
  static constexpr int kBufs = kBuf * 4 <= 64 * 1024 ? 4 : 2;
  static_assert(kBuf * kBufs <= 80 * 1024, "two workgroups per CU");
};

template <int XDT, int RT, int CT>
__global__ __launch_bounds__(kGradWaves * 64, 2) void grad_gemm_kernel(
    GradArgs g) {
  using T = GradTile<RT, CT>;
  constexpr int NB = T::kBufs, D = NB - 1;
  constexpr int XD = CT;  // 1 KiB gy requests of one wave per chunk
  __shared__ __align__(1024) uint8_t xb0[T::kBuf], xb1[T::kBuf];
  __shared__ __align__(1024) uint8_t xb2[NB == 4 ? T::kBuf : 16], xb3[NB == 4 ? T::kBuf : 16];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int id = blockIdx.x;
  {
    const int total = gridDim.x, q = total >> 3, r = total & 7, xcd = id & 7, k = id >> 3;
    id = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + k;
  }
  const int per = g.tiles_k * g.tiles_m;
  const int p = id / per;
  id -= p * per;
  const int grp = id / (4 * g.tiles_k), gm = min(4, g.tiles_m - grp * 4);
  const int rem = id - grp * 4 * g.tiles_k;
  const int tk = rem / gm, tm = grp * 4 + (rem - tk * gm);

  const int c0 = p * g.cpp, c1 = min(g.total, c0 + g.cpp);
  const int m0 = tm * T::kCols, rows = min(T::kCols, g.M - m0);
  const int t0 = tk * (RT * kGradWaves) + wave * RT;
  const int64_t tile_bytes = (int64_t)g.QN * kTileBytes;

  unsigned xoff[4];
  int xn[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int row = (wave * XD + j) * 4 + (lane >> 4);
    const int u = (lane & 15) ^ (row & 15);
    xoff[j] = (unsigned)row * (unsigned)g.ldb * 2u + u * 16;
    xn[j] = u * 8;
  }
  // the last row of a tile ends with its readable values
  const int brange = ((rows - 1) * g.ldb + g.Nb) * 2;
  auto stage = [&](int c, uint8_t* buf) {
    const int pr = c / g.QN, q = c - pr * g.QN;
    const rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(g.b) + ((g.pb >> (4 * pr)) & 15) * g.plane_b +
            (int64_t)m0 * g.ldb * 2,
        (short)0, brange, kRsrcWord3);
    const int left = g.Nb - q * kChunkN;
#pragma unroll
    for (int j = 0; j < XD; ++j) {
      const unsigned off = xn[j & 3] < left
                               ? xoff[j & 3] + (unsigned)((j >> 2) * 16) * (unsigned)g.ldb * 2u +
                                     (unsigned)q * 256u
                               : kXOutOfRange;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rs, (lds_byte*)(buf + (wave * XD + j) * 1024), 16, off, 0, 0, 0);
    }
  };
  u32x4 A[2][RT][4];
  auto load_a = [&](int c, u32x4 (&d)[RT][4]) {
    const int pr = c / g.QN, q = c - pr * g.QN;
    const uint8_t* base = g.a + ((g.pa >> (4 * pr)) & 15) * g.plane_a;
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const int t = min(t0 + r, g.KT - 1);
      const u32x4* src = reinterpret_cast<const u32x4*>(base + t * tile_bytes +
                                                        (int64_t)q * kTileBytes) + lane;
#pragma unroll
      for (int s = 0; s < 4; ++s) d[r][s] = src[s * 64];
    }
  };
  f32x4 acc[RT][CT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) acc[r][ct] = f32x4{0.f, 0.f, 0.f, 0.f};

  // B operand of column tile ct, k-step s: gy row lane % 16, unit 4 s + lane / 16
  const unsigned rrow = (lane & 15) * kRowBytes;
  unsigned rs4[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) rs4[s] = rrow + (((s * 4 + (lane >> 4)) ^ (lane & 15)) << 4);
  auto compute = [&](const uint8_t* buf, const u32x4 (&a)[RT][4]) {
    u32x4 B[3];
    auto readb = [&](int i) {
      return *reinterpret_cast<const u32x4*>(buf + rs4[i / CT] + (i % CT) * 16 * kRowBytes);
    };
    B[0] = readb(0);
    B[1] = readb(1);
#pragma unroll
    for (int i = 0; i < 4 * CT; ++i) {
      if (i + 2 < 4 * CT) B[(i + 2) % 3] = readb(i + 2);
#pragma unroll
      for (int r = 0; r < RT; ++r)
        acc[r][i % CT] = mfma<XDT>(a[r][i / CT], B[i % 3], acc[r][i % CT]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  uint8_t* const bufs[4] = {xb0, xb1, NB == 4 ? xb2 : xb0, NB == 4 ? xb3 : xb1};
  if (c0 < c1) {
    load_a(c0, A[0]);
#pragma unroll
    for (int c = 0; c < D; ++c) {
      stage(min(c0 + c, c1 - 1), bufs[c]);
      request_group_end();
    }
    for (int cb = c0; cb < c1; cb += 4) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        // Chunk cb + c's gy was requested D chunks ago.  Younger requests: D - 1 chunks' gy,
        // and after the first chunks, which were requested before any other A operands, as
        // many chunks' A operands.
        if (cb == c0)
          wait_barrier<(D - 1) * XD>();
        else
          wait_barrier<(D - 1) * (XD + 4 * RT)>();
        load_a(min(cb + c + 1, c1 - 1), A[(c + 1) & 1]);
        stage(min(cb + c + D, c1 - 1), bufs[(c + D) & 3]);
        if (cb + c < c1) compute(bufs[c], A[c & 1]);
      }
    }
  }
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const int m = ct * 16 + (lane & 15);
    if (m >= rows) continue;
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      if (t0 + r >= g.KT) continue;
      const int k = g.k0 + (t0 + r) * 16 + (lane >> 4) * 4;
      const f32x4 v = acc[r][ct];
      const int64_t o = (int64_t)(m0 + m) * g.ldx + k;
      if (g.part) {
        float* d = g.part + (int64_t)p * g.M * g.ldx + o;
        if (g.vec && k + 4 <= g.K) {
          *reinterpret_cast<f32x4*>(d) = v;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (k + e < g.K) d[e] = v[e];
        }
      } else if (g.vec && k + 4 <= g.K) {
        store4(g.gx, o, v, g.dt);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (k + e < g.K) store_y(g.gx, o + e, v[e], g.dt);
      }
    }
  }
}

// ---------------------------------------------------------------------------------
// A rotated layer's gradient, rotated back: every `fb`-wide block of v [rows, K] (fp32) becomes
// H v / sqrt(fb), written as dt.  One workgroup per 4096 values of a row, 16 per thread: the
// butterflies of strides 1-8, 16-128 and 256-2048 run in registers, with the values redistributed
// through LDS between them (17 floats per 16: no bank conflict).  One read and one write of
// the gradient, so bound by memory.
// ---------------------------------------------------------------------------------
constexpr int kRotPiece = 4096;
__global__ __launch_bounds__(256) void grad_rotate_kernel(const float* __restrict__ v,
                                                          void* __restrict__ out, int K,
                                                          int pieces, int fb, float sc, int dt) {
  __shared__ float l[kRotPiece / 16 * 17];
  const int t = threadIdx.x;
  const int64_t row = blockIdx.x / pieces;
  const int k0 = (int)(blockIdx.x - row * pieces) * kRotPiece;
  const int kw = min(kRotPiece, K - k0);  // whole blocks, a multiple of 128
  const float* src = v + row * K + k0;
  float x[16];
  auto stages = [&](int h0) {
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      if ((h0 << b) >= fb) break;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        if (i & (1 << b)) continue;
        const float a = x[i], c = x[i | (1 << b)];
        x[i] = a + c;
        x[i | (1 << b)] = a - c;
      }
    }
  };
  auto at = [](int i) { return i + (i >> 4); };
#pragma unroll
  for (int e = 0; e < 16; e += 4) {
    f32x4 f{0.f, 0.f, 0.f, 0.f};
    if (16 * t + e < kw) f = *reinterpret_cast<const f32x4*>(src + 16 * t + e);
#pragma unroll
    for (int j = 0; j < 4; ++j) x[e + j] = f[j];
  }
  stages(1);
#pragma unroll
  for (int e = 0; e < 16; ++e) l[at(16 * t + e)] = x[e];
  __syncthreads();
  const int b0 = (t >> 4) * 256 + (t & 15);
#pragma unroll
  for (int e = 0; e < 16; ++e) x[e] = l[at(b0 + 16 * e)];
  stages(16);
#pragma unroll
  for (int e = 0; e < 16; ++e) l[at(b0 + 16 * e)] = x[e];  // the places this thread read
  __syncthreads();
#pragma unroll
  for (int e = 0; e < 16; ++e) x[e] = l[at(256 * e + t)];
  stages(256);
#pragma unroll
  for (int e = 0; e < 16; ++e)
    if (256 * e + t < kw) store_y(out, row * K + k0 + 256 * e + t, x[e] * sc, dt);
}

// gb[n] = sum over m of gy[m, n], fp32 sums in a fixed order: a workgroup takes 16 columns, its 64
// row groups (4 to a wave) every 64th row, then 16 threads add the 64 sums in order.  Few columns
// per workgroup because it is bound by the latency of M / 64 dependent reads (64 columns and 16
// row groups: 7.8 us at 256 x 4096).
__global__ __launch_bounds__(1024) void grad_bias_kernel(const void* __restrict__ gy, int M, int N,
                                                         int dt, void* __restrict__ gb, int odt) {
  __shared__ float l[64][17];
  const int col = threadIdx.x & 15, row = threadIdx.x >> 4;
  const int n = blockIdx.x * 16 + col;
  float a = 0.f;
  if (n < N) {
#pragma unroll 8
    for (int m = row; m < M; m += 64) a += load_as_float(gy, (int64_t)m * N + n, dt);
  }
  l[row][col] = a;
  __syncthreads();
  if (row == 0 && n < N) {
    float s = l[0][col];
#pragma unroll
    for (int w = 1; w < 64; ++w) s += l[w][col];
    store_y(gb, n, s, odt);
  }
}

// The same for many rows: column sums of a run of rows per workgroup, for grad_bias_kernel (or
// another of this) to add.  gy is read as m rows of W = q N values, so that 8 values of 16 bytes
// (fp32: 32) per lane fill a workgroup's 512 columns whatever N is; the workgroup's waves take
// every 4th of its R rows, and their sums are added in order through LDS.  The rows past m q, less
// than W values, go to the sums as they are.  Bound by memory.
template <int DT>
__global__ __launch_bounds__(256) void grad_bias_part_kernel(const void* __restrict__ gy, int64_t m,
                                                             int64_t W, int64_t R, int64_t tail,
                                                             int P, int vec,
                                                             float* __restrict__ part) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t b0 = (int64_t)blockIdx.x * 512;
  if ((int)blockIdx.y == P) {
    for (int64_t c = b0 + threadIdx.x; c < b0 + 512 && c < tail; c += 256)
      part[(int64_t)P * W + c] = load_as_float(gy, m * W + c, DT);
    return;
  }
  __shared__ __align__(16) float l[4][512];
  const int64_t c0 = b0 + lane * 8;  // W % 8 == 0
  const int64_t r0 = (int64_t)blockIdx.y * R, r1 = min(m, r0 + R);
  float a[8] = {};
  auto add = [&](int64_t at) {
    if (!vec) {
#pragma unroll
      for (int e = 0; e < 8; ++e) a[e] += load_as_float(gy, at + e, DT);
    } else if constexpr (DT == FB_DT_F32) {
      const f32x4* p = reinterpret_cast<const f32x4*>(static_cast<const float*>(gy) + at);
      const f32x4 x = p[0], y = p[1];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        a[e] += x[e];
        a[4 + e] += y[e];
      }
    } else {
      const u32x4 v = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(gy) + at);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const unsigned short h = (unsigned short)(v[e >> 1] >> (16 * (e & 1)));
        a[e] += DT == FB_DT_F16 ? (float)__builtin_bit_cast(_Float16, h)
                                : (float)__builtin_bit_cast(__bf16, h);
      }
    }
  };
  if (c0 < W) {
#pragma unroll 8
    for (int64_t r = r0 + wave; r < r1; r += 4) add(r * W + c0);
  }
  *reinterpret_cast<f32x4*>(&l[wave][lane * 8]) = f32x4{a[0], a[1], a[2], a[3]};
  *reinterpret_cast<f32x4*>(&l[wave][lane * 8 + 4]) = f32x4{a[4], a[5], a[6], a[7]};
  __syncthreads();
  for (int c = threadIdx.x; c < 512 && b0 + c < W; c += 256)
    part[(int64_t)blockIdx.y * W + b0 + c] = ((l[0][c] + l[1][c]) + l[2][c]) + l[3][c];
}

// ---------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------
// Whether grad_bias_kernel sums a gradient by itself.  Measured (us, one launch / parts; fp16 unless
// said): 2048 x 48 7.1 / 8.1, 4096 x 48 12.5 / 7.7, 2^18 x 48 1423 / 12 (torch's sum 25), 1024 x 4096
// 5.6 / 7.9, 1025 x 11008 18.0 / 8.6, 65536 x 4096 545 / 93 (torch 113), 16384 x 28672 fp32 589 / 339.
bool bias_alone(int64_t M, int64_t N) {
  return M <= 2048 && (M <= 64 || M * N <= (6 << 20));
}

// One pass of grad_bias_part_kernel over M rows of N values.
struct BiasParts {
  int64_t q, m, W, R;
  int P;
  int64_t rows;  // of the sums it leaves
};
BiasParts bias_parts(int64_t M, int64_t N) {
  BiasParts b;
  b.q = N >= 64 ? 8 : 512 / N / 8 * 8;
  b.m = M / b.q;
  b.W = b.q * N;
  // About four workgroups of 256 threads per CU, of 32 rows at least (8 per wave in flight) and
  // 1024 at most (256 additions in a row, whatever M is).
  const int64_t wide = (b.W + 511) / 512;
  const int64_t fill = std::min((1024 + wide - 1) / wide, (b.m + 31) / 32);
  b.P = (int)std::min<int64_t>(std::max(fill, (b.m + 1023) / 1024), 65000);  // the grid's y range
  b.R = (b.m + b.P - 1) / b.P;
  b.rows = b.P * b.q + (M - b.m * b.q);
  return b;
}

int launch_bias_parts(const void* gy, int dt, int64_t M, int64_t N, const BiasParts& b, float* part,
                      hipStream_t hs) {
  const int64_t tail = (M - b.m * b.q) * N;
  const dim3 grid((unsigned)((b.W + 511) / 512), (unsigned)(b.P + (tail ? 1 : 0)));
  const int vec = (reinterpret_cast<uintptr_t>(gy) & 15u) == 0;
  if (dt == FB_DT_F32)
    hipLaunchKernelGGL(grad_bias_part_kernel<FB_DT_F32>, grid, dim3(256), 0, hs, gy, b.m, b.W, b.R,
                       tail, b.P, vec, part);
  else if (dt == FB_DT_F16)
    hipLaunchKernelGGL(grad_bias_part_kernel<FB_DT_F16>, grid, dim3(256), 0, hs, gy, b.m, b.W, b.R,
                       tail, b.P, vec, part);
  else
    hipLaunchKernelGGL(grad_bias_part_kernel<FB_DT_BF16>, grid, dim3(256), 0, hs, gy, b.m, b.W, b.R,
                       tail, b.P, vec, part);
  return hipGetLastError() == hipSuccess ? FB_OK : FB_ERR_HIP;
}

constexpr int64_t kMaxOperandBytes = 256ll << 20;  // transposed weight held at once
constexpr int kMaxRowsW = 1 << 18;  // one span of these is 256 MiB of 16-bit operands per plane
constexpr int64_t kMaxPartBytes = 256ll << 20;
constexpr int kMaxParts = 8;

size_t align256(size_t v) { return (v + 255) & ~size_t(255); }

// Tile shapes with the time in us that a chunk (128 contraction values) of one tile takes on a
// CU when one workgroup runs there and when two do.  Fitted to timings of these and of six other
// shapes at every part count, over M = 17..1024, 1 to 6 term pairs and 5 layers of 1024 -> 2048 to
// 8192^2.  Timed again with every shape and part count (80 cases of 4096^2 to 8192 -> 28672,
// profiles/gemm_plan_vs_all_tiles.md): the whole call on the plan it picks is 1.6% (geometric
// mean; 11.6% at worst) from the best.
struct GradShape {
  int rt, ct;
  float one, two;
};
constexpr GradShape kGradShapes[] = {
    {3, 8, 1.41f, 2.39f}, {2, 8, 1.05f, 1.84f}, {2, 4, 0.66f, 1.21f}, {2, 2, 0.50f, 0.92f}};
constexpr float kSumCost = 4.6f, kSumPerMillion = 1.17f;  // the part sum's, the same fit

struct GradPlan {
  int mode = 0;      // grad_decode_kernel's MODE
  int xdt = 0;       // operand dtype
  int pairs = 1, pa = 0, pb = 0;
  int a_planes = 1;
  int b_planes = 0;  // 0: gy itself is the operand
  int want = 0;      // terms of gy to make: bit 0 t0, 1 finite t0, 2 t1, 3 t2
  int QN = 0, GS = 0, ldb = 0;
  int spans = 0;     // spans of K decoded at once
  int rt = 0, ct = 0, P = 1;
  size_t a_bytes = 0, b_bytes = 0, part_bytes = 0, rot_bytes = 0;
  size_t total() const { return a_bytes + b_bytes + part_bytes + rot_bytes; }
};

void grad_tiles(GradPlan& pl, int M, int K, int cus) {
  const int total = pl.pairs * pl.QN;
  double bt = 0;
  bool have = false;
  for (const GradShape& c : kGradShapes) {
    const int kw = std::min(K, pl.spans * 512);
    const int64_t T = (int64_t)((kw + c.rt * 64 - 1) / (c.rt * 64)) *
                      ((M + c.ct * 16 - 1) / (c.ct * 16));
    for (int P = 1; P <= kMaxParts && P <= total; ++P) {
      const int S = (total + P - 1) / P;
      if (S * (P - 1) >= total) continue;
      if (P > 1 && 4 * (int64_t)P * M * K > kMaxPartBytes) break;
      const int64_t slots = 2 * (int64_t)cus, full = T * P / slots, rem = T * P % slots;
      double t = S * (full * c.two + (rem == 0 ? 0.0 : rem <= cus ? c.one : c.two));
      if (P > 1) t += kSumCost + kSumPerMillion * 1e-6 * M * (double)K * P;
      if (!have || t < bt) {
        have = true;
        bt = t;
        pl.rt = c.rt;
        pl.ct = c.ct;
        pl.P = P;
      }
    }
  }
}

// s->y_dtype is gy's dtype.
int grad_plan(const fb_shape_t* s, const void* gy, int f16_exact, GradPlan& pl) {
  const int st = fb_validate(s);
  if (st != FB_OK) return st;
  if (s->N > kMaxRowsW || s->B > (1 << 24)) return FB_ERR_SHAPE;
  const bool gf4 = s->fmt == FB_FMT_GF4;
  const int dt = s->y_dtype;
  if (dt == FB_DT_F16 && (gf4 || f16_exact)) {
    pl.mode = 0;
    pl.xdt = FB_DT_F16;
    pl.want = 1;
  } else {
    pl.xdt = FB_DT_BF16;
    pl.mode = gf4 ? 2 : 1;
    const int terms = dt == FB_DT_BF16 ? 1 : dt == FB_DT_F16 ? 2 : 3;
    pl.want = 1 | (gf4 ? 2 : 0) | (terms > 1 ? 4 : 0) | (terms > 2 ? 8 : 0);
    pl.pairs = 0;
    auto pair = [&](int a, int b) {
      pl.pa |= a << (4 * pl.pairs);
      pl.pb |= b << (4 * pl.pairs);
      ++pl.pairs;
    };
    pair(0, 0);
    if (gf4) pair(1, 1);
    for (int t = 1; t < terms; ++t) {
      pair(0, (gf4 ? 1 : 0) + t);
      if (gf4) pair(1, 1 + t);
    }
  }
  pl.a_planes = pl.mode == 2 ? 2 : 1;
  pl.QN = (s->N + kChunkN - 1) / kChunkN;
  pl.GS = (s->K / 128 + 3) / 4;
  // a 16-bit gy of one term is read in place where its rows are 16-byte aligned
  const bool direct = pl.want == 1 && dt != FB_DT_F32 && s->N % 8 == 0 &&
                      (reinterpret_cast<uintptr_t>(gy) & 15u) == 0;
  pl.b_planes = direct ? 0 : __builtin_popcount(pl.want);
  pl.ldb = direct ? s->N : pl.QN * kChunkN;
  const int64_t span_bytes = (int64_t)pl.a_planes * 32 * pl.QN * kTileBytes;
  pl.spans = (int)std::max<int64_t>(1, std::min<int64_t>(pl.GS, kMaxOperandBytes / span_bytes));
  grad_tiles(pl, s->B, s->K, fb_gpu::cu_count());
  pl.a_bytes = (size_t)(span_bytes * pl.spans);
  pl.b_bytes = align256((size_t)pl.b_planes * s->B * pl.ldb * 2);
  pl.part_bytes = pl.P > 1 ? align256((size_t)pl.P * s->B * s->K * 4) : 0;
  pl.rot_bytes = s->fwht_block ? align256((size_t)s->B * s->K * 4) : 0;
  return FB_OK;
}

template <int XDT, int RT, int CT>
int launch_grad(GradArgs g, int P, int kw, hipStream_t hs) {
  using T = GradTile<RT, CT>;
  g.tiles_k = (kw + T::kRows - 1) / T::kRows;
  g.tiles_m = (g.M + T::kCols - 1) / T::kCols;
  const int64_t grid = (int64_t)g.tiles_k * g.tiles_m * P;
  if (grid > INT32_MAX) return FB_ERR_SHAPE;
  hipLaunchKernelGGL((grad_gemm_kernel<XDT, RT, CT>), dim3((unsigned)grid),
                     dim3(kGradWaves * 64), 0, hs, g);
  return hipGetLastError() == hipSuccess ? FB_OK : FB_ERR_HIP;
}

template <int XDT>
int launch_grad_tile(const GradArgs& g, const GradPlan& pl, int kw, hipStream_t hs) {
  switch (pl.rt * 100 + pl.ct) {
    case 308: return launch_grad<XDT, 3, 8>(g, pl.P, kw, hs);
    case 208: return launch_grad<XDT, 2, 8>(g, pl.P, kw, hs);
    case 204: return launch_grad<XDT, 2, 4>(g, pl.P, kw, hs);
    default: return launch_grad<XDT, 2, 2>(g, pl.P, kw, hs);
  }
}

int launch_decode(const GradPlan& pl, const fb_shape_t* s, const void* wdev, uint8_t* out, int sp0,
                  int nsp, int64_t plane, hipStream_t hs) {
  const dim3 grid(pl.QN, nsp), block(512);
  const int T = (s->N + 15) / 16;
  const uint8_t* w = static_cast<const uint8_t*>(wdev);
  if (s->fmt == FB_FMT_GF4) {
    if (pl.mode == 0)
      hipLaunchKernelGGL((grad_decode_kernel<FB_FMT_GF4, 0>), grid, block, 0, hs, w, out, T, pl.GS,
                         sp0, pl.QN, plane);
    else
      hipLaunchKernelGGL((grad_decode_kernel<FB_FMT_GF4, 2>), grid, block, 0, hs, w, out, T, pl.GS,
                         sp0, pl.QN, plane);
  } else if (pl.mode == 0) {
    hipLaunchKernelGGL((grad_decode_kernel<FB_FMT_E2M1, 0>), grid, block, 0, hs, w, out, T, pl.GS,
                       sp0, pl.QN, plane);
  } else {
    hipLaunchKernelGGL((grad_decode_kernel<FB_FMT_E2M1, 1>), grid, block, 0, hs, w, out, T, pl.GS,
                       sp0, pl.QN, plane);
  }
  return hipGetLastError() == hipSuccess ? FB_OK : FB_ERR_HIP;
}

int grad_run(const GradPlan& pl, const fb_shape_t* s, const void* wdev, const void* gy, void* gx,
             int gx_dtype, uint8_t* ws, hipStream_t hs) {
  uint8_t* const aw = ws;
  uint8_t* const bw = aw + pl.a_bytes;
  float* const part = reinterpret_cast<float*>(bw + pl.b_bytes);
  float* const rot = reinterpret_cast<float*>(bw + pl.b_bytes + pl.part_bytes);
  GradArgs g{};
  g.a = aw;
  g.b = pl.b_planes ? bw : static_cast<const uint8_t*>(gy);
  g.gx = s->fwht_block ? rot : gx;
  g.dt = s->fwht_block ? FB_DT_F32 : gx_dtype;
  g.part = pl.P > 1 ? part : nullptr;
  g.M = s->B;
  g.Nb = pl.b_planes ? pl.ldb : s->N;
  g.ldb = pl.ldb;
  g.ldx = s->K;
  g.K = s->K;
  g.QN = pl.QN;
  g.total = pl.pairs * pl.QN;
  g.cpp = (g.total + pl.P - 1) / pl.P;
  g.pa = pl.pa;
  g.pb = pl.pb;
  g.plane_b = (int64_t)s->B * pl.ldb * 2;
  g.vec = (reinterpret_cast<uintptr_t>(g.gx) & 15u) == 0;  // K % 128 == 0
  if (pl.b_planes) {
    GyPlanes pp{};
    int n = 0;
    for (int t = 0; t < 4; ++t)
      if (pl.want >> t & 1)
        pp.p[t] = reinterpret_cast<unsigned short*>(bw + (int64_t)n++ * g.plane_b);
    const int64_t items = (int64_t)s->B * pl.ldb;
    if ((items + 255) / 256 > INT32_MAX) return FB_ERR_SHAPE;
    hipLaunchKernelGGL(grad_gy_kernel, dim3((unsigned)((items + 255) / 256)), dim3(256), 0, hs, gy,
                       (int64_t)s->B, s->N, pl.ldb, s->y_dtype, pp);
    if (hipGetLastError() != hipSuccess) return FB_ERR_HIP;
  }
  for (int sp0 = 0; sp0 < pl.GS; sp0 += pl.spans) {
    const int nsp = std::min(pl.spans, pl.GS - sp0);
    g.KT = nsp * 32;
    g.plane_a = (int64_t)g.KT * pl.QN * kTileBytes;
    g.k0 = sp0 * 512;
    const int kw = std::min(nsp * 512, s->K - g.k0);
    int st = launch_decode(pl, s, wdev, aw, sp0, nsp, g.plane_a, hs);
    if (st != FB_OK) return st;
    st = pl.xdt == FB_DT_F16 ? launch_grad_tile<FB_DT_F16>(g, pl, kw, hs)
                             : launch_grad_tile<FB_DT_BF16>(g, pl, kw, hs);
    if (st != FB_OK) return st;
  }
  if (pl.P > 1) {
    const int st = fb_gpu::sum_parts(part, pl.P, (int64_t)s->B * s->K, g.gx, g.dt, g.vec,
                                     nullptr, 0, s->K, hs);
    if (st != FB_OK) return st;
  }
  if (s->fwht_block) {
    const int pieces = (s->K + kRotPiece - 1) / kRotPiece;
    if ((int64_t)pieces * s->B > INT32_MAX) return FB_ERR_SHAPE;
    hipLaunchKernelGGL(grad_rotate_kernel, dim3((unsigned)(pieces * (int64_t)s->B)), dim3(256), 0,
                       hs, rot, gx, s->K, pieces, s->fwht_block,
                       1.0f / std::sqrt((float)s->fwht_block), gx_dtype);
    if (hipGetLastError() != hipSuccess) return FB_ERR_HIP;
  }
  return FB_OK;
}

}  // namespace

extern "C" {

size_t fb_grad_bias_workspace_bytes(int32_t M, int32_t N) {
  if (M < 1 || N < 1) return 0;
  size_t bytes = 0;
  for (int64_t rows = M; !bias_alone(rows, N);) {
    rows = bias_parts(rows, N).rows;
    bytes += align256((size_t)rows * N * 4);
  }
  return bytes;
}

int fb_grad_bias_ws(const void* gy, int32_t gy_dtype, int32_t M, int32_t N, void* gb,
                    int32_t gb_dtype, void* ws, size_t ws_bytes, void* stream) {
  if (!gy || !gb) return FB_ERR_NULL;
  if (M < 1 || N < 1) return FB_ERR_SHAPE;
  for (int32_t d : {gy_dtype, gb_dtype})
    if (d != FB_DT_F16 && d != FB_DT_BF16 && d != FB_DT_F32) return FB_ERR_DTYPE;
  if (reinterpret_cast<uintptr_t>(gy) & (gy_dtype == FB_DT_F32 ? 3u : 1u)) return FB_ERR_ALIGN;
  const size_t need = fb_grad_bias_workspace_bytes(M, N);
  if (need && !ws) return FB_ERR_NULL;
  if (need && (reinterpret_cast<uintptr_t>(ws) & 255u)) return FB_ERR_ALIGN;
  if (need > ws_bytes) return FB_ERR_WORKSPACE;
  uint8_t* at = static_cast<uint8_t*>(ws);
  int64_t rows = M;
  while (!bias_alone(rows, N)) {
    const BiasParts b = bias_parts(rows, N);
    const int st = launch_bias_parts(gy, gy_dtype, rows, N, b, reinterpret_cast<float*>(at),
                                     static_cast<hipStream_t>(stream));
    if (st != FB_OK) return st;
    gy = at;
    gy_dtype = FB_DT_F32;
    rows = b.rows;
    at += align256((size_t)rows * N * 4);
  }
  return fb_grad_bias(gy, gy_dtype, (int32_t)rows, N, gb, gb_dtype, stream);
}

int fb_grad_bias(const void* gy, int32_t gy_dtype, int32_t M, int32_t N, void* gb,
                 int32_t gb_dtype, void* stream) {
  if (!gy || !gb) return FB_ERR_NULL;
  if (M < 1 || N < 1) return FB_ERR_SHAPE;
  for (int32_t d : {gy_dtype, gb_dtype})
    if (d != FB_DT_F16 && d != FB_DT_BF16 && d != FB_DT_F32) return FB_ERR_DTYPE;
  if ((reinterpret_cast<uintptr_t>(gy) & (gy_dtype == FB_DT_F32 ? 3u : 1u)) ||
      (reinterpret_cast<uintptr_t>(gb) & (gb_dtype == FB_DT_F32 ? 3u : 1u)))
    return FB_ERR_ALIGN;
  hipLaunchKernelGGL(grad_bias_kernel, dim3((N + 15) / 16), dim3(1024), 0,
                     static_cast<hipStream_t>(stream), gy, M, N, gy_dtype, gb, gb_dtype);
  return hipGetLastError() == hipSuccess ? FB_OK : FB_ERR_HIP;
}

size_t fb_grad_x_workspace_bytes(const fb_shape_t* s, int32_t f16_exact) {
  GradPlan pl;
  // planned as for a gy that cannot be read in place: enough for either
  if (!s || grad_plan(s, reinterpret_cast<const void*>(1), f16_exact, pl) != FB_OK) return 0;
  return pl.total();
}

int fb_grad_x(const void* wdev, const void* gy, void* gx, const fb_shape_t* s, int32_t gx_dtype,
              int32_t f16_exact, void* ws, size_t ws_bytes, void* stream) {
  if (!s || !wdev || !gy || !gx || !ws) return FB_ERR_NULL;
  GradPlan pl;
  const int st = grad_plan(s, gy, f16_exact, pl);
  if (st != FB_OK) return st;
  if (gx_dtype != FB_DT_F16 && gx_dtype != FB_DT_BF16 && gx_dtype != FB_DT_F32)
    return FB_ERR_DTYPE;
  if ((reinterpret_cast<uintptr_t>(wdev) & 15u) || (reinterpret_cast<uintptr_t>(gy) & 1u) ||
      (s->y_dtype == FB_DT_F32 && (reinterpret_cast<uintptr_t>(gy) & 3u)) ||
      (reinterpret_cast<uintptr_t>(gx) & 3u) || (reinterpret_cast<uintptr_t>(ws) & 255u))
    return FB_ERR_ALIGN;
  if (pl.total() > ws_bytes) return FB_ERR_WORKSPACE;
  return grad_run(pl, s, wdev, gy, gx, gx_dtype, static_cast<uint8_t*>(ws),
                  static_cast<hipStream_t>(stream));
}

}  // extern "C"
