// Device-side types and the in-register 4-bit decoders shared by the GEMV, the GEMM and the
// device decoder.  Everything here is inlined into the kernels that use it.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "fourbit.h"

namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf168_t __attribute__((ext_vector_type(8)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------------
// small device helpers
// ---------------------------------------------------------------------------------
__device__ __forceinline__ unsigned perm(unsigned s0, unsigned s1, unsigned sel) {
  return __builtin_amdgcn_perm(s0, s1, sel);
}

__device__ __forceinline__ u32x4 ldg16(const uint8_t* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
}

__device__ __forceinline__ void store_y(void* y, int64_t idx, float v, int ydt) {
  if (ydt == FB_DT_F32) {
    static_cast<float*>(y)[idx] = v;
  } else if (ydt == FB_DT_F16) {
    static_cast<_Float16*>(y)[idx] = (_Float16)v;
  } else {
    static_cast<__bf16*>(y)[idx] = (__bf16)v;
  }
}

__device__ __forceinline__ float load_as_float(const void* p, int64_t idx, int dt) {
  return dt == FB_DT_F32   ? static_cast<const float*>(p)[idx]
         : dt == FB_DT_F16 ? (float)static_cast<const _Float16*>(p)[idx]
                           : (float)static_cast<const __bf16*>(p)[idx];
}

// Four outputs at idx, which 16-byte alignment of y and idx % 4 == 0 make one store.
__device__ __forceinline__ void store4(void* y, int64_t idx, const f32x4& v, int ydt) {
  if (ydt == FB_DT_F32) {
    *reinterpret_cast<f32x4*>(static_cast<float*>(y) + idx) = v;
  } else {
    unsigned h[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      h[e] = ydt == FB_DT_F16 ? __builtin_bit_cast(unsigned short, (_Float16)v[e])
                              : __builtin_bit_cast(unsigned short, (__bf16)v[e]);
    *reinterpret_cast<uint2*>(static_cast<uint16_t*>(y) + idx) =
        make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
  }
}

typedef __attribute__((address_space(3))) uint8_t lds_byte;

// Workgroup barrier once this wave has at most N vector memory operations in flight (of which
// loads into LDS are some) and has received every LDS read.
template <int N>
__device__ __forceinline__ void wait_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// Ends a group of requests: the compiler issues no memory operation of one side on the other.
// wait_barrier's counts are of whole groups (a chunk's x pieces and weights); inside a pipeline
// its barriers part them, before the first one this does.
__device__ __forceinline__ void request_group_end() { asm volatile("" ::: "memory"); }

// GF4 decode of one 32-bit word (8 codes, layout order) into 4 fp16 pairs in element
// order (e0,e1) (e2,e3) (e4,e5) (e6,e7).  tl/th: lo/hi byte-plane tables
// {A'[0..3], A'[4..7], B'[0..3], B'[4..7]}.
__device__ __forceinline__ u32x4 gf4_decode8(unsigned q, const u32x4& tl, const u32x4& th) {
  const unsigned sa = q & 0x0F0F0F0Fu;
  const unsigned sb = (q >> 4) & 0x0F0F0F0Fu;
  const unsigned sa8 = sa ^ 0x08080808u;
  const unsigned sb8 = sb ^ 0x08080808u;
  const unsigned loA = perm(tl.y, tl.x, sa) ^ perm(tl.w, tl.z, sa8);
  const unsigned hiA = perm(th.y, th.x, sa) ^ perm(th.w, th.z, sa8);
  const unsigned loB = perm(tl.y, tl.x, sb) ^ perm(tl.w, tl.z, sb8);
  const unsigned hiB = perm(th.y, th.x, sb) ^ perm(th.w, th.z, sb8);
  u32x4 w;
  w.x = perm(hiA, loA, 0x05010400u);
  w.y = perm(hiA, loA, 0x07030602u);
  w.z = perm(hiB, loB, 0x05010400u);
  w.w = perm(hiB, loB, 0x07030602u);
  return w;
}

// Two independent 8-code decodes written stage by stage, so the scheduler sees twice the
// instruction-level parallelism of one decode chain.
__device__ __forceinline__ void gf4_decode16(unsigned q0, unsigned q1, const u32x4& tl,
                                             const u32x4& th, u32x4& w0, u32x4& w1) {
  const unsigned sa0 = q0 & 0x0F0F0F0Fu, sa1 = q1 & 0x0F0F0F0Fu;
  const unsigned t0 = q0 >> 4, t1 = q1 >> 4;
  const unsigned sa80 = sa0 ^ 0x08080808u, sa81 = sa1 ^ 0x08080808u;
  const unsigned sb0 = t0 & 0x0F0F0F0Fu, sb1 = t1 & 0x0F0F0F0Fu;
  const unsigned sb80 = sb0 ^ 0x08080808u, sb81 = sb1 ^ 0x08080808u;
  const unsigned la0 = perm(tl.y, tl.x, sa0), la1 = perm(tl.y, tl.x, sa1);
  const unsigned lb0 = perm(tl.w, tl.z, sa80), lb1 = perm(tl.w, tl.z, sa81);
  const unsigned ha0 = perm(th.y, th.x, sa0), ha1 = perm(th.y, th.x, sa1);
  const unsigned hb0 = perm(th.w, th.z, sa80), hb1 = perm(th.w, th.z, sa81);
  const unsigned loA0 = la0 ^ lb0, loA1 = la1 ^ lb1, hiA0 = ha0 ^ hb0, hiA1 = ha1 ^ hb1;
  const unsigned lc0 = perm(tl.y, tl.x, sb0), lc1 = perm(tl.y, tl.x, sb1);
  const unsigned ld0 = perm(tl.w, tl.z, sb80), ld1 = perm(tl.w, tl.z, sb81);
  const unsigned hc0 = perm(th.y, th.x, sb0), hc1 = perm(th.y, th.x, sb1);
  const unsigned hd0 = perm(th.w, th.z, sb80), hd1 = perm(th.w, th.z, sb81);
  w0.x = perm(hiA0, loA0, 0x05010400u); w1.x = perm(hiA1, loA1, 0x05010400u);
  w0.y = perm(hiA0, loA0, 0x07030602u); w1.y = perm(hiA1, loA1, 0x07030602u);
  const unsigned loB0 = lc0 ^ ld0, loB1 = lc1 ^ ld1, hiB0 = hc0 ^ hd0, hiB1 = hc1 ^ hd1;
  w0.z = perm(hiB0, loB0, 0x05010400u); w1.z = perm(hiB1, loB1, 0x05010400u);
  w0.w = perm(hiB0, loB0, 0x07030602u); w1.w = perm(hiB1, loB1, 0x07030602u);
}

// E2M1 decode of one 32-bit word (8 codes, canonical order) times `scale`.
template <int XDT>
__device__ __forceinline__ u32x4 e2m1_decode8(unsigned q, float scale) {
  u32x4 w;
  if constexpr (XDT == FB_DT_BF16) {
    w.x = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(q, scale, 0));
    w.y = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(q, scale, 1));
    w.z = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(q, scale, 2));
    w.w = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(q, scale, 3));
  } else {
    w.x = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(q, scale, 0));
    w.y = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(q, scale, 1));
    w.z = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(q, scale, 2));
    w.w = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(q, scale, 3));
  }
  return w;
}

template <int XDT>
__device__ __forceinline__ f32x4 mfma(const u32x4& a, const u32x4& b, const f32x4& c) {
  if constexpr (XDT == FB_DT_BF16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf168_t, a),
                                                   __builtin_bit_cast(bf168_t, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, a),
                                                  __builtin_bit_cast(half8_t, b), c, 0, 0, 0);
  }
}

// One lane's record of a work unit.
template <int FMT>
struct Rec {
  u32x4 nib[4];
  u32x4 t0, t1;  // GF4: lo / hi tables.  E2M1: t0.x holds the 4 scale bytes.
};

typedef __amdgpu_buffer_rsrc_t rsrc_t;
constexpr int kRsrcWord3 = 0x00020000;  // raw (untyped) buffer, gfx9 family
constexpr int kNT = 2;                  // streaming (non-temporal) cache policy
// a buffer offset past every resource's range: the load returns zeros and moves no data
constexpr unsigned kXOutOfRange = 0x7FFFFFF0u;

// Record read for the device decoder (plain global loads).
template <int FMT>
__device__ __forceinline__ void load_rec_global(const uint8_t* __restrict__ blk, int lane,
                                                Rec<FMT>& r) {
  const uint8_t* base = blk + lane * 16;
#pragma unroll
  for (int c = 0; c < 4; ++c) r.nib[c] = ldg16(base + c * 1024);
  if constexpr (FMT == FB_FMT_GF4) {
    r.t0 = ldg16(base + 4096);
    r.t1 = ldg16(base + 5120);
  } else {
    r.t0.x = __builtin_nontemporal_load(reinterpret_cast<const unsigned*>(blk + 4096 + lane * 4));
  }
}

}  // namespace
