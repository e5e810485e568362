"""Device prelude shared by every generated HIP program (gfx950, wave64).

No headers are included: hipRTC supplies the HIP device builtins and the
math library (erff, expf, ...).  Storage types are ``float``, ``_Float16``,
``int`` and ``unsigned short`` (bf16 bits); all arithmetic is fp32.  Vector
helpers move 16 bytes per lane (``global_load_dwordx4``) and unpack to fp32;
bf16 stores round to nearest even, as torch does (gfx950's packed
``v_cvt_pk_bf16_f32``).
"""
from __future__ import annotations

from ..ir import DType

CTYPE = {DType.f32: "float", DType.f16: "_Float16", DType.bf16: "unsigned short", DType.i32: "int"}

PRELUDE = r"""// generated by tensorjit (hip backend, gfx950)
typedef unsigned int tj_u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int tj_u32x2 __attribute__((ext_vector_type(2)));
typedef float tj_f32x4 __attribute__((ext_vector_type(4)));
typedef float tj_f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 tj_f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 tj_bf16x8 __attribute__((ext_vector_type(8)));
typedef short tj_i16x8 __attribute__((ext_vector_type(8)));
typedef short tj_i16x4 __attribute__((ext_vector_type(4)));

typedef float tj_f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 tj_bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 tj_f16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float tj_bf2f(unsigned int bits16) { return __builtin_bit_cast(float, bits16 << 16); }
// fp32 -> bf16 with round to nearest even: gfx950's v_cvt_pk_bf16_f32 (two values per instruction)
__device__ __forceinline__ unsigned int tj_f2bf(float f) { return __builtin_bit_cast(unsigned short, (__bf16)f); }
__device__ __forceinline__ unsigned int tj_f2bf2(float lo, float hi) {
  tj_f32x2 v; v[0] = lo; v[1] = hi;
  return __builtin_bit_cast(unsigned int, __builtin_convertvector(v, tj_bf16x2));
}
__device__ __forceinline__ float tj_ld(float v) { return v; }
__device__ __forceinline__ float tj_ld(_Float16 v) { return (float)v; }
__device__ __forceinline__ float tj_ld(int v) { return (float)v; }
__device__ __forceinline__ float tj_ld(unsigned short v) { return tj_bf2f(v); }
__device__ __forceinline__ void tj_st(float* p, float v) { *p = v; }
__device__ __forceinline__ void tj_st(_Float16* p, float v) { *p = (_Float16)v; }
__device__ __forceinline__ void tj_st(int* p, float v) { *p = (int)v; }
__device__ __forceinline__ void tj_st(unsigned short* p, float v) { *p = (unsigned short)tj_f2bf(v); }

// 16-byte vector loads/stores unpacked to / packed from fp32.  Stores carry the
// nontemporal hint (global_store_dwordx4 ... nt): outputs are written once and
// not re-read by the kernel, and the hint measured 2-20% faster on the
// bandwidth-bound families (a plain copy: 6.0 -> 7.4 TB/s).
__device__ __forceinline__ void tj_st16(void* p, tj_u32x4 x) { __builtin_nontemporal_store(x, (tj_u32x4*)p); }
// tj_unpackv: 16 loaded bytes of the element type named by the (unused) pointer -> fp32
__device__ __forceinline__ void tj_unpackv(tj_u32x4 x, const float*, float* v) {
  // bit-cast the whole vector: hipcc bit-casts an element subscript of an ext-vector
  // as element 0
  const tj_f32x4 f = __builtin_bit_cast(tj_f32x4, x);
  v[0] = f[0]; v[1] = f[1]; v[2] = f[2]; v[3] = f[3];
}
__device__ __forceinline__ void tj_unpackv(tj_u32x4 x, const int*, float* v) {
  for (int i = 0; i < 4; ++i) v[i] = (float)(int)x[i];
}
__device__ __forceinline__ void tj_unpackv(tj_u32x4 x, const unsigned short*, float* v) {
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = __builtin_bit_cast(float, x[i] << 16);
    v[2 * i + 1] = __builtin_bit_cast(float, x[i] & 0xffff0000u);
  }
}
__device__ __forceinline__ float tj_h2f(unsigned int bits16) {
  return (float)__builtin_bit_cast(_Float16, (unsigned short)bits16);
}
__device__ __forceinline__ unsigned int tj_f2h(float f) {
  return __builtin_bit_cast(unsigned short, (_Float16)f);
}
// two at once, the same rounding: gfx950's v_cvt_pk_f16_f32, one instruction where two
// conversions and a shift-or took three (us, fp16 attention [4, 32, 2000, 64] 180.4 -> 173.2,
// [4, 32, 2000, 128] 259.5 -> 252.9, softmax [200000, 64] 9.7 -> 9.4)
__device__ __forceinline__ unsigned int tj_f2h2(float lo, float hi) {
  tj_f32x2 v; v[0] = lo; v[1] = hi;
  return __builtin_bit_cast(unsigned int, __builtin_convertvector(v, tj_f16x2));
}
__device__ __forceinline__ void tj_unpackv(tj_u32x4 x, const _Float16*, float* v) {
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = tj_h2f(x[i] & 0xffffu);
    v[2 * i + 1] = tj_h2f(x[i] >> 16);
  }
}
template <typename T> __device__ __forceinline__ void tj_ldv(const T* p, float* v) {
  tj_unpackv(*(const tj_u32x4*)p, p, v);
}
template <typename T> __device__ __forceinline__ void tj_ldv_nt(const T* p, float* v) {
  tj_unpackv(__builtin_nontemporal_load((const tj_u32x4*)p), p, v);
}
__device__ __forceinline__ tj_u32x4 tj_packv(const float*, const float* v) {
  tj_f32x4 x; x[0] = v[0]; x[1] = v[1]; x[2] = v[2]; x[3] = v[3];
  return __builtin_bit_cast(tj_u32x4, x);
}
__device__ __forceinline__ tj_u32x4 tj_packv(const int*, const float* v) {
  tj_u32x4 x;
  for (int i = 0; i < 4; ++i) x[i] = (unsigned int)(int)v[i];
  return x;
}
__device__ __forceinline__ tj_u32x4 tj_packv(const unsigned short*, const float* v) {
  tj_u32x4 x;
  for (int i = 0; i < 4; ++i) x[i] = tj_f2bf2(v[2 * i], v[2 * i + 1]);
  return x;
}
__device__ __forceinline__ tj_u32x4 tj_packv(const _Float16*, const float* v) {
  tj_u32x4 x;
  for (int i = 0; i < 4; ++i) x[i] = tj_f2h2(v[2 * i], v[2 * i + 1]);
  return x;
}
template <typename T> __device__ __forceinline__ void tj_stv(T* p, const float* v) { tj_st16(p, tj_packv(p, v)); }
// The same 16 bytes at any element's address (rows of an odd length): the global memory
// instructions take unaligned addresses, and a wave's accesses stay contiguous.
typedef tj_u32x4 tj_u32x4a2 __attribute__((aligned(2)));
template <typename T> __device__ __forceinline__ void tj_ldv_u(const T* p, float* v) {
  tj_unpackv(*(const tj_u32x4a2*)p, p, v);
}
template <typename T> __device__ __forceinline__ void tj_ldv_u_nt(const T* p, float* v) {
  tj_unpackv(__builtin_nontemporal_load((const tj_u32x4a2*)p), p, v);
}
template <typename T> __device__ __forceinline__ void tj_stv_u(T* p, const float* v) {
  __builtin_nontemporal_store(tj_packv(p, v), (tj_u32x4a2*)p);
}

// Fast fp32 math on the native transcendental units.  exp(x) = 2^(x*log2 e) on
// v_exp_f32 and 1/x on v_rcp_f32 (each ~1 ulp); erf is Abramowitz & Stegun 7.1.26
// (|error| <= 1.5e-7, the same published formula the CPU c backend uses), with |x|
// clamped at 4 where erf is +-1 to fp32 precision.
__device__ __forceinline__ float tj_exp(float x) { return __builtin_amdgcn_exp2f(x * 1.4426950408889634f); }
__device__ __forceinline__ float tj_rcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float tj_erf(float x) {
  const float z = fminf(fabsf(x), 4.0f);
  const float t = tj_rcp(1.0f + 0.3275911f * z);
  const float p = t * (0.254829592f + t * (-0.284496736f + t * (1.421413741f + t * (-1.453152027f + t * 1.061405429f))));
  return __builtin_copysignf(1.0f - p * tj_exp(-z * z), x);
}
__device__ __forceinline__ float tj_gelu(float x) { return 0.5f * x * (1.0f + tj_erf(x * 0.70710678118654752f)); }
// gelu for GEMM epilogues whose outputs are all bf16 / fp16, where this VALU work is not
// hidden under the MFMAs: erf by Abramowitz & Stegun 7.1.25 (three terms, |error| <=
// 2.5e-5, so |error| <= 1.3e-5 |x| in gelu), written as 0.5 (x + |x|) - a q with
// a = min(|x|, 4 sqrt 2) and q = P(t) e^(-a^2/2) / 2 -- the algebra of
// 0.5 x (1 + erf(x / sqrt 2)) with fewer instructions.  NaN and -inf give NaN and +inf
// gives +inf, as in tj_gelu.
__device__ __forceinline__ float tj_gelu16(float x) {
  const float a = fminf(fabsf(x), 5.656854249f);
  const float t = tj_rcp(__builtin_fmaf(0.47047f * 0.70710678118654752f, a, 1.0f));
  const float p = t * (0.5f * 0.3480242f + t * (0.5f * -0.0958798f + t * (0.5f * 0.7478556f)));
  const float e = __builtin_amdgcn_exp2f(a * a * (-0.5f * 1.4426950408889634f));
  return __builtin_fmaf(0.5f, x + fabsf(x), -a * (p * e));
}
__device__ __forceinline__ float tj_sigmoid(float x) { return tj_rcp(1.0f + tj_exp(-x)); }

// wave64 all-reductions on DPP lane moves inside each 16-lane row (quad xor 1, quad xor 2,
// half-row mirror, row mirror: every lane ends with its row's total), then the four row
// totals read from lanes 0/16/32/48 and combined in one fixed order, so every lane holds
// the same bits.  No LDS traffic (a __shfl_xor butterfly is one ds_bpermute per step);
// measured 1-10% faster on the row family.  Every lane of the wave must be active.
#define TJ_DPP(v, ctrl) \
  __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ctrl, 0xf, 0xf, false))
__device__ __forceinline__ float tj_lane(float v, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}
__device__ __forceinline__ float tj_wave_sum(float v) {
  v += TJ_DPP(v, 0xb1);    // quad_perm [1,0,3,2]
  v += TJ_DPP(v, 0x4e);    // quad_perm [2,3,0,1]
  v += TJ_DPP(v, 0x141);   // row_half_mirror
  v += TJ_DPP(v, 0x140);   // row_mirror
  return (tj_lane(v, 0) + tj_lane(v, 16)) + (tj_lane(v, 32) + tj_lane(v, 48));
}
__device__ __forceinline__ float tj_wave_max(float v) {
  v = fmaxf(v, TJ_DPP(v, 0xb1));
  v = fmaxf(v, TJ_DPP(v, 0x4e));
  v = fmaxf(v, TJ_DPP(v, 0x141));
  v = fmaxf(v, TJ_DPP(v, 0x140));
  return fmaxf(fmaxf(tj_lane(v, 0), tj_lane(v, 16)), fmaxf(tj_lane(v, 32), tj_lane(v, 48)));
}

// the same inside groups of L lanes (2-32, aligned; a group's lanes are all active): several
// short rows per wave.  32 lanes: the two 16-lane rows' totals are exchanged by
// v_permlane16_swap.
template <int L> __device__ __forceinline__ float tj_group_sum(float v) {
  if (L >= 2) v += TJ_DPP(v, 0xb1);
  if (L >= 4) v += TJ_DPP(v, 0x4e);
  if (L >= 8) v += TJ_DPP(v, 0x141);
  if (L >= 16) v += TJ_DPP(v, 0x140);
  if (L >= 32) {
    const unsigned int u = __builtin_bit_cast(unsigned int, v);
    const auto s = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    v = __builtin_bit_cast(float, (unsigned int)s[0]) + __builtin_bit_cast(float, (unsigned int)s[1]);
  }
  return v;
}
template <int L> __device__ __forceinline__ float tj_group_max(float v) {
  if (L >= 2) v = fmaxf(v, TJ_DPP(v, 0xb1));
  if (L >= 4) v = fmaxf(v, TJ_DPP(v, 0x4e));
  if (L >= 8) v = fmaxf(v, TJ_DPP(v, 0x141));
  if (L >= 16) v = fmaxf(v, TJ_DPP(v, 0x140));
  if (L >= 32) {
    const unsigned int u = __builtin_bit_cast(unsigned int, v);
    const auto s = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    v = fmaxf(__builtin_bit_cast(float, (unsigned int)s[0]), __builtin_bit_cast(float, (unsigned int)s[1]));
  }
  return v;
}

// lane l and lane l ^ 32 combined: gfx950's v_permlane32_swap exchanges the two halves
// of the wave in one VALU instruction (the attention kernel's query halves)
__device__ __forceinline__ float tj_pair_max(float x) {
  const unsigned int u = __builtin_bit_cast(unsigned int, x);
  const auto sw = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return fmaxf(__builtin_bit_cast(float, (unsigned int)sw[0]), __builtin_bit_cast(float, (unsigned int)sw[1]));
}
__device__ __forceinline__ float tj_pair_sum(float x) {
  const unsigned int u = __builtin_bit_cast(unsigned int, x);
  const auto sw = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __builtin_bit_cast(float, (unsigned int)sw[0]) + __builtin_bit_cast(float, (unsigned int)sw[1]);
}
"""


def vec_width(dtype: DType) -> int:
    """Elements per 16-byte vector access."""
    return 16 // dtype.itemsize
