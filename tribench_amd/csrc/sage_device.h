// sage_device.h — small gfx950 device helpers shared by the pre-pass and the
// attention kernel: element types, 16-byte loads, conversions, wave
// reductions, error reporting of the C ABI.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define SAGE_HD __host__ __device__
#include "sage_quant_math.h"
#include "../../include/sage_attn.h"

namespace sage {

typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));

// ---------------------------------------------------------------------------
// element types
// ---------------------------------------------------------------------------
template <typename T>
struct Elt;
template <>
struct Elt<float> {
  static constexpr int kBytes = 4;
  static constexpr int kCode = SAGE_DTYPE_F32;
};
template <>
struct Elt<_Float16> {
  static constexpr int kBytes = 2;
  static constexpr int kCode = SAGE_DTYPE_F16;
};
template <>
struct Elt<__bf16> {
  static constexpr int kBytes = 2;
  static constexpr int kCode = SAGE_DTYPE_BF16;
};

// 8 consecutive elements of T held raw: 16 B for 2-byte types, 32 B for fp32.
template <typename T>
struct Raw8 {
  static constexpr int kU4 = Elt<T>::kBytes * 8 / 16;
  uint4 u[kU4];
};

template <typename T>
__device__ __forceinline__ Raw8<T> load8(const T* p) {
  Raw8<T> r;
  const uint4* s = reinterpret_cast<const uint4*>(p);
#pragma unroll
  for (int i = 0; i < Raw8<T>::kU4; ++i) r.u[i] = s[i];
  return r;
}

template <typename T>
__device__ __forceinline__ Raw8<T> zero8() {
  Raw8<T> r;
#pragma unroll
  for (int i = 0; i < Raw8<T>::kU4; ++i) r.u[i] = make_uint4(0, 0, 0, 0);
  return r;
}

__device__ __forceinline__ uint32_t word(const uint4& u, int i) {
  return i == 0 ? u.x : (i == 1 ? u.y : (i == 2 ? u.z : u.w));
}

// element e (0..7) of a raw 8-pack as fp32 (exact for every input type)
template <typename T>
__device__ __forceinline__ float elem(const Raw8<T>& r, int e);
template <>
__device__ __forceinline__ float elem<float>(const Raw8<float>& r, int e) {
  return __uint_as_float(word(r.u[e >> 2], e & 3));
}
template <>
__device__ __forceinline__ float elem<__bf16>(const Raw8<__bf16>& r, int e) {
  uint32_t w = word(r.u[0], e >> 1);
  return __uint_as_float((e & 1) ? (w & 0xFFFF0000u) : (w << 16));
}
template <>
__device__ __forceinline__ float elem<_Float16>(const Raw8<_Float16>& r, int e) {
  uint32_t w = word(r.u[0], e >> 1);
  uint16_t hb = (uint16_t)((e & 1) ? (w >> 16) : (w & 0xFFFFu));
  _Float16 h = __builtin_bit_cast(_Float16, hb);
  return (float)h;
}

// ---------------------------------------------------------------------------
// wave64 reductions (xor butterflies over all 64 lanes)
// ---------------------------------------------------------------------------
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
  return v;
}

// ---------------------------------------------------------------------------
// max of a non-negative value over the wave: DPP steps inside each 16-lane row
// (quad xor 1, quad xor 2, half-row mirror, row mirror), then the four row
// results via readlane.  Result is wave-uniform.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xF, 0xF, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xF, 0xF, false));
  const uint32_t r0 = __builtin_amdgcn_readlane(v, 0), r1 = __builtin_amdgcn_readlane(v, 16);
  const uint32_t r2 = __builtin_amdgcn_readlane(v, 32), r3 = __builtin_amdgcn_readlane(v, 48);
  return max(max(r0, r1), max(r2, r3));
}

// max of a non-negative value over each group of W consecutive lanes (W = 4
// or 8: quad xor 1, quad xor 2, then the half-row mirror for 8); every lane
// of a group gets the group's max
template <int W>
__device__ __forceinline__ uint32_t group_max_u32(uint32_t v) {
  static_assert(W == 4 || W == 8, "group of 4 or 8 lanes");
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, false));
  if constexpr (W == 8) v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xF, 0xF, false));
  return v;
}

}  // namespace sage

// ---------------------------------------------------------------------------
// C-ABI error plumbing (defined in sage_abi.hip)
// ---------------------------------------------------------------------------
namespace sage {
int fail(const char* fmt, ...);
int check_launch(const char* what);

// Whether launch B of the pre-pass quantizes 16-bit K one block to a wave
// instead of one to a work-group; nblk: K blocks of the call, vt_in_b: V tiles
// (of pv_mode's type) in the launch.  Pre-pass in us, work-group role -> wave role, bf16.
// It takes 4 blocks to a CU to pay beside V tiles (512 blocks with fp16 tiles, D =
// 128: 14.4 -> 15.2), 8 without, where it depends on the shape below (1024 blocks of
// 4096 keys 16.6 -> 15.3, 1136 of short ones at D = 64 14.7 -> 15.5).  D = 64, from
// there on 4 to 22 % less: 1024 blocks 15.0 -> 12.5, 16384 127 -> 114, with FP8 tiles
// 215 -> 185.  D = 128, whose wave role takes 106 VGPRs and leaves the launch's other
// roles 4 waves to a SIMD of 7: 1024 blocks 20.2 -> 17.9, 2048 without tiles 24.0 -> 20.3,
// 4448 71.0 -> 68.0, but 8192 118 -> 118 (Q blocks beside 157 -> 160), 16384 229 ->
// 231 (Q 300 -> 311); and FP8 tiles, bound by the VALU, lose at every size: 1024
// 25.4 -> 26.7, 8192 164 -> 177, 16384 285 -> 317.
inline bool k_waves_pay(int64_t nblk, int64_t D, bool vt_in_b, int pv_mode) {
  if (D == 128 && (nblk >= 8192 || (vt_in_b && pv_mode == SAGE_PV_FP8))) return false;
  return nblk >= (vt_in_b ? 1024 : 2048);
}

// sage_prepass (vt NULL) or sage_prepass_vt, reporting errors as `who`
int prepass_any(const char* who, const void* q, const void* k, const void* v, int in_dtype, int64_t B, int64_t Hq,
                int64_t Hkv, int64_t Nq, int64_t Nkv, int64_t D, const int64_t* q_strides, const int64_t* k_strides,
                const int64_t* v_strides, float q_mul, int blkq, int blkk, int q_sub, int smooth_k, int v_mode,
                int8_t* q8, const int64_t* q8_strides, float* q_scale, int8_t* k8, const int64_t* k8_strides,
                float* k_scale, float* km, uint8_t* v8, const int64_t* v8_strides, float* v_scale, void* workspace,
                size_t workspace_bytes, int pv_mode, void* vt, size_t vt_bytes, void* stream);
}  // namespace sage
