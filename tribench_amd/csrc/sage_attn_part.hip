// sage_attn_part.hip — attention split over the keys: the partial kernels and
// the merge of their results.
//
// One work-group per 128 query rows leaves most of the chip idle when there
// are few rows, and each work-group then sweeps all keys alone.  The partial
// kernels (attn_fwd_kernel with kPart) split the keys into ranges and, with
// grouped KV heads, put the query rows of a group's heads side by side in one
// work-group; each range's unnormalised O, running max and row sum go to a
// workspace in fp32, and attn_merge forms
//   O = sum_s 2^(m_s - M) O_s / sum_s 2^(m_s - M) l_s,  M = max_s m_s
// (times v_scale with FP8 V).  One range (packed heads alone) has weight 1 and
// the factors of the unsplit kernel's epilogue: its outputs bit for bit.
#include "sage_attn_kernel.h"

namespace sage {

template <int QKM, int D, int PVM, bool kVRow>
static int launch_part(const AttnArgs& a, hipStream_t st, const char* who) {
  const int64_t rows = (int64_t)a.grp * a.Nq;
  const int64_t grid = (rows + 127) / 128 * (a.Hq / a.grp) * a.B * a.nsplit;
  if (grid > 0x7FFFFFFF) return fail("%s: invalid argument: grid too large", who);
  hipLaunchKernelGGL((attn_fwd_kernel<QKM, D, PVM, float, 4, 2, kVRow, true>), dim3((unsigned)grid), dim3(256), 0, st, a);
  return check_launch(who);
}

// D/4 lanes to a row, 4 channels each.  The splits' maxima and sums are read
// side by side (lane i: splits i, i + D/4, ..) and the partial O in groups of 8
// splits, so that a row costs three load latencies at up to 8 splits instead
// of one per split (a serial loop: 0.5 us per split at 57 rows of 16 heads).
template <int D, typename TO>
__global__ __launch_bounds__(256) void attn_merge_kernel(AttnArgs a) {
  constexpr int TPR = D / 4;
  const int64_t nrow = (int64_t)a.B * a.Hq * a.Nq;
  const int64_t r0 = (int64_t)blockIdx.x * (256 / TPR) + threadIdx.x / TPR;
  const int t = threadIdx.x % TPR, c = 4 * t;
  const int64_t row = min(r0, nrow - 1);  // (every lane takes part in the shuffles)
  float m = -INFINITY, l = 0.0f;
  for (int s0 = 0; s0 < a.nsplit; s0 += TPR)
    if (s0 + t < a.nsplit) m = fmaxf(m, a.part_ml[(s0 + t) * nrow + row].x);
#pragma unroll
  for (int o = TPR / 2; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
  if (m == -INFINITY) m = 0.0f;  // every score -inf: sums of 0, as in one sweep
  v4f o = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int s0 = 0; s0 < a.nsplit; s0 += 8) {
    v4f po[8];
    float2 ml[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int s = min(s0 + i, a.nsplit - 1);
      ml[i] = a.part_ml[s * nrow + row];
      po[i] = *reinterpret_cast<const v4f*>(a.part_o + (s * nrow + row) * D + c);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (s0 + i < a.nsplit) {
        const float w = __builtin_amdgcn_exp2f(ml[i].x - m);
        l += w * ml[i].y;
        o += w * po[i];
      }
  }
  if (r0 >= nrow) return;
  const float inv = 1.0f / l;
  const int64_t q = row % a.Nq, bh = row / a.Nq;
  v4f f = {inv, inv, inv, inv};
  if (a.v_scale) {  // FP8 V
    const int64_t hk = bh / a.Hq * a.Hkv + bh % a.Hq / (a.Hq / a.Hkv);
    f = inv * *reinterpret_cast<const v4f*>(a.v_scale + hk * D + c);
  }
  TO* p = static_cast<TO*>(a.o) + bh / a.Hq * a.so[0] + bh % a.Hq * a.so[1] + q * a.son + c;
  store4<TO>(p, o[0] * f[0], o[1] * f[1], o[2] * f[2], o[3] * f[3]);
}

template <int D, typename TO>
static int launch_merge(const AttnArgs& a, hipStream_t st, const char* who) {
  constexpr int RPB = 256 / (D / 4);
  const int64_t nrow = (int64_t)a.B * a.Hq * a.Nq;
  hipLaunchKernelGGL((attn_merge_kernel<D, TO>), dim3((unsigned)((nrow + RPB - 1) / RPB)), dim3(256), 0, st, a);
  return check_launch(who);
}

template <int D>
static int launch_part_d(const AttnArgs& a, int pv_mode, bool i8, int o_dtype, hipStream_t st, const char* who) {
  int rc;
  if (i8) {
    if (a.vrow)
      rc = pv_mode == SAGE_PV_F16 ? launch_part<kQkI8, D, SAGE_PV_F16, true>(a, st, who)
                                  : launch_part<kQkI8, D, SAGE_PV_BF16, true>(a, st, who);
    else if (pv_mode == SAGE_PV_F16) rc = launch_part<kQkI8, D, SAGE_PV_F16, false>(a, st, who);
    else if (pv_mode == SAGE_PV_BF16) rc = launch_part<kQkI8, D, SAGE_PV_BF16, false>(a, st, who);
    else rc = launch_part<kQkI8, D, SAGE_PV_FP8, false>(a, st, who);
  } else if (o_dtype == SAGE_DTYPE_F16) {
    rc = launch_part<kQkF16, D, SAGE_PV_F16, true>(a, st, who);
  } else {
    rc = launch_part<kQkBF16, D, SAGE_PV_BF16, true>(a, st, who);
  }
  if (rc) return rc;
  switch (o_dtype) {
    case SAGE_DTYPE_F32: return launch_merge<D, float>(a, st, who);
    case SAGE_DTYPE_F16: return launch_merge<D, _Float16>(a, st, who);
    default: return launch_merge<D, __bf16>(a, st, who);
  }
}

int launch_attn_part(const AttnArgs& a, int D, int pv_mode, bool i8, int o_dtype, hipStream_t st, const char* who) {
  return D == 64 ? launch_part_d<64>(a, pv_mode, i8, o_dtype, st, who)
                 : launch_part_d<128>(a, pv_mode, i8, o_dtype, st, who);
}

}  // namespace sage
