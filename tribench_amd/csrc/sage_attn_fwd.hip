// sage_attn_fwd.hip — C ABI of the attention kernels (sage_attn_kernel.h):
// argument checks and the choice of the launch.
#include "sage_attn_kernel.h"
#include "../../include/sage_attn_run.h"

#include <cmath>

namespace sage {

#if SAGE_TRACE
unsigned long long* g_trace = nullptr;
int64_t g_trace_words = 0;
#endif

// ---------------------------------------------------------------------------
// The launch of one attention: waves per work-group, query heads packed into
// a work-group's rows, key ranges.
// ---------------------------------------------------------------------------
struct AttnPlan {
  int nw = 8, wpe = 2, grp = 1, nsplit = 1;
  bool part() const { return grp > 1 || nsplit > 1; }
};

// Chosen by a model of each launch's cost: work-groups fill 256 slots (8 waves)
// or 512 (4 waves, two to a CU) in rounds, a round costs its start (Q, first
// tiles, epilogue) plus a cost per 64-key block; the partial kernels add the
// merge and its traffic.  The unit is arbitrary: an attention takes 1.7 to 2.8
// us for each, by type and shape, so the sums rank the launches of one call and
// predict no times.  The constants were fitted to timed calls of both packs.
// Over 110 other random calls, 811 launches timed (1 to 25000 rows and keys),
// the pick is 1.4 % slower than the call's best launch on average and within
// 5 % for 102 of them, 26 % at worst (unquantized causal, B2 H8 N2517 D64: 8
// waves 43 us, 4 waves 34); 8 waves without a split are 50 % slower on average.
// What the constants stand for: 8 waves share every tile, which is worth 3 % of
// an attention on a full chip at INT8 D = 128 (B4 H32 N4096: 931 us a call
// against 958); 4 waves overlap one work-group's start with another's blocks
// and cut the rows finer (B2 H32 N2048 causal: 136 us against 149; 226 keys:
// 291 against 332); splits and packed heads fill the chip when rows are few (one
// row, 4 heads to a KV head, 8192 keys: 52 us against 146).
static AttnPlan attn_plan(int64_t B, int64_t Hq, int64_t Hkv, int64_t Nq, int64_t Nkv, int64_t D, bool causal,
                          bool i8, int pv_mode, int dtype, bool may_split) {
  const double start8 = 5.2, start4 = 3.7, split_cost = 4.2, merge_bytes_per_unit = 7.4e6;
  double blk8 = i8 ? 0.50 : 0.48, blk4 = i8 ? 0.505 : 0.525;  // D = 64
  if (D == 128) {
    blk8 = !i8 ? 0.98 : pv_mode == SAGE_PV_F16 ? 0.64 : pv_mode == SAGE_PV_BF16 ? 0.90 : 0.565;
    blk4 = !i8 ? 1.02 : pv_mode == SAGE_PV_FP8 ? 0.58 : 0.73;
  }
  const int64_t nt = (Nkv + 63) / 64, G = Hq / Hkv;
  // blocks of a work-group: all of them, or with causal rows over several rounds the mean
  auto sweep = [&](int64_t wgs, int64_t slots, double start, double blk, int64_t nsplit) {
    const double blocks = causal && wgs > slots ? 0.5 * (double)(nt + 2) : (double)nt;
    // (over many rounds the work-groups' ends spread and the last round fills)
    const double full = (double)wgs / (double)slots;
    return (full < 3.0 ? ceil(full) : full) * (start + ceil(blocks / (double)nsplit) * blk);
  };
  AttnPlan best;
  double t = sweep((Nq + 255) / 256 * Hq * B, 256, start8, blk8, 1);
  auto consider = [&](int grp, int nsplit) {
    const bool part = grp > 1 || nsplit > 1;
    const int64_t wgs = (grp * Nq + 127) / 128 * (Hq / grp) * B * nsplit;
    // (a work-group that has its CU to itself takes 0.8 of a block's time)
    double c = sweep(wgs, 512, start4, wgs <= 256 ? 0.8 * blk4 : blk4, nsplit);
    if (part) c += split_cost + (double)(B * Hq * Nq * nsplit * D * 8) / merge_bytes_per_unit;
    if (c < t) {
      t = c;
      best.nw = 4;
      best.wpe = 2;
      best.grp = grp;
      best.nsplit = nsplit;
    }
  };
  consider(1, 1);
  if (D == 64 && wpe3_fits(i8, pv_mode, dtype == SAGE_DTYPE_F32)) {
    // Three 4-wave work-groups to a CU hide more of each one's start, without
    // the second S buffer (168 VGPRs): a block takes 1.5x (INT8) to 1.7x as
    // long, shared by three.  226 keys: 267 us -> 215 per call (B2 H48
    // N17776), 697 keys 110 -> 99 (B3 H12 N10198); at 8070 keys 571 -> 620.
    const double c = sweep((Nq + 127) / 128 * Hq * B, 768, start4, i8 ? 0.78 : 0.90, 1);
    if (c < t) {
      t = c;
      best.nw = 4;
      best.wpe = 3;
    }
  }
  if (!may_split) return best;
  // FP8 P is rounded to e4m3 (relative error up to 2^-4) against the running
  // max of its own sweep.  Over ranges with maxima of their own every code
  // rounds anew: outputs 3.4 to 3.7 % apart (relative L2) from one sweep's, by
  // how many rows share the call.  Its keys stay in one sweep; packed heads
  // keep each row's blocks, hence its codes and its output bit for bit.
  const bool split_keys = !(i8 && pv_mode == SAGE_PV_FP8);
  for (const int nsplit : {1, 2, 3, 4, 6, 8, 12, 16, 24, 32}) {
    if (nsplit > (split_keys ? nt : 1)) break;
    if (nsplit > 1) consider(1, nsplit);
    if (G > 1 && !causal && Nq < 128) consider((int)G, nsplit);
  }
  return best;
}

// Workspace of the partial results: O, then (max, sum) pairs.
static int64_t part_rows(const AttnPlan& p, int64_t B, int64_t Hq, int64_t Nq) { return p.nsplit * B * Hq * Nq; }
static size_t part_bytes(const AttnPlan& p, int64_t B, int64_t Hq, int64_t Nq, int64_t D) {
  return p.part() ? (size_t)part_rows(p, B, Hq, Nq) * (D * 4 + 8) : 0;
}
static void part_setup(AttnArgs& a, const AttnPlan& p, int64_t D, char* ws) {
  a.grp = p.grp;
  a.nsplit = p.nsplit;
  a.part_o = reinterpret_cast<float*>(ws);
  a.part_ml = reinterpret_cast<float2*>(ws + (size_t)part_rows(p, a.B, a.Hq, a.Nq) * D * 4);
}

static bool strides_ok(const int64_t* s, int esize) {
  for (int i = 0; i < 3; ++i)
    if (s[i] < 0 || (s[i] * esize) % 16 != 0) return false;
  return true;
}

static bool is_float_code(int c) { return c == SAGE_DTYPE_F32 || c == SAGE_DTYPE_F16 || c == SAGE_DTYPE_BF16; }

// Checks and fills everything of AttnArgs but the Q operand.
static int attn_setup(AttnArgs& a, const char* who, const int64_t* q_strides, int q_es, const int8_t* k8,
                      const int64_t* k8_strides, const float* k_scale, const void* v, int v_dtype,
                      const float* v_scale, void* o, int o_dtype, const int64_t* o_strides, int64_t B, int64_t Hq,
                      int64_t Hkv, int64_t Nq, int64_t Nkv, int64_t D, int causal, int blkq, int blkk, int q_sub,
                      int pv_mode) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || Nq <= 0 || Nkv <= 0) return fail("%s: invalid argument: empty shape", who);
  if (D != 64 && D != 128) return fail("%s: invalid argument: head_dim %lld (supported: 64, 128)", who, (long long)D);
  if (Hq % Hkv != 0) return fail("%s: invalid argument: Hq %% Hkv != 0", who);
  if (Nq > 0x7FFFFFFF || Nkv > 0x7FFFFFFF || Hq > 0xFFFF || B > 0xFFFF)
    return fail("%s: invalid argument: shape too large", who);
  if (blkk != 64 && blkk != 128 && blkk != 256)
    return fail("%s: invalid argument: blkk=%d (64, 128 or 256)", who, blkk);
  if (q_sub != 1 && (q_sub < 32 || q_sub % 32 != 0 || blkq % q_sub != 0))
    return fail("%s: invalid argument: q_sub=%d blkq=%d (q_sub: 1 or a multiple of 32 dividing blkq)", who, q_sub,
                blkq);
  if (!k_scale || !k8 || !v || !o || !q_strides || !k8_strides || !o_strides)
    return fail("%s: invalid argument: null pointer", who);
  if (pv_mode != SAGE_PV_F16 && pv_mode != SAGE_PV_BF16 && pv_mode != SAGE_PV_FP8)
    return fail("%s: invalid argument: pv_mode %d", who, pv_mode);
  if (!is_float_code(o_dtype)) return fail("%s: invalid argument: o_dtype %d", who, o_dtype);
  if (v_dtype != SAGE_DTYPE_VTILES)
    return fail("%s: invalid argument: v_dtype %d (V must be in the tile layout of sage_vtiles)", who, v_dtype);
  if (pv_mode == SAGE_PV_FP8 && !v_scale) return fail("%s: invalid argument: FP8 P.V needs v_scale", who);
  const int oes = o_dtype == SAGE_DTYPE_F32 ? 4 : 2;
  const bool rows32 = (Nq * q_strides[2] + D) * q_es < 0x7FFFFFFF && Nkv * k8_strides[2] + D < 0x7FFFFFFF &&
                      Nq * o_strides[2] + D < 0x7FFFFFFF;
  if (!rows32) return fail("%s: invalid argument: a head's rows must span < 2^31 elements", who);
  if (!strides_ok(q_strides, q_es) || !strides_ok(k8_strides, 1) || !strides_ok(o_strides, oes))
    return fail("%s: invalid argument: strides must keep 16-byte aligned rows", who);
  if (((uintptr_t)k8 | (uintptr_t)v | (uintptr_t)o) % 16 != 0)
    return fail("%s: invalid argument: base pointers must be 16-byte aligned", who);
  a.k8 = k8;
  a.k_scale = k_scale;
  a.v = v;
  a.v_scale = v_scale;
  a.o = o;
  for (int i = 0; i < 2; ++i) {
    a.sq[i] = q_strides[i];
    a.sk[i] = k8_strides[i];
    a.so[i] = o_strides[i];
  }
  a.sqn = (int)q_strides[2];
  a.skn = (int)k8_strides[2];
  a.son = (int)o_strides[2];
  a.B = (int)B;
  a.Hq = (int)Hq;
  a.Hkv = (int)Hkv;
  a.Nq = (int)Nq;
  a.Nkv = (int)Nkv;
  a.causal = causal ? 1 : 0;
  a.q_sub = q_sub;
  a.blkk_shift = blkk == 64 ? 0 : (blkk == 128 ? 1 : 2);
  a.nqs = (int)(((Nq + blkq - 1) / blkq) * (blkq / q_sub));
  a.nks = (int)((Nkv + blkk - 1) / blkk);
  return 0;
}

// waves per work-group of the entry points that have no workspace
static int stage_nw(AttnArgs& a, int64_t D, int pv_mode, int dtype) {
#if SAGE_TRACE
  if (g_trace) return 8;  // what is traced
#endif
  // A head's rows within one 4-wave work-group, each with a CU to itself: 4 waves
  // have nothing to gain, and at D = 128 with fp16 or bf16 P the idle waves of 8
  // are worth their share of the tile loads.  58 rows over 9570 keys, B4 H6: 108.6
  // us against 114.0, fp32 outputs 107.9 against 159.9; over 1500, 25.2 against
  // 26.2.  (At D = 64 4 waves are 1 to 4 % faster there, with FP8 P 0 to 7 %; the
  // whole calls split such keys.)
  if (D == 128 && pv_mode != SAGE_PV_FP8 && a.Nq <= 128 && (int64_t)a.B * a.Hq <= 256) return 8;
  const AttnPlan p = attn_plan(a.B, a.Hq, a.Hkv, a.Nq, a.Nkv, D, a.causal != 0, true, pv_mode, dtype, false);
  a.wpe = p.wpe;
  return p.nw;
}

}  // namespace sage

using namespace sage;

extern "C" int sage_attn_fwd(const int8_t* q8, const int64_t* q8_strides, const float* q_scale,
                             const int8_t* k8, const int64_t* k8_strides, const float* k_scale,
                             const void* v, int v_dtype, const int64_t* v_strides, const float* v_scale,
                             void* o, int o_dtype, const int64_t* o_strides, int64_t B, int64_t Hq,
                             int64_t Hkv, int64_t Nq, int64_t Nkv, int64_t D, int causal, int blkq,
                             int blkk, int q_sub, int pv_mode, void* stream) {
  (void)v_strides;
  const char* who = "sage_attn_fwd";
  if (!q8 || !q_scale || !q8_strides) return fail("%s: invalid argument: null pointer", who);
  AttnArgs a{};
  if (int rc = attn_setup(a, who, q8_strides, 1, k8, k8_strides, k_scale, v, v_dtype, v_scale, o, o_dtype,
                          o_strides, B, Hq, Hkv, Nq, Nkv, D, causal, blkq, blkk, q_sub, pv_mode))
    return rc;
  if ((uintptr_t)q8 % 16 != 0) return fail("%s: invalid argument: base pointers must be 16-byte aligned", who);
  a.q8 = q8;
  a.q_scale = q_scale;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return launch_attn_i8(a, (int)D, pv_mode, o_dtype, stage_nw(a, D, pv_mode, o_dtype), st, who);
}

extern "C" int sage_attn_fwd_q(const void* q, const int64_t* q_strides, int q_dtype, float q_mul, int8_t* q8_out,
                               float* q_scale_out, const int8_t* k8, const int64_t* k8_strides,
                               const float* k_scale, const void* v, int v_dtype, const int64_t* v_strides,
                               const float* v_scale, void* o, const int64_t* o_strides, int64_t B, int64_t Hq,
                               int64_t Hkv, int64_t Nq, int64_t Nkv, int64_t D, int causal, int blkq, int blkk,
                               int q_sub, int pv_mode, void* stream) {
  (void)v_strides;
  const char* who = "sage_attn_fwd_q";
  if (!q || !q_strides) return fail("%s: invalid argument: null pointer", who);
  if (!is_float_code(q_dtype)) return fail("%s: invalid argument: q_dtype %d", who, q_dtype);
  if (blkq != 128) return fail("%s: invalid argument: blkq=%d (128: the rows of 4 waves)", who, blkq);
  if (!(q_mul > 0.0f) || q_mul == INFINITY) return fail("%s: invalid argument: q_mul %g", who, q_mul);
  const int qes = q_dtype == SAGE_DTYPE_F32 ? 4 : 2;
  AttnArgs a{};
  if (int rc = attn_setup(a, who, q_strides, qes, k8, k8_strides, k_scale, v, v_dtype, v_scale, o, q_dtype,
                          o_strides, B, Hq, Hkv, Nq, Nkv, D, causal, blkq, blkk, q_sub, pv_mode))
    return rc;
  if (((uintptr_t)q | (uintptr_t)q8_out) % 16 != 0)
    return fail("%s: invalid argument: base pointers must be 16-byte aligned", who);
  a.q8 = q;
  a.q_mul = q_mul;
  a.q8_out = q8_out;
  a.qs_out = q_scale_out;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return launch_attn_i8q(a, (int)D, pv_mode, q_dtype, stage_nw(a, D, pv_mode, q_dtype), st, who);
}

#if SAGE_TRACE
// Measurement build only (include/sage_trace.h): the attention launches that
// follow write their phase trace into buf (at least grid * 8 * 16 words), or
// into nothing again after a call with buf = NULL.
extern "C" int sage_trace_attach(unsigned long long* buf, int64_t words) {
  if (buf && words <= 0) return fail("sage_trace_attach: invalid argument: words %lld", (long long)words);
  g_trace = buf;
  g_trace_words = buf ? words : 0;
  return 0;
}
#endif

// Checks of the unquantized kernel and everything of AttnArgs but V.
static int flash_setup(AttnArgs& a, const char* who, const void* q, const int64_t* q_strides, const void* k,
                       const int64_t* k_strides, void* o, const int64_t* o_strides, int in_dtype, int64_t B,
                       int64_t Hq, int64_t Hkv, int64_t Nq, int64_t Nkv, int64_t D, float qk_mul, int causal) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || Nq <= 0 || Nkv <= 0) return fail("%s: invalid argument: empty shape", who);
  if (D != 64 && D != 128)
    return fail("%s: invalid argument: head_dim %lld (supported: 64, 128)", who, (long long)D);
  if (Hq % Hkv != 0) return fail("%s: invalid argument: Hq %% Hkv != 0", who);
  if (Nq > 0x7FFFFFFF || Nkv > 0x7FFFFFFF || Hq > 0xFFFF || B > 0xFFFF)
    return fail("%s: invalid argument: shape too large", who);
  if (in_dtype != SAGE_DTYPE_F16 && in_dtype != SAGE_DTYPE_BF16)
    return fail("%s: invalid argument: in_dtype %d (fp16 or bf16)", who, in_dtype);
  if (!q || !k || !o || !q_strides || !k_strides || !o_strides)
    return fail("%s: invalid argument: null pointer", who);
  if (!(qk_mul > 0.0f) || qk_mul == INFINITY) return fail("%s: invalid argument: qk_mul %g", who, qk_mul);
  const bool rows32 = (Nq * q_strides[2] + D) * 2 < 0x7FFFFFFF && (Nkv * k_strides[2] + D) * 2 < 0x7FFFFFFF &&
                      Nq * o_strides[2] + D < 0x7FFFFFFF;
  if (!rows32) return fail("%s: invalid argument: a head's rows must span < 2^31 bytes", who);
  if (!strides_ok(q_strides, 2) || !strides_ok(k_strides, 2) || !strides_ok(o_strides, 2))
    return fail("%s: invalid argument: strides must keep 16-byte aligned rows", who);
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)o) % 16 != 0)
    return fail("%s: invalid argument: base pointers must be 16-byte aligned", who);
  a.q8 = q;
  a.k8 = k;
  a.o = o;
  for (int i = 0; i < 2; ++i) {
    a.sq[i] = q_strides[i];
    a.sk[i] = k_strides[i];
    a.so[i] = o_strides[i];
  }
  a.sqn = (int)q_strides[2];
  a.skn = (int)k_strides[2];
  a.son = (int)o_strides[2];
  a.B = (int)B;
  a.Hq = (int)Hq;
  a.Hkv = (int)Hkv;
  a.Nq = (int)Nq;
  a.Nkv = (int)Nkv;
  a.causal = causal ? 1 : 0;
  a.q_sub = 32;
  a.nqs = a.nks = 1;
  a.qk_mul = qk_mul;
  return 0;
}

extern "C" int sage_flash_fwd(const void* q, const int64_t* q_strides, const void* k, const int64_t* k_strides,
                              const void* v, int v_dtype, const int64_t* v_strides, void* o,
                              const int64_t* o_strides, int in_dtype, int64_t B, int64_t Hq, int64_t Hkv,
                              int64_t Nq, int64_t Nkv, int64_t D, float qk_mul, int causal, void* stream) {
  (void)v_strides;
  const char* who = "sage_flash_fwd";
  AttnArgs a{};
  if (int rc = flash_setup(a, who, q, q_strides, k, k_strides, o, o_strides, in_dtype, B, Hq, Hkv, Nq, Nkv, D,
                           qk_mul, causal))
    return rc;
  if (!v) return fail("%s: invalid argument: null pointer", who);
  if (v_dtype != SAGE_DTYPE_VTILES)
    return fail("%s: invalid argument: v_dtype %d (V must be in the tile layout of sage_vtiles)", who, v_dtype);
  if ((uintptr_t)v % 16 != 0) return fail("%s: invalid argument: base pointers must be 16-byte aligned", who);
  a.v = v;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return launch_attn_flash(a, (int)D, in_dtype, 8, st, who);
}

// V read in place (sage_attn_kernel.h, kVRow)
static bool vrow_ok(const sage_call& c) {
  return c.v && (uintptr_t)c.v % 16 == 0 && strides_ok(c.v_strides, 2) && c.v_strides[2] < (1 << 25);
}
static void set_vrow(AttnArgs& a, const sage_call& c) {
  a.v = c.v;
  a.sv[0] = c.v_strides[0];
  a.sv[1] = c.v_strides[1];
  a.svn = (int)c.v_strides[2];
  a.vrow = 1;
}

static bool call_ok(const sage_call* c) { return c && c->size == (int64_t)sizeof(sage_call); }
static bool shape_ok(const sage_call* c) {
  return c->B > 0 && c->Hq > 0 && c->Hkv > 0 && c->Nq > 0 && c->Nkv > 0 && c->Hq % c->Hkv == 0;
}

extern "C" size_t sage_flash_run_workspace_bytes(const sage_call* c) {
  if (!call_ok(c) || !shape_ok(c)) return 0;
  return part_bytes(attn_plan(c->B, c->Hq, c->Hkv, c->Nq, c->Nkv, c->D, c->causal != 0, false, 0, (int)c->dtype, true), c->B, c->Hq, c->Nq, c->D);
}

extern "C" int sage_flash_run(const sage_call* c, void* stream) {
  const char* who = "sage_flash_run";
  if (!call_ok(c)) return fail("%s: invalid argument: sage_call size", who);
  AttnArgs a{};
  if (int rc = flash_setup(a, who, c->q, c->q_strides, c->k, c->k_strides, c->o, c->o_strides, (int)c->dtype, c->B,
                           c->Hq, c->Hkv, c->Nq, c->Nkv, c->D, (float)c->mul, (int)c->causal))
    return rc;
  if (!vrow_ok(*c))
    return fail("%s: invalid argument: V must have 16-byte aligned rows less than 2^25 elements apart", who);
  set_vrow(a, *c);
  const AttnPlan p = attn_plan(c->B, c->Hq, c->Hkv, c->Nq, c->Nkv, c->D, c->causal != 0, false, 0, (int)c->dtype, true);
  const size_t need = part_bytes(p, c->B, c->Hq, c->Nq, c->D);
  if (need && (!c->workspace || (size_t)c->workspace_bytes < need || (uintptr_t)c->workspace % 256 != 0))
    return fail("%s: invalid argument: workspace (%zu bytes, 256-byte aligned)", who, need);
  hipStream_t st = static_cast<hipStream_t>(stream);
#if SAGE_TRACE  // only 8-wave launches are traced: another plan's writes the output after one of those
  if (g_trace && (p.part() || p.nw != 8)) {
    a.trace_extra = 1;
    if (int rc = launch_attn_flash(a, (int)c->D, (int)c->dtype, 8, st, who)) return rc;
  }
#endif
  if (p.part()) {
    part_setup(a, p, c->D, static_cast<char*>(c->workspace));
    return launch_attn_part(a, (int)c->D, 0, false, (int)c->dtype, st, who);
  }
  a.wpe = p.wpe;
  return launch_attn_flash(a, (int)c->D, (int)c->dtype, p.nw, st, who);
}

namespace sage {

// AttnArgs of a sage_run call: INT8 Q from the pre-pass (quantized) or Q itself.
static int attn_args(AttnArgs& a, const char* who, const sage_call& c, bool quantized, int8_t* q8,
                     const int64_t* q8_strides, float* qs, const int8_t* k8, const int64_t* k8_strides,
                     const float* ks, const void* vt, const float* vs) {  // vt NULL: V read in place
  const float mul = (float)c.mul;
  const int qes = quantized ? 1 : (c.dtype == SAGE_DTYPE_F32 ? 4 : 2);
  if (int rc = attn_setup(a, who, quantized ? q8_strides : c.q_strides, qes, k8, k8_strides, ks, vt ? vt : c.v,
                          SAGE_DTYPE_VTILES, vs, c.o, (int)c.dtype, c.o_strides, c.B, c.Hq, c.Hkv, c.Nq, c.Nkv, c.D,
                          (int)c.causal, 128, 64, (int)c.q_sub, (int)c.pv_mode))
    return rc;
  if (((uintptr_t)c.q | (uintptr_t)q8) % 16 != 0)
    return fail("%s: invalid argument: base pointers must be 16-byte aligned", who);
  if (!vt) set_vrow(a, c);
  if (quantized) {
    a.q8 = q8;
    a.q_scale = qs;
  } else {
    if (!c.q) return fail("%s: invalid argument: null pointer", who);
    a.q8 = c.q;
    a.q_mul = mul;
    a.q8_out = q8;
    a.qs_out = qs;
  }
  return 0;
}

// Q the attention's prologue can quantize: a positive finite multiplier, a
// head's rows within 2^31 bytes (32-bit row offsets).
static bool q_fusable(const sage_call& c) {
  const float mul = (float)c.mul;
  const int qes = c.dtype == SAGE_DTYPE_F32 ? 4 : 2;
  return mul > 0.0f && mul != INFINITY && (c.Nq * c.q_strides[2] + c.D) * qes < 0x7FFFFFFF;
}

// Stages of one sage_run call and the pieces of its workspace.
struct RunPlan {
  AttnPlan attn;
  bool fuse_q;   // Q quantized in the prologue, if the attention's plan allows it
  bool quant_q;  // Q quantized in the pre-pass
  bool vrow;     // V read in place instead of through V tiles
  int v_mode;
  size_t off_q8, off_qs, off_k8, off_ks, off_km, off_vs, off_pre, off_vt, off_part, pre_bytes, vt_bytes, bytes;
};

static RunPlan run_plan(const sage_call* c) {
  RunPlan r;
  r.attn = attn_plan(c->B, c->Hq, c->Hkv, c->Nq, c->Nkv, c->D, c->causal != 0, true, (int)c->pv_mode, (int)c->dtype, true);
  // The prologue saves a pass over Q (written and read again) and lengthens
  // each work-group's start.  By 128-row blocks of Q, whole calls: many times
  // the CUs, it is 3 to 15 % faster (226 keys, B2 H48 N17776 D64: 215 us
  // against 249; B2 H32 N2048 D128: 140.5 against 145.5); fewer than the CUs,
  // the start is what counts and the pre-pass is up to 11 % faster (B1 H18 N159
  // D128: 18.6 us against 20.6).  Between, 257 to 512 blocks in one round of
  // work-groups, they are within 3 % either way (B1 H24 N1333 D128 bf16 51.9
  // prologue, 51.1 pre-pass; B1 H24 N2000 62.6 and 64.4; B1 H40 N900 D64 33.5
  // and 33.1), so the line at the number of CUs costs nothing there.
  // (the prologue takes only what sage_attn_fwd_q does: q_fusable; it writes a
  // caller's Q8 with q's strides, which is the layout of fuse_q 1 alone)
  r.fuse_q = c->fuse_q < 0 ? (c->Nq + 127) / 128 * c->Hq * c->B > 256 && q_fusable(*c) && !c->q8 : c->fuse_q != 0;
  r.quant_q = !r.fuse_q || r.attn.part();  // the partial kernels read Q8
  // V already in the P.V type: read in place, no V tiles (4 bytes of traffic
  // per element less: fp16 B8 H16 N4096 D64 548 us -> 536, 32 rows over 16384
  // keys B2 8 KV heads D128 99 -> 87, B1 H24 N1333 D128 51.7 -> 49.8; no shape
  // measured slower by more than its runs differ)
  r.vrow = ((c->dtype == SAGE_DTYPE_F16 && c->pv_mode == SAGE_PV_F16) ||
            (c->dtype == SAGE_DTYPE_BF16 && c->pv_mode == SAGE_PV_BF16)) &&
           vrow_ok(*c);
  r.v_mode = c->pv_mode == SAGE_PV_FP8 ? SAGE_V_FP8_SCALE : SAGE_V_NONE;
  r.pre_bytes = sage_prepass_workspace_bytes(c->B, c->Hkv, c->Nkv, c->D, (int)c->smooth_k, r.v_mode);
  r.vt_bytes = r.vrow ? 0 : sage_vtile_bytes(c->B, c->Hkv, c->Nkv, c->D, (int)c->pv_mode);
  size_t at = 0;
  auto take = [&](size_t n) {
    const size_t o = at;
    at += (n + 255) / 256 * 256;
    return o;
  };
  const size_t kvd = (size_t)c->B * c->Hkv * c->D;
  r.off_q8 = take(r.quant_q && !c->q8 ? (size_t)c->B * c->Hq * c->Nq * c->D : 0);
  r.off_qs = take(r.quant_q && !c->q_scale ? (size_t)c->B * c->Hq * ((c->Nq + 127) / 128) * (128 / c->q_sub) * 4 : 0);
  r.off_k8 = take(c->k8 ? 0 : kvd * c->Nkv);
  r.off_ks = take(c->k_scale ? 0 : (size_t)c->B * c->Hkv * ((c->Nkv + 63) / 64) * 4);
  r.off_km = take(c->km || !c->smooth_k ? 0 : kvd * 4);
  r.off_vs = take(c->v_scale || r.v_mode == SAGE_V_NONE ? 0 : kvd * 4);
  r.off_pre = take(r.pre_bytes);
  r.off_vt = take(r.vt_bytes);
  r.off_part = take(part_bytes(r.attn, c->B, c->Hq, c->Nq, c->D));
  r.bytes = at;
  return r;
}

static bool run_options_ok(const sage_call* c) {
  return (c->D == 64 || c->D == 128) && (c->q_sub == 1 || c->q_sub == 32 || c->q_sub == 128) &&
         (c->pv_mode == SAGE_PV_F16 || c->pv_mode == SAGE_PV_BF16 || c->pv_mode == SAGE_PV_FP8);
}

}  // namespace sage

extern "C" size_t sage_run_workspace_bytes(const sage_call* c) {
  if (!call_ok(c) || !shape_ok(c) || !run_options_ok(c)) return 0;
  return run_plan(c).bytes;
}

static int run_check(const char* who, const sage_call* c) {
  if (!call_ok(c)) return fail("%s: invalid argument: sage_call size", who);
  if (!shape_ok(c)) return fail("%s: invalid argument: empty shape or Hq %% Hkv != 0", who);
  if (c->D != 64 && c->D != 128)
    return fail("%s: invalid argument: head_dim %lld (supported: 64, 128)", who, (long long)c->D);
  if (!run_options_ok(c)) return fail("%s: invalid argument: q_sub or pv_mode", who);
  return 0;
}

extern "C" int sage_run_stages(const sage_call* c, int* quant_q, int* v_tiles) {
  const char* who = "sage_run_stages";
  if (int rc = run_check(who, c)) return rc;
  if (!quant_q || !v_tiles) return fail("%s: invalid argument: null pointer", who);
  const RunPlan r = run_plan(c);
  *quant_q = r.quant_q;
  *v_tiles = !r.vrow;
  return 0;
}

extern "C" int sage_run(const sage_call* c, void* stream) {
  const char* who = "sage_run";
  if (int rc = run_check(who, c)) return rc;
  const RunPlan r = run_plan(c);
  char* ws = static_cast<char*>(c->workspace);
  if (r.bytes && (!ws || (size_t)c->workspace_bytes < r.bytes || (uintptr_t)ws % 256 != 0))
    return fail("%s: invalid argument: workspace (%zu bytes, 256-byte aligned)", who, r.bytes);

  const int64_t q8_dense[3] = {c->Hq * c->Nq * c->D, c->Nq * c->D, c->D};
  const int64_t k8_dense[3] = {c->Hkv * c->Nkv * c->D, c->Nkv * c->D, c->D};
  // the layout of a caller's Q8 goes by the options, not by which launch writes it
  const bool q8_as_q = c->q8 && c->fuse_q > 0;
  const int64_t* q8_strides = q8_as_q ? c->q_strides : c->q8 ? c->q8_strides : q8_dense;
  const int64_t* k8_strides = c->k8 ? c->k8_strides : k8_dense;
  int8_t* q8 = static_cast<int8_t*>(c->q8 || !r.quant_q ? c->q8 : ws + r.off_q8);
  float* qs = static_cast<float*>(c->q_scale || !r.quant_q ? c->q_scale : ws + r.off_qs);
  int8_t* k8 = static_cast<int8_t*>(c->k8 ? c->k8 : ws + r.off_k8);
  float* ks = static_cast<float*>(c->k_scale ? c->k_scale : ws + r.off_ks);
  float* km = static_cast<float*>(c->smooth_k ? (c->km ? c->km : ws + r.off_km) : nullptr);
  float* vs = static_cast<float*>(r.v_mode != SAGE_V_NONE ? (c->v_scale ? c->v_scale : ws + r.off_vs) : nullptr);
  const float mul = (float)c->mul;
  // A call is held to the prologue's limits by its options (left to choose, by
  // the head dim), not by where its shape has Q quantized.
  if ((c->fuse_q < 0 ? c->D == 128 : c->fuse_q != 0) && !q_fusable(*c)) {
    if (!(mul > 0.0f) || mul == INFINITY) return fail("%s: invalid argument: mul %g", who, mul);
    return fail("%s: invalid argument: a head's rows must span < 2^31 bytes", who);
  }
  if (q8_as_q && !strides_ok(c->q_strides, 1))
    return fail("%s: invalid argument: q8 with q's strides must keep 16-byte aligned rows", who);

  const int pv = (int)c->pv_mode, dt = (int)c->dtype, q_sub = (int)c->q_sub;
  const bool dq = r.quant_q;
  void* vt = r.vrow ? nullptr : ws + r.off_vt;
  if (int rc = prepass_any(who, dq ? c->q : nullptr, c->k, r.vrow ? nullptr : c->v, dt, c->B, c->Hq, c->Hkv, c->Nq,
                           c->Nkv, c->D, dq ? c->q_strides : nullptr, c->k_strides, c->v_strides, mul, 128, 64, q_sub,
                           (int)c->smooth_k, r.v_mode, dq ? q8 : nullptr, dq ? q8_strides : nullptr,
                           dq ? qs : nullptr, k8, k8_strides, ks, km, nullptr, nullptr, vs, ws + r.off_pre,
                           r.pre_bytes, pv, vt, r.vt_bytes, stream))
    return rc;
  hipStream_t st = static_cast<hipStream_t>(stream);
  AttnArgs a{};
  if (int rc = attn_args(a, who, *c, dq, q8, q8_strides, qs, k8, k8_strides, ks, vt, vs)) return rc;
#if SAGE_TRACE  // as in sage_flash_run
  if (g_trace && (r.attn.part() || r.attn.nw != 8)) {
    a.trace_extra = 1;
    if (int rc = dq ? launch_attn_i8(a, (int)c->D, pv, dt, 8, st, who) : launch_attn_i8q(a, (int)c->D, pv, dt, 8, st, who))
      return rc;
  }
#endif
  if (r.attn.part()) {
    part_setup(a, r.attn, c->D, ws + r.off_part);
    return launch_attn_part(a, (int)c->D, pv, true, dt, st, who);
  }
  a.wpe = r.attn.wpe;
  return dq ? launch_attn_i8(a, (int)c->D, pv, dt, r.attn.nw, st, who)
            : launch_attn_i8q(a, (int)c->D, pv, dt, r.attn.nw, st, who);
}
