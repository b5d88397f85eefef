// sage_attn_i8.hip — the INT8 attention kernels, Q8 and q_scale from the pre-pass.
#include "sage_attn_kernel.h"

int sage::launch_attn_i8(const AttnArgs& a, int D, int pv_mode, int o_dtype, int nw, hipStream_t st, const char* who) {
  switch (o_dtype) {
    case SAGE_DTYPE_F32: return launch_attn_int8<kQkI8, float>(a, D, pv_mode, nw, st, who);
    case SAGE_DTYPE_F16: return launch_attn_int8<kQkI8, _Float16>(a, D, pv_mode, nw, st, who);
    default: return launch_attn_int8<kQkI8, __bf16>(a, D, pv_mode, nw, st, who);
  }
}
