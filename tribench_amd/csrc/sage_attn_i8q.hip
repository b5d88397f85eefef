// sage_attn_i8q.hip — the INT8 attention kernels, Q (in the output type) quantized in the prologue.
#include "sage_attn_kernel.h"

int sage::launch_attn_i8q(const AttnArgs& a, int D, int pv_mode, int o_dtype, int nw, hipStream_t st, const char* who) {
  switch (o_dtype) {
    case SAGE_DTYPE_F32: return launch_attn_int8<kQkI8Q, float>(a, D, pv_mode, nw, st, who);
    case SAGE_DTYPE_F16: return launch_attn_int8<kQkI8Q, _Float16>(a, D, pv_mode, nw, st, who);
    default: return launch_attn_int8<kQkI8Q, __bf16>(a, D, pv_mode, nw, st, who);
  }
}
