// sage_attn_flash.hip — the unquantized attention kernels: QK and P.V in the
// input type (the reference casts P to V's dtype,
// kernels/flash_attn/triton_impl.py:87-88), V in tiles or in place.
#include "sage_attn_kernel.h"

namespace sage {

template <int QKM, int D, typename TO>
static int launch_flash_d(const AttnArgs& a, int nw, hipStream_t st, const char* who) {
  constexpr int PVM = QKM == kQkF16 ? SAGE_PV_F16 : SAGE_PV_BF16;
  if (!a.vrow) return launch_attn_nw<QKM, D, PVM, TO, 8, false>(a, st, who);
  return nw == 4 ? launch_attn_nw<QKM, D, PVM, TO, 4, true>(a, st, who)
                 : launch_attn_nw<QKM, D, PVM, TO, 8, true>(a, st, who);
}

int launch_attn_flash(const AttnArgs& a, int D, int dtype, int nw, hipStream_t st, const char* who) {
  if (dtype == SAGE_DTYPE_F16)
    return D == 64 ? launch_flash_d<kQkF16, 64, _Float16>(a, nw, st, who)
                   : launch_flash_d<kQkF16, 128, _Float16>(a, nw, st, who);
  return D == 64 ? launch_flash_d<kQkBF16, 64, __bf16>(a, nw, st, who)
                 : launch_flash_d<kQkBF16, 128, __bf16>(a, nw, st, who);
}

}  // namespace sage
