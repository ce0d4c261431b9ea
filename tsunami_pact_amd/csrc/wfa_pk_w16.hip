// Packed kernel, 16 waves per pair.
#include "wfa_pk_pick.h"

namespace tsu {
KernelFn pick_pk_w16(const Shape& sh) {
    if (sh.reg_c == 9) return pick_pk_shape<16, 9>(sh);
    return nullptr;
}
}  // namespace tsu
