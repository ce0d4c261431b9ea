// Packed kernel, 4 waves per pair.
#include "wfa_pk_pick.h"

namespace tsu {
KernelFn pick_pk_w4(const Shape& sh) {
    if (sh.reg_c == 3) return pick_pk_queue<4, 3>(sh);
    if (sh.reg_c == 5) return pick_pk_queue<4, 5>(sh);
    if (sh.reg_c == 9) return pick_pk_shape<4, 9>(sh);
    return nullptr;
}
}  // namespace tsu
