// Packed kernel, 2 waves per pair.
#include "wfa_pk_pick.h"

namespace tsu {
KernelFn pick_pk_w2(const Shape& sh) {
    if (sh.reg_c == 3) return pick_pk_queue<2, 3>(sh);
    if (sh.reg_c == 5) return pick_pk_queue<2, 5>(sh);
    if (sh.reg_c == 9) return pick_pk_shape<2, 9>(sh);
    return nullptr;
}
}  // namespace tsu
