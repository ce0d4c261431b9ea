// Packed kernel, one wave per pair.
#include "wfa_pk_pick.h"

namespace tsu {
KernelFn pick_pk_w1(const Shape& sh) {
    if (sh.reg_c == 1) return pick_pk_shape<1, 1>(sh);
    if (sh.reg_c == 3) return pick_pk_shape<1, 3>(sh);
    if (sh.reg_c == 5) return pick_pk_shape<1, 5>(sh);
    if (sh.reg_c == 9) return pick_pk_shape<1, 9>(sh);
    return nullptr;
}
}  // namespace tsu
