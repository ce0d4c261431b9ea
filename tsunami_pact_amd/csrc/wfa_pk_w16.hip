// Packed kernel, 16 waves per pair.
#include "wfa_pk_pick.h"

namespace tsu {
KernelFn pick_pk_w16(const Shape& sh) {
    if (sh.reg_c == 3) return pick_pk_queue<16, 3>(sh);
    if (sh.reg_c == 5) return pick_pk_queue<16, 5>(sh);
    if (sh.reg_c == 9) return pick_pk_shape<16, 9>(sh);
    if (sh.reg_c == 14 && sh.queue && !sh.bt && !sh.probe)  // the widest window, queue-fed, scores only
        return sh.expand ? wfa_pk_kernel<16, 14, true, true> : wfa_pk_kernel<16, 14, false, true>;
    return nullptr;
}
}  // namespace tsu
