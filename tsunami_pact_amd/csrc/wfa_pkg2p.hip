// Packed kernel, two gap pieces; scores only.
#include "wfa_pkg_pick.h"

namespace tsu {

template <int E1, int E2>
static KernelFn pick_registers(const Shape& sh) {
    if (sh.expand) return sh.queue ? wfa_pkg_kernel<8, 2, true, true, E1, E2> : wfa_pkg_kernel<8, 2, true, false, E1, E2>;
    return sh.queue ? wfa_pkg_kernel<8, 2, false, true, E1, E2> : wfa_pkg_kernel<8, 2, false, false, E1, E2>;
}

KernelFn pick_pkg2p(const Shape& sh) {
    if (!pkg_in_registers(sh) || sh.bt || sh.probe) return pick_pkg_waves<2>(sh);
    switch (sh.reg_e) {
    case 11: return pick_registers<1, 1>(sh);
    case 21: return pick_registers<2, 1>(sh);
    case 31: return pick_registers<3, 1>(sh);
    default: return nullptr;
    }
}

}  // namespace tsu
