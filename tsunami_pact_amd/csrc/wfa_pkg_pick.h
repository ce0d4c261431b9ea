// wfa_pkg_pick.h -- instances of the packed kernel for any penalties.
#pragma once

#include "wfa_pkg.h"

namespace tsu {

template <int NW, int P>
KernelFn pick_pkg_shape(const Shape& sh) {
    if (sh.expand) return sh.queue ? wfa_pkg_kernel<NW, P, true, true> : wfa_pkg_kernel<NW, P, true, false>;
    return sh.queue ? wfa_pkg_kernel<NW, P, false, true> : wfa_pkg_kernel<NW, P, false, false>;
}

template <int P>
KernelFn pick_pkg_waves(const Shape& sh) {
    if (sh.bt || sh.probe) return nullptr;
    switch (sh.nw) {
    case 1: return pick_pkg_shape<1, P>(sh);
    case 2: return pick_pkg_shape<2, P>(sh);
    case 4: return pick_pkg_shape<4, P>(sh);
    case 8: return pick_pkg_shape<8, P>(sh);
    case 16: return pick_pkg_shape<16, P>(sh);
    default: return nullptr;
    }
}

}  // namespace tsu
