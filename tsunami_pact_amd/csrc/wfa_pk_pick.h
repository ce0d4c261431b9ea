// wfa_pk_pick.h -- the packed kernel's instances for one shape; each wave
// count has a translation unit of its own (wfa_pk_w*.hip).
#pragma once

#include "wfa_pk.h"

namespace tsu {

template <int NW, int C>
KernelFn pick_pk_shape(const Shape& sh) {
    if (sh.probe) {
        if constexpr (NW == 1 && C == 5) return sh.queue && !sh.expand ? wfa_pk_kernel<1, 5, false, true, true> : nullptr;
        return nullptr;
    }
    if (sh.bt) {  // CIGAR launches are always queue-fed
        if (!sh.queue) return nullptr;
        return sh.expand ? wfa_pk_kernel<NW, C, true, true, false, true> : wfa_pk_kernel<NW, C, false, true, false, true>;
    }
    if (sh.expand) return sh.queue ? wfa_pk_kernel<NW, C, true, true> : wfa_pk_kernel<NW, C, true, false>;
    return sh.queue ? wfa_pk_kernel<NW, C, false, true> : wfa_pk_kernel<NW, C, false, false>;
}

// Shapes that only queue-fed launches take.
template <int NW, int C>
KernelFn pick_pk_queue(const Shape& sh) {
    if (!sh.queue || sh.probe) return nullptr;
    if (sh.bt) return sh.expand ? wfa_pk_kernel<NW, C, true, true, false, true> : wfa_pk_kernel<NW, C, false, true, false, true>;
    return sh.expand ? wfa_pk_kernel<NW, C, true, true> : wfa_pk_kernel<NW, C, false, true>;
}

}  // namespace tsu
