// Packed kernel, two gap pieces; scores only.
#include "wfa_pkg_pick.h"

namespace tsu {

KernelFn pick_pkg2p(const Shape& sh) { return pick_pkg_waves<2>(sh); }

}  // namespace tsu
