// Packed kernel for penalties other than 2/3/1 after the gcd, one gap piece;
// scores only.  Two pieces: wfa_pkg2p.hip.
#include "wfa_pkg_pick.h"

namespace tsu {

KernelFn pick_pkg2p(const Shape& sh);
KernelFn pick_pkg(const Shape& sh) { return sh.two_piece ? pick_pkg2p(sh) : pick_pkg_waves<1>(sh); }

int64_t lds_bytes_pkg(const Shape& sh, const KArgs& a) {
    const uint32_t sw = (uint32_t)a.seq_words;
    return pk_lds_bytes(sh, sw, 16 + pkg_ring_bytes(sh, a));
}

}  // namespace tsu
