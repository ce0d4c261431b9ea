// Shapes of the packed kernel (scaled penalties 2/3/1): one wave of 1, 3,
// 5 or 9 chunks of 128 diagonals (windows of 64-128, 256, 512 and 1024), or
// 2-16 waves of 9 chunks (windows of 2048 to 16384; 14 chunks: 24576), or the
// same windows over twice or four times the waves with 5 or 3 chunks; with
// expanded or packed sequences, scores only or with backtrace records; and
// the probe, one wave of 5 chunks.
#include "wfa_pk.h"

namespace tsu {

KernelFn pick_pk_w1(const Shape& sh);
KernelFn pick_pk_w2(const Shape& sh);
KernelFn pick_pk_w4(const Shape& sh);
KernelFn pick_pk_w8(const Shape& sh);
KernelFn pick_pk_w16(const Shape& sh);

KernelFn pick_pk(const Shape& sh) {
    if (!sh.fixed_242) return nullptr;
    switch (sh.nw) {
    case 1: return pick_pk_w1(sh);
    case 2: return pick_pk_w2(sh);
    case 4: return pick_pk_w4(sh);
    case 8: return pick_pk_w8(sh);
    case 16: return pick_pk_w16(sh);
    default: return nullptr;
    }
}

int64_t lds_bytes_pk(const Shape& sh, const KArgs& a) {
    const uint32_t sw = (uint32_t)a.seq_words;
    int64_t x = 0;
    switch (100 * sh.nw + sh.reg_c) {
    case 101: x = PkLayout<1, 1>::WORDS; break;
    case 103: x = PkLayout<1, 3>::WORDS; break;
    case 105: x = PkLayout<1, 5>::WORDS; break;
    case 109: x = PkLayout<1, 9>::WORDS; break;
    case 203: x = PkLayout<2, 3>::WORDS; break;
    case 205: x = PkLayout<2, 5>::WORDS; break;
    case 209: x = PkLayout<2, 9>::WORDS; break;
    case 403: x = PkLayout<4, 3>::WORDS; break;
    case 405: x = PkLayout<4, 5>::WORDS; break;
    case 409: x = PkLayout<4, 9>::WORDS; break;
    case 803: x = PkLayout<8, 3>::WORDS; break;
    case 805: x = PkLayout<8, 5>::WORDS; break;
    case 809: x = PkLayout<8, 9>::WORDS; break;
    case 1603: x = PkLayout<16, 3>::WORDS; break;
    case 1605: x = PkLayout<16, 5>::WORDS; break;
    case 1609: x = PkLayout<16, 9>::WORDS; break;
    default: x = PkLayout<16, 14>::WORDS; break;
    }
    return pk_lds_bytes(sh, sw, 4 * x);
}

}  // namespace tsu
