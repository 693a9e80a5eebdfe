// Lazily reduced Fr arithmetic of the transform passes (ntt.hip), compiled for
// the host as well, where a test drives it to its bounds.
#pragma once

#include "field29.h"

namespace nkr {

// Inside a pass every value stays in the 29-bit form (field.h) and is lazily
// reduced: the canonical residue x 2^256 of the data is taken as it is, and
// the factors (twiddles, roots, coset powers) are stored as w 2^261, so that a
// reduced-radix product of the two is (x w) 2^256 with no conversion on either
// side.  Sums and differences are added limb by limb without carries; a value
// is carry-normalised when it goes back to LDS.  A pass is bound by the
// products' multiply-adds, half a product per element and stage.  (On 32-bit
// limbs each butterfly converted both operands and the product, and each sum
// and difference was a carry chain and a conditional subtraction: a whole
// transform of 2^21 took 349 us against 294 now with its reordering, the
// passes alone 279 against 261, one of 2^11 34.5 against 29.2.)
using fr29 = Fp29<FrParams>;

// a * b * 2^-261, limbs below 2^29, value below 1.5 r + a b / 2^261.  One
// operand may have limbs up to 2.5 * 2^30 (a column is at most 9 * 2.5 * 2^59
// + 9 * 2^58 and a carry, below 2^64); b is a canonical factor.
NKR_HD fr29 mul29(const fr29 &a, const fr29 &b)
{
    return fp29_reduce_terms<FrParams, 8>([&](int k, uint64_t &acc) { fp29_column(a, b, k, acc); });
}
NKR_HD fr29 load29(const fr_t &x) { return fp29_from_bits(x); }

// Limbs below 2^29 (the top one takes what is left), value unchanged.
NKR_HD fr29 normalise29(const fr29 &x)
{
    fr29 r;
    uint32_t c = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t t = x.l[i] + c;
        r.l[i] = t & kMask29;
        c = t >> 29;
    }
    r.l[8] = x.l[8] + c;
    return r;
}

NKR_HD fr29 add29(const fr29 &x, const fr29 &y)
{
    fr29 r;
#pragma unroll
    for (int i = 0; i < 9; ++i) r.l[i] = x.l[i] + y.l[i];
    return r;
}

// K r with 2^30 borrowed into every limb from the next, so that limbs up to
// 2^30 - 2 can be taken from it without a borrow.
struct Borrowed {
    uint32_t l[9];
};
constexpr Borrowed borrowed(uint32_t K)
{
    Borrowed b{};
    const auto kp = P29<FrParams>::times(K);
    for (int i = 0; i < 9; ++i) b.l[i] = kp.l[i] + (i < 8 ? (1u << 30) : 0u) - (i > 0 ? 2u : 0u);
    return b;
}

// x + K r - y for y below (K - 0.01) r with limbs up to 2^30 - 2; the result's
// limbs are below x's + 1.5 * 2^30.
NKR_HD fr29 sub29(const fr29 &x, const fr29 &y, const Borrowed &k)
{
    fr29 r;
#pragma unroll
    for (int i = 0; i < 9; ++i) r.l[i] = x.l[i] + k.l[i] - y.l[i];
    return r;
}

// x below 169 r, normalised -> below 1.04 r: the quotient's estimate from the
// top limb is at most 1 too small and never too large.
NKR_HD fr29 reduce29(const fr29 &x)
{
    constexpr uint32_t top = P29<FrParams>::bits(8) + 1;
    constexpr uint32_t recip = (uint32_t)((1ull << 32) / top);
    const uint32_t q = (uint32_t)(((uint64_t)x.l[8] * recip) >> 32);
    fr29 r;
    int64_t c = 0;
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        const int64_t t = (int64_t)x.l[i] - (int64_t)((uint64_t)q * P29<FrParams>::bits(i)) + c;
        r.l[i] = (uint32_t)t & kMask29;
        c = t >> 29;
    }
    return r;
}

// The canonical residue of x (below 169 r, normalised).
NKR_HD fr_t canonical29(const fr29 &x) { return fp_reduce_once(fp29_to_bits(reduce29(x))); }

// Product of two factors in the 2^261 form, canonical in that form.
NKR_HD fr_t factor_mul(const fr_t &a, const fr_t &b)
{
    return canonical29(mul29(load29(a), load29(b)));
}
// x 2^256 -> x 2^261.
NKR_HD fr_t factor_from_mont(const fr_t &x) { return fp_dbl(fp_dbl(fp_dbl(fp_dbl(fp_dbl(x))))); }

}  // namespace nkr
