// CPU check of the reduced-radix field and its mixed addition
// (nkr-zkp_amd/csrc/field29.h, curve29.h) against the canonical 32-bit-limb
// code (field.h, curve.h), compiled as host code.
//   * conversions: canonical -> 29-bit -> canonical is the identity; the
//     29-bit Montgomery one converts to the canonical one;
//   * products: every input bound the formulas use (below 2p, 10p, and 32p
//     against 2p), built as x + k*p, gives fp_mul's canonical result;
//     squarings give fp29_mul(a, a)'s limbs, and a sum of two products with
//     one reduction the canonical sum;
//   * the canonical product through the 29-bit form (fp_mul_r29) of any 256-bit
//     value is below 2p;
//   * products, sums of products and Fq2 products whose inputs are at the top of
//     what is allowed (145 p^2 in all, in several shapes) come out below 2p;
//   * the transforms' arithmetic (ntt29.h) at its bounds: products of values near
//     160 r with limbs near 2.5 * 2^30, reductions near 169 r, differences of
//     values near K r with limbs up to 2^30 - 2;
//   * lazy sums and differences: a + b and a + K*p - b are congruent to the
//     canonical ones;
//   * mixed addition: chains of xyzz29_add_affine over random bases, repeated
//     bases (doubling), negated ones (infinity) and infinity restarts give,
//     after every step, the canonical coordinates of xyzz_add_affine;
//   * full addition: chains of xyzz29_add over partial sums (ZZ != 1),
//     doublings, cancellations and infinity operands give xyzz_add's
//     coordinates after every step;
//   * the same over Fq2 (G2): products, squares and the four-product sum at
//     their input bounds, and chains of xyzz2_29_add_affine against
//     xyzz_add_affine.
//     The formulas are field identities, so random coordinates (not on the
//     curve) exercise them as well as curve points do.
// Prints "ok <checks>" or the first mismatches; exit status 1 on a mismatch.
#include <cstdio>
#include <vector>

#include "curve29.h"
#include "ntt29.h"

using namespace nkr;

static uint64_t g_state = 0x9E3779B97F4A7C15ull;
static uint32_t rnd()
{
    g_state ^= g_state << 13;
    g_state ^= g_state >> 7;
    g_state ^= g_state << 17;
    return (uint32_t)(g_state >> 11);
}

template <class P>
static Fp<P> rand_fp()
{
    Fp<P> x;
    for (int i = 0; i < 8; ++i) x.l[i] = rnd();
    x.l[7] %= P::P[7] + 1;  // below 2p
    return fp_reduce_once(x);
}

static int g_bad = 0;
static long g_doublings = 0, g_cancels = 0;
static long g_checks = 0;
static void expect(bool ok, const char *what, int i)
{
    ++g_checks;
    if (!ok && g_bad++ < 10) std::printf("mismatch: %s at %d\n", what, i);
}

// x + K*p in the 29-bit form, x canonical (value below (K + 2) p)
template <class P, uint32_t K>
static Fp29<P> widen(const Fp<P> &x)
{
    return fp29_sub<P, K>(fp29_reduce_to_2p(fp29_from_mont(x)), Fp29<P>::zero());
}

template <class P>
static void check_field(int n)
{
    for (int i = 0; i < n; ++i) {
        Fp<P> x = rand_fp<P>(), y = rand_fp<P>();
        if (i == 0) x = y = Fp<P>::zero();
        if (i == 1) x = y = Fp<P>::one();
        if (i == 2) {
            x = Fp<P>::modulus();
            x.l[0] -= 1;  // p - 1
            y = x;
        }
        const Fp<P> want = fp_mul(x, y);
        expect(fp29_to_mont(fp29_from_mont(x)) == x, "round trip", i);
        expect(fp29_to_mont(fp29_mul(fp29_from_mont(x), fp29_reduce_to_2p(fp29_from_mont(y)))) == want,
               "mul 32p x 2p", i);
        expect(fp29_to_mont(fp29_mul(widen<P, 8>(x), widen<P, 8>(y))) == want, "mul 10p x 10p", i);
        expect(fp29_to_mont(fp29_mul(widen<P, 0>(x), widen<P, 0>(y))) == want, "mul 2p x 2p", i);
        expect(fp29_to_mont(fp29_sqr(widen<P, 8>(x))) == fp_mul(x, x), "sqr 10p", i);
        {
            const Fp29<P> wx = widen<P, 8>(x), s0 = fp29_sqr(wx), s1 = fp29_mul(wx, wx);
            bool same = true;
            for (int k = 0; k < 9; ++k) same = same && s0.l[k] == s1.l[k];
            expect(same, "sqr limbs equal mul(a, a)", i);
        }
        {
            // the G1 Y3 shape: 10p x 10p + 8p x 2p in one reduction
            const Fp<P> u = rand_fp<P>(), v = rand_fp<P>();
            const Fp29<P> s = fp29_mul_add(widen<P, 8>(x), widen<P, 8>(y), widen<P, 6>(u), widen<P, 0>(v));
            bool limbs = true;
            for (int k = 0; k < 9; ++k) limbs = limbs && (s.l[k] >> 29) == 0;
            expect(limbs && fp29_to_mont(s) == fp_add(fp_mul(x, y), fp_mul(u, v)), "mul_add", i);
        }
        const Fp29<P> m = fp29_mul(widen<P, 8>(x), widen<P, 8>(y));
        bool limbs = true;
        for (int k = 0; k < 9; ++k) limbs = limbs && (m.l[k] >> 29) == 0;
        expect(limbs, "product limbs below 2^29", i);
        expect(fp29_to_mont(fp29_add(widen<P, 0>(x), widen<P, 4>(y))) == fp_add(x, y), "add", i);
        expect(fp29_to_mont(fp29_sub<P, 8>(widen<P, 0>(x), widen<P, 4>(y))) == fp_sub(x, y), "sub", i);
        expect(fp29_to_mont(fp29_reduce_to_8p(fp29_from_mont(x))) == x, "reduce to 8p", i);
        const bool z = fp_sub(x, y).is_zero();
        const Fp29<P> d = fp29_sub<P, 8>(widen<P, 0>(x), widen<P, 0>(y));
        expect(!z || fp29_may_be_zero<P, 10>(d), "zero filter", i);
    }
    expect(fp29_to_mont(Fp29<P>::one()) == Fp<P>::one(), "one", 0);
    // the zero filter passes every multiple j*p below 10p
    const Fp29<P> z = Fp29<P>::zero();
    expect(fp29_may_be_zero<P, 10>(z) && fp29_may_be_zero<P, 10>(fp29_sub<P, 1>(z, z)) &&
               fp29_may_be_zero<P, 10>(fp29_sub<P, 5>(z, z)) && fp29_may_be_zero<P, 10>(fp29_sub<P, 9>(z, z)),
           "zero filter on multiples of p", 0);
}

// K p - 1 - d, the d-th value below K p.
template <class P, uint32_t K>
static Fp29<P> below(const Fp<P> &d)
{
    Fp29<P> one = Fp29<P>::zero();
    one.l[0] = 1;
    return fp29_sub<P, K>(Fp29<P>::zero(), fp29_add(fp29_from_bits(d), one));
}
// What below(d) stands for, canonical (the same for every K).
template <class P>
static Fp<P> below_residue(const Fp<P> &d)
{
    return fp29_to_mont(below<P, 2>(d));
}
// The smallest offsets most of the time, any other now and then.
template <class P>
static Fp<P> offset(int i)
{
    Fp<P> d = Fp<P>::zero();
    d.l[0] = i < 4 ? i : rnd();
    return i % 5 == 4 ? rand_fp<P>() : d;
}
template <class P, uint32_t K>
static bool is_below(const Fp29<P> &x)
{
    const Fp29<P> y = fp29_sub_if_ge<P, K>(x);
    bool same = true;
    for (int k = 0; k < 9; ++k) same = same && x.l[k] == y.l[k];
    return same;
}
template <class P>
static void expect_product(const Fp29<P> &r, const Fp<P> &want, const char *what, int i)
{
    bool limbs = true;
    for (int k = 0; k < 9; ++k) limbs = limbs && (r.l[k] >> 29) == 0;
    expect(limbs && is_below<P, 2>(r) && fp29_to_mont(r) == want, what, i);
}

template <class P, uint32_t A, uint32_t B>
static void check_product_at(int i)
{
    static_assert(A * B <= 145, "allowed");
    const Fp<P> d = offset<P>(i), e = offset<P>(i + 1);
    expect_product(fp29_mul(below<P, A>(d), below<P, B>(e)), fp_mul(below_residue<P>(d), below_residue<P>(e)),
                   "product at 145 p^2", i);
}

template <class P>
static void check_bounds(int n)
{
    for (int i = 0; i < n; ++i) {
        check_product_at<P, 145, 1>(i);
        check_product_at<P, 72, 2>(i);
        check_product_at<P, 48, 3>(i);
        check_product_at<P, 36, 4>(i);
        check_product_at<P, 24, 6>(i);
        check_product_at<P, 18, 8>(i);
        check_product_at<P, 12, 12>(i);
        Fp<P> d[8], r[8];
        for (int k = 0; k < 8; ++k) {
            d[k] = offset<P>(i + k);
            r[k] = below_residue<P>(d[k]);
        }
        expect_product(fp29_sqr(below<P, 12>(d[0])), fp_sqr(r[0]), "square at 12p", i);
        expect_product(fp29_mul_add(below<P, 12>(d[0]), below<P, 6>(d[1]), below<P, 6>(d[2]), below<P, 12>(d[3])),
                       fp_add(fp_mul(r[0], r[1]), fp_mul(r[2], r[3])), "mul_add at 144 p^2", i);
        expect_product(fp29_mul_add4(below<P, 6>(d[0]), below<P, 6>(d[1]), below<P, 6>(d[2]), below<P, 6>(d[3]),
                                     below<P, 4>(d[4]), below<P, 9>(d[5]), below<P, 9>(d[6]), below<P, 4>(d[7])),
                       fp_add(fp_add(fp_mul(r[0], r[1]), fp_mul(r[2], r[3])),
                              fp_add(fp_mul(r[4], r[5]), fp_mul(r[6], r[7]))),
                       "mul_add4 at 144 p^2", i);
    }
}

static void check_fq2_bounds(int n)
{
    using P = FqParams;
    for (int i = 0; i < n; ++i) {
        const fq_t d[4] = {offset<P>(i), offset<P>(i + 1), offset<P>(i + 2), offset<P>(i + 3)};
        const fq2_t x = {below_residue<P>(d[0]), below_residue<P>(d[1])};
        const fq2_t y = {below_residue<P>(d[2]), below_residue<P>(d[3])};
        const fq2_t want = fq2_mul(x, y), sq = fq2_sqr(x);
        // 36p x 2p with b1 negated by 2p: c1 at 2 * 72; b1 = 0 brings c0 to 36 * 4
        for (int zero = 0; zero < 2; ++zero) {
            const Fq2_29<P> a = {below<P, 36>(d[0]), below<P, 36>(d[1])};
            const Fq2_29<P> b = {below<P, 2>(d[2]), zero ? Fp29<P>::zero() : below<P, 2>(d[3])};
            const fq2_t w = zero ? fq2_mul(x, {y.c0, fq_t::zero()}) : want;
            const Fq2_29<P> m = fq2_29_mul<P, 2>(a, b);
            expect_product(m.c0, w.c0, "fq2 product c0 at its bound", i);
            expect_product(m.c1, w.c1, "fq2 product c1 at its bound", i);
        }
        const Fq2_29<P> s = fq2_29_sqr<P, 6>({below<P, 6>(d[0]), below<P, 6>(d[1])});
        expect_product(s.c0, sq.c0, "fq2 square c0 at its bound", i);
        expect_product(s.c1, sq.c1, "fq2 square c1 at its bound", i);
    }
}

// The value of x modulo r as a canonical element, through textbook steps.
static fr_t residue29(const fr29 &x)
{
    fr29 one = fr29::zero();
    one.l[0] = 1;
    const fr29 n = normalise29(x);
    const fr29 t = fp29_reduce_terms<FrParams, 0>([&](int k, uint64_t &acc) { fp29_column(n, one, k, acc); });
    return fp_reduce_once(fp29_to_bits(t));
}
static bool equal29(const fr29 &a, const fr29 &b)
{
    for (int k = 0; k < 9; ++k)
        if (a.l[k] != b.l[k]) return false;
    return true;
}

template <uint32_t K>
static void check_sub29(int i)
{
    using P = FrParams;
    constexpr Borrowed bk = borrowed(K);
    // y: the sum of two values of K/2 r each less a little, so that its limbs
    // reach 2^30 - 2 and it stays below (K - 0.01) r
    fr_t d = rand_fp<P>();
    if (d.l[7] < P::P[7] / 50) d.l[7] += P::P[7] / 50;
    const fr29 x = i % 2 ? fr29::zero() : below<P, 79>(offset<P>(i)), p = below<P, K / 2>(offset<P>(i)),
               q = below<P, K / 2>(fp_reduce_once(d));
    const fr29 y = add29(p, q), r = sub29(x, y, bk);
    bool limbs = true;
    for (int k = 0; k < 9; ++k) limbs = limbs && r.l[k] <= x.l[k] + 3u * (1u << 29);
    const fr29 back = normalise29(add29(normalise29(r), normalise29(y)));
    expect(limbs && equal29(back, fp29_sub<P, K>(x, fr29::zero())), "sub29 at its bound", i);
}

static void check_ntt29(int n)
{
    using P = FrParams;
    for (int i = 0; i < n; ++i) {
        // a: limbs up to 2.5 * 2^30 and a value just below 160 r
        fr29 a;
        for (int k = 0; k < 8; ++k) a.l[k] = 5u * (1u << 29) - (i < 3 ? 0u : rnd() % (i % 2 ? 1000 : 1u << 31));
        a.l[8] = P29<P>::times(160).l[8] - 6 - (i < 3 ? 0u : rnd() % 1000);
        expect(is_below<P, 160>(normalise29(a)), "the operand is below 160 r", i);
        const fr_t d = offset<P>(i);
        const fr29 b = below<P, 1>(d);
        const fr29 m = mul29(a, b);
        bool limbs = true;
        for (int k = 0; k < 9; ++k) limbs = limbs && (m.l[k] >> 29) == 0;
        // m = a b 2^-261: both sides as canonical Montgomery elements of 2^261
        const fr29 ra = reduce29(normalise29(a));
        const fr29 t = fp29_reduce_terms<P, 0>([&](int k, uint64_t &acc) { fp29_column(ra, b, k, acc); });
        expect(limbs && is_below<P, 5>(fp29_add(m, m)) && residue29(m) == residue29(t), "mul29 at its bound", i);

        const fr29 top = below<P, 169>(d);
        fr29 r25 = fr29::zero();
        const fr29 red = reduce29(top);
        for (int k = 0; k < 25; ++k) r25 = fp29_add(r25, red);
        expect(is_below<P, 26>(r25) && residue29(red) == residue29(top), "reduce29 near 169 r", i);
        const fr29 any = fp29_add(below<P, 100>(rand_fp<P>()), fp29_from_mont(rand_fp<P>()));
        const fr_t c = canonical29(any);
        expect(c == fp_reduce_once(c) && residue29(load29(c)) == residue29(any), "canonical29", i);
        check_sub29<4>(i);
        check_sub29<40>(i);
        check_sub29<80>(i);
        const fr_t w = rand_fp<P>(), v = rand_fp<P>();
        expect(factor_mul(factor_from_mont(w), factor_from_mont(v)) == factor_from_mont(fp_mul(w, v)), "factor_mul", i);
    }
}

// x*w*2^-256 for any 256-bit x: below 2p, so that one subtraction makes it
// canonical, and congruent to the product of the reduced x.
template <class P>
static void check_mul_r29(int n)
{
    for (int i = 0; i < n; ++i) {
        Fp<P> x, w = rand_fp<P>();
        for (int k = 0; k < 8; ++k) x.l[k] = rnd();
        if (i % 4 != 0) {  // near 2^256, against a factor near p
            for (int k = 4; k < 8; ++k) x.l[k] = 0xffffffffu;
            w = Fp<P>::modulus();
            w.l[0] -= 1 + rnd() % 1000;
        }
        Fp<P> r = x;
        for (int k = 0; k < 5; ++k) r = fp_reduce_once(r);  // 2^256 is below 6p
        const Fp<P> got = fp_reduce_once(fp_mul_r29(x, w));
        expect(got == fp_reduce_once(got) && got == fp_mul(r, w), "mul of any 256-bit value", i);
    }
}

static Affine<fq_t> random_base(const Affine<fq_t> &g)
{
    uint32_t k[8];
    for (int i = 0; i < 8; ++i) k[i] = rnd();
    k[7] &= 0x0fffffffu;
    return xyzz_to_affine(xyzz_mul_u256(Xyzz<fq_t>::from_affine(g), k));
}

static void check_madd(int chains, int len)
{
    Affine<fq_t> g;
    g.x = fp_to_mont(fq_t::zero());
    g.x.l[0] = 1;
    g.x = fp_to_mont(g.x);
    g.y = fq_t::zero();
    g.y.l[0] = 2;
    g.y = fp_to_mont(g.y);
    std::vector<Affine<fq_t>> pool;
    for (int i = 0; i < 24; ++i) pool.push_back(random_base(g));
    for (int c = 0; c < chains; ++c) {
        Xyzz<fq_t> a32 = Xyzz<fq_t>::infinity();
        Xyzz29<FqParams> a29 = Xyzz29<FqParams>::infinity();
        for (int e = 0; e < len; ++e) {
            const uint32_t r = rnd();
            Affine<fq_t> b = pool[r % pool.size()];
            if ((r >> 8) % 5 == 0 && !a32.is_inf()) {  // doubling
                b = xyzz_to_affine(a32);
                ++g_doublings;
            }
            if ((r >> 12) % 7 == 0) b.y = fp_neg(b.y);
            if ((r >> 16) % 11 == 0 && !a32.is_inf()) {  // back to infinity
                b = xyzz_to_affine(a32);
                b.y = fp_neg(b.y);
                ++g_cancels;
            }
            a32 = xyzz_add_affine(a32, b.x, b.y);
            a29 = xyzz29_add_affine(a29, fp29_from_mont(b.x), fp29_from_mont(b.y));
            const Xyzz<fq_t> got = xyzz29_to(a29);
            expect(got.X == a32.X && got.Y == a32.Y && got.ZZ == a32.ZZ && got.ZZZ == a32.ZZZ, "madd chain",
                   c * len + e);
        }
    }
}

// Full additions: sums of random partial sums (each a chain of mixed
// additions, so ZZ != 1), including a + a (doubling), a + (-a) (infinity)
// and infinity operands, against xyzz_add after every step.
static void check_add(int chains, int len)
{
    Affine<fq_t> g;
    g.x = fq_t::zero();
    g.x.l[0] = 1;
    g.x = fp_to_mont(g.x);
    g.y = fq_t::zero();
    g.y.l[0] = 2;
    g.y = fp_to_mont(g.y);
    std::vector<Affine<fq_t>> pool;
    for (int i = 0; i < 16; ++i) pool.push_back(random_base(g));
    auto partial = [&](int n, Xyzz<fq_t> &c32, Xyzz29<FqParams> &c29) {
        c32 = Xyzz<fq_t>::infinity();
        c29 = Xyzz29<FqParams>::infinity();
        for (int e = 0; e < n; ++e) {
            const Affine<fq_t> b = pool[rnd() % pool.size()];
            c32 = xyzz_add_affine(c32, b.x, b.y);
            c29 = xyzz29_add_affine(c29, fp29_from_mont(b.x), fp29_from_mont(b.y));
        }
    };
    for (int c = 0; c < chains; ++c) {
        Xyzz<fq_t> a32;
        Xyzz29<FqParams> a29;
        partial(1 + rnd() % 3, a32, a29);
        for (int e = 0; e < len; ++e) {
            const uint32_t r = rnd();
            Xyzz<fq_t> b32;
            Xyzz29<FqParams> b29;
            partial((r >> 4) % 4, b32, b29);  // 0: infinity
            if ((r >> 8) % 6 == 0) {          // a + a
                b32 = a32;
                b29 = a29;
                ++g_doublings;
            } else if ((r >> 12) % 7 == 0 && !a32.is_inf()) {  // a + (-a)
                b32 = a32;
                b32.Y = fp_neg(b32.Y);
                b29 = a29;
                b29.Y = fp29_sub<FqParams, 8>(Fp29<FqParams>::zero(), a29.Y);
                ++g_cancels;
            }
            a32 = xyzz_add(a32, b32);
            a29 = xyzz29_add(a29, b29);
            const Xyzz<fq_t> got = xyzz29_to(a29);
            const Affine<fq_t> w = xyzz_to_affine(a32), h = xyzz_to_affine(got);
            expect(got.is_inf() == a32.is_inf() && (a32.is_inf() || (w.x == h.x && w.y == h.y)), "add chain",
                   c * len + e);
            expect(got.X == a32.X && got.Y == a32.Y && got.ZZ == a32.ZZ && got.ZZZ == a32.ZZZ, "add chain coords",
                   c * len + e);
            if (a32.is_inf()) partial(1, a32, a29);
        }
    }
}

static fq2_t rand_fq2() { return {rand_fp<FqParams>(), rand_fp<FqParams>()}; }

// a + K*p per component (values below (K + 2) p)
template <uint32_t K>
static Fq2_29<FqParams> widen2(const fq2_t &a)
{
    return {widen<FqParams, K>(a.c0), widen<FqParams, K>(a.c1)};
}

static void check_fq2(int n)
{
    for (int i = 0; i < n; ++i) {
        const fq2_t a = rand_fq2(), b = rand_fq2();
        const fq2_t want = fq2_mul(a, b);
        // the products' input bounds in the G2 addition: 32p x 2p (U2, S2),
        // 8p x 2p (Q), 6p x 2p (PPP), 2p x 2p (ZZ3, ZZZ3)
        expect(fq2_29_to(fq2_29_mul<FqParams, 2>(widen2<30>(a), widen2<0>(b))) == want, "fq2 mul 32p x 2p", i);
        expect(fq2_29_to(fq2_29_mul<FqParams, 2>(widen2<6>(a), widen2<0>(b))) == want, "fq2 mul 8p x 2p", i);
        expect(fq2_29_to(fq2_29_mul<FqParams, 2>(widen2<0>(a), widen2<0>(b))) == want, "fq2 mul 2p x 2p", i);
        expect(fq2_29_to(fq2_29_sqr<FqParams, 6>(widen2<4>(a))) == fq2_sqr(a), "fq2 sqr 6p", i);
        {
            // Y3's shape: R (6p) T (9.2p, as 10p) + Y (2p) N (2p), per component
            const fq2_t c = rand_fq2(), d = rand_fq2();
            const Fq2_29<FqParams> R = widen2<4>(a), T = widen2<8>(b), Y = widen2<0>(c), N = widen2<0>(d);
            const Fp29<FqParams> nT1 = fp29_sub<FqParams, 10>(Fp29<FqParams>::zero(), T.c1);
            const Fp29<FqParams> nN1 = fp29_sub<FqParams, 2>(Fp29<FqParams>::zero(), N.c1);
            const Fq2_29<FqParams> y = {fp29_mul_add4(R.c0, T.c0, R.c1, nT1, Y.c0, N.c0, Y.c1, nN1),
                                        fp29_mul_add4(R.c0, T.c1, R.c1, T.c0, Y.c0, N.c1, Y.c1, N.c0)};
            expect(fq2_29_to(y) == fq2_add(fq2_mul(a, b), fq2_mul(c, d)), "fq2 four-product sum", i);
            bool limbs = true;
            for (int k = 0; k < 9; ++k) limbs = limbs && (y.c0.l[k] >> 29) == 0 && (y.c1.l[k] >> 29) == 0;
            expect(limbs, "fq2 four-product limbs", i);
        }
        const Fq2_29<FqParams> m = fq2_29_mul<FqParams, 2>(widen2<30>(a), widen2<0>(b));
        bool limbs = true;
        for (int k = 0; k < 9; ++k) limbs = limbs && (m.c0.l[k] >> 29) == 0 && (m.c1.l[k] >> 29) == 0;
        expect(limbs, "fq2 product limbs", i);
        expect(fq2_29_to(fq2_29_from<FqParams>(a)) == a, "fq2 round trip", i);
    }
}

static void check_madd_g2(int chains, int len)
{
    std::vector<Affine<fq2_t>> pool;
    for (int i = 0; i < 24; ++i) pool.push_back({rand_fq2(), rand_fq2()});
    for (int c = 0; c < chains; ++c) {
        Xyzz<fq2_t> a32 = Xyzz<fq2_t>::infinity();
        Xyzz2_29<FqParams> a29 = Xyzz2_29<FqParams>::infinity();
        for (int e = 0; e < len; ++e) {
            const uint32_t r = rnd();
            Affine<fq2_t> b = pool[r % pool.size()];
            if ((r >> 8) % 5 == 0 && !a32.is_inf()) {
                b = xyzz_to_affine(a32);
                ++g_doublings;
            }
            if ((r >> 12) % 7 == 0) b.y = fq2_neg(b.y);
            if ((r >> 16) % 11 == 0 && !a32.is_inf()) {
                b = xyzz_to_affine(a32);
                b.y = fq2_neg(b.y);
                ++g_cancels;
            }
            a32 = xyzz_add_affine(a32, b.x, b.y);
            a29 = xyzz2_29_add_affine(a29, fq2_29_from<FqParams>(b.x), fq2_29_from<FqParams>(b.y));
            const Xyzz<fq2_t> got = xyzz2_29_to(a29);
            expect(got.X == a32.X && got.Y == a32.Y && got.ZZ == a32.ZZ && got.ZZZ == a32.ZZZ, "g2 madd chain",
                   c * len + e);
        }
    }
}

// Full G2 additions over partial sums, as check_add.
static void check_add_g2(int chains, int len)
{
    std::vector<Affine<fq2_t>> pool;
    for (int i = 0; i < 16; ++i) pool.push_back({rand_fq2(), rand_fq2()});
    auto partial = [&](int n, Xyzz<fq2_t> &c32, Xyzz2_29<FqParams> &c29) {
        c32 = Xyzz<fq2_t>::infinity();
        c29 = Xyzz2_29<FqParams>::infinity();
        for (int e = 0; e < n; ++e) {
            const Affine<fq2_t> b = pool[rnd() % pool.size()];
            c32 = xyzz_add_affine(c32, b.x, b.y);
            c29 = xyzz2_29_add_affine(c29, fq2_29_from<FqParams>(b.x), fq2_29_from<FqParams>(b.y));
        }
    };
    for (int c = 0; c < chains; ++c) {
        Xyzz<fq2_t> a32;
        Xyzz2_29<FqParams> a29;
        partial(1 + rnd() % 3, a32, a29);
        for (int e = 0; e < len; ++e) {
            const uint32_t r = rnd();
            Xyzz<fq2_t> b32;
            Xyzz2_29<FqParams> b29;
            partial((r >> 4) % 4, b32, b29);
            if ((r >> 8) % 6 == 0) {
                b32 = a32;
                b29 = a29;
                ++g_doublings;
            } else if ((r >> 12) % 7 == 0 && !a32.is_inf()) {
                b32 = a32;
                b32.Y = fq2_neg(b32.Y);
                b29 = a29;
                b29.Y = fq2_29_sub<FqParams, 2>({Fp29<FqParams>::zero(), Fp29<FqParams>::zero()}, a29.Y);
                ++g_cancels;
            }
            a32 = xyzz_add(a32, b32);
            a29 = xyzz2_29_add(a29, b29);
            const Xyzz<fq2_t> got = xyzz2_29_to(a29);
            expect(got.X == a32.X && got.Y == a32.Y && got.ZZ == a32.ZZ && got.ZZZ == a32.ZZZ, "g2 add chain",
                   c * len + e);
            if (a32.is_inf()) partial(1, a32, a29);
        }
    }
}

int main()
{
    check_field<FqParams>(20000);
    check_field<FrParams>(20000);
    check_bounds<FqParams>(4000);
    check_bounds<FrParams>(4000);
    check_fq2_bounds(4000);
    check_ntt29(4000);
    check_mul_r29<FqParams>(4000);
    check_mul_r29<FrParams>(4000);
    check_madd(200, 80);
    check_add(150, 60);
    check_fq2(5000);
    check_madd_g2(60, 60);
    check_add_g2(60, 40);
    if (g_bad) {
        std::printf("FAILED %d of %ld checks\n", g_bad, g_checks);
        return 1;
    }
    std::printf("ok %ld checks (%ld doublings, %ld cancellations)\n", g_checks, g_doublings, g_cancels);
    return 0;
}
