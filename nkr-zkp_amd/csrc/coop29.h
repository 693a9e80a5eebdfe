// Point additions shared by a group of lanes, for the bucket reduction (fold,
// completion, bit-plane tree) on gfx950 (device code only).
//
// After the accumulation an MSM has few additions in flight and long chains
// of them, so what bounds it is the time of one addition.  A lane alone does
// the 14 products of a full XYZZ addition one after the other (about 6 us at
// G1, 16 us at G2; one wave per SIMD already issues at 85 % of the SIMD's
// rate).  Here each lane of the group holds one coordinate component of the
// point (G1: X, Y, ZZ, ZZZ in 4 lanes; G2: twice that in 8), and the products
// run in four rounds, one product of every lane per round:
//   1. U1 = X1 ZZ2, S1 = Y1 ZZZ2, U2 = ZZ1 X2, S2 = ZZZ1 Y2
//   2. PP = P^2, RR = R^2, ZZ1 ZZ2, ZZZ1 ZZZ2     (P = U2 - U1, R = S2 - S1)
//   3. Q = U1 PP, PPP = P PP, ZZ3 = (ZZ1 ZZ2) PP
//   4. R (Q - X3), S1 PPP, ZZZ3 = (ZZZ1 ZZZ2) PPP (X3 = RR - PPP - 2Q)
// Operands move between lanes with DPP moves (quad permutes, and for the
// 8-lane group the half-row mirror).  2.5 us at G1 and 3.8 us at G2 per
// addition, measured on MI355X.
//
// Bounds (p the modulus), closed under the addition and satisfied by the
// accumulators of curve29.h: X, Y below 8p at G1; X below 8p, Y below 4p at
// G2; ZZ, ZZZ below 2p; infinity is ZZ = 0 exactly.
//
// Every call must be reached by whole groups (a group's lanes are adjacent
// and aligned), since a DPP move reads its neighbours' registers.
#pragma once

#include "curve29.h"

namespace nkr {

template <int Ctrl, int Banks = 0xf>
__device__ __forceinline__ uint32_t dpp_mov(uint32_t old, uint32_t x)
{
    return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)x, Ctrl, 0xf, Banks, false);
}

constexpr int quad_perm(int a, int b, int c, int d) { return a | b << 2 | c << 4 | d << 6; }
constexpr int kHalfMirror = 0x141;  // lane i of each 8 reads lane 7 - i
constexpr int kLowQuads = 0x5, kHighQuads = 0xa;

template <int Ctrl, class P>
__device__ __forceinline__ Fp29<P> fp29_dpp(const Fp29<P> &x)
{
    Fp29<P> r;
#pragma unroll
    for (int i = 0; i < 9; ++i) r.l[i] = dpp_mov<Ctrl>(x.l[i], x.l[i]);
    return r;
}

// Low quads read `lo` through quad_perm CLo, high quads `hi` through CHi.
template <int CLo, int CHi, class P>
__device__ __forceinline__ Fp29<P> fp29_dpp2(const Fp29<P> &lo, const Fp29<P> &hi)
{
    Fp29<P> r;
#pragma unroll
    for (int i = 0; i < 9; ++i) r.l[i] = dpp_mov<CHi, kHighQuads>(dpp_mov<CLo>(lo.l[i], lo.l[i]), hi.l[i]);
    return r;
}

template <class P>
__device__ __forceinline__ Fp29<P> fp29_select(bool c, const Fp29<P> &a, const Fp29<P> &b)
{
    Fp29<P> r;
#pragma unroll
    for (int i = 0; i < 9; ++i) r.l[i] = c ? a.l[i] : b.l[i];
    return r;
}

template <class P>
__device__ __forceinline__ uint32_t fp29_or(const Fp29<P> &x)
{
    uint32_t v = 0;
#pragma unroll
    for (int i = 0; i < 9; ++i) v |= x.l[i];
    return v;
}

// Coop<F>: one lane's view of a point shared by kLanes lanes.  `v` is the
// lane's component, component index kLanes * point + word() of a partial sum
// in memory (Xyzz29 / Xyzz2_29 as arrays of Fp29).
template <class F>
struct Coop;

template <>
struct Coop<fq_t> {
    using P = FqParams;
    static constexpr uint32_t kLanes = 4;
    Fp29<P> v;

    __device__ static uint32_t lane() { return threadIdx.x & 3u; }
    // the component this lane holds: X, Y, ZZ, ZZZ
    __device__ static uint32_t word() { return lane(); }
    __device__ static Coop infinity() { return {Fp29<P>::zero()}; }
    // non-zero on every lane iff the point is not infinity
    __device__ uint32_t finite() const
    {
        const uint32_t z = fp29_or(v);
        return dpp_mov<quad_perm(2, 2, 2, 2)>(z, z);
    }
};

template <>
struct Coop<fq2_t> {
    using P = FqParams;
    static constexpr uint32_t kLanes = 8;
    Fp29<P> v;

    __device__ static uint32_t lane() { return threadIdx.x & 7u; }
    // X0 X1 Y0 Y1 | ZZZ1 ZZZ0 ZZ1 ZZ0: the mirror swaps X with ZZ and Y with
    // ZZZ, and a component's sibling is the neighbouring lane
    __device__ static uint32_t word() { return lane() < 4 ? lane() : 11u - lane(); }
    __device__ static bool second() { return word() & 1u; }  // holds a c1
    __device__ static Coop infinity() { return {Fp29<P>::zero()}; }
    __device__ uint32_t finite() const
    {
        uint32_t z = fp29_or(v);
        z |= dpp_mov<quad_perm(1, 0, 3, 2)>(z, z);
        const uint32_t m = dpp_mov<kHalfMirror>(z, z);
        return dpp_mov<quad_perm(3, 3, 3, 3), kHighQuads>(dpp_mov<quad_perm(0, 0, 0, 0)>(m, m), z);
    }
};

// x * y over Fq2 with each operand's components on neighbouring lanes:
// c0 = x0 y0 + x1 (10p - y1), c1 = x0 y1 + x1 y0.  x below A p, y below B p,
// B <= 10, A (B + 10) at most 145: below 2p.
__device__ __forceinline__ Fp29<FqParams> coop_fq2_mul(const Fp29<FqParams> &x, const Fp29<FqParams> &y, bool c1)
{
    using P = FqParams;
    const Fp29<P> xo = fp29_dpp<quad_perm(1, 0, 3, 2)>(x), yo = fp29_dpp<quad_perm(1, 0, 3, 2)>(y);
    const Fp29<P> ny = fp29_sub<P, 10>(Fp29<P>::zero(), yo);
    return fp29_mul_add(x, fp29_select(c1, yo, y), xo, fp29_select(c1, y, ny));
}

// 2a for a finite a (dbl-2008-s-1: V = 4Y^2, M = 3X^2, S = X V, W = 2Y V),
// the addition's case P = R = 0.  Bounds as the addition's.
__device__ __forceinline__ Fp29<FqParams> coop_double(const Coop<fq_t> &a)
{
    using P = FqParams;
    const uint32_t q = Coop<fq_t>::lane();
    const Fp29<P> r1 = fp29_mul(a.v, a.v);  // X^2 Y^2 - - (8p x 8p)
    const Fp29<P> x2 = fp29_dpp<quad_perm(0, 0, 0, 0)>(r1), y2 = fp29_dpp<quad_perm(1, 1, 1, 1)>(r1);
    const Fp29<P> M = fp29_add(fp29_add(x2, x2), x2);              // below 6p
    const Fp29<P> yy = fp29_add(y2, y2), V = fp29_add(yy, yy);     // below 8p
    // S, Y V, ZZ3, M^2
    const Fp29<P> r2 = fp29_mul(fp29_select(q == 3, M, a.v), fp29_select(q == 3, M, V));
    const Fp29<P> S = fp29_dpp<quad_perm(0, 0, 0, 0)>(r2), h = fp29_dpp<quad_perm(1, 1, 1, 1)>(r2);
    const Fp29<P> W = fp29_add(h, h);                                                       // below 4p
    const Fp29<P> X3 = fp29_sub<P, 4>(fp29_dpp<quad_perm(3, 3, 3, 3)>(r2), fp29_add(S, S));  // below 6p
    // M (S - X3), -W Y, -, ZZZ3
    const Fp29<P> T = fp29_sub<P, 6>(S, X3), N = fp29_sub<P, 4>(Fp29<P>::zero(), W);
    const Fp29<P> r3 =
        fp29_mul(fp29_select(q == 0, M, a.v), fp29_select(q == 0, T, fp29_select(q == 1, N, W)));
    const Fp29<P> Y3 = fp29_add(r3, fp29_dpp<quad_perm(0, 0, 2, 3)>(r3));
    return fp29_select(q < 2, fp29_select(q == 0, X3, Y3), fp29_select(q == 2, r2, r3));
}
__device__ __forceinline__ Fp29<FqParams> coop_double(const Coop<fq2_t> &a)
{
    using P = FqParams;
    const uint32_t q = Coop<fq2_t>::lane();
    const bool c1 = Coop<fq2_t>::second();
    const bool low = q < 4, onX = q < 2, onZZZ = q == 4 || q == 5;
    const Fp29<P> r1 = coop_fq2_mul(a.v, a.v, c1);  // X^2 Y^2 | - - (8p x 8p)
    const Fp29<P> m1 = fp29_dpp<kHalfMirror>(r1);
    const Fp29<P> x2 = fp29_dpp2<quad_perm(0, 1, 0, 1), quad_perm(2, 3, 2, 3)>(r1, m1);
    const Fp29<P> y2 = fp29_dpp2<quad_perm(2, 3, 2, 3), quad_perm(0, 1, 0, 1)>(r1, m1);
    const Fp29<P> M = fp29_add(fp29_add(x2, x2), x2);           // below 6p
    const Fp29<P> yy = fp29_add(y2, y2), V = fp29_add(yy, yy);  // below 8p
    // S, Y V | M^2, ZZ3
    const Fp29<P> r2 = coop_fq2_mul(fp29_select(onZZZ, M, a.v), fp29_select(onZZZ, M, V), c1);
    const Fp29<P> MM = fp29_dpp<quad_perm(2, 3, 2, 3)>(fp29_dpp<kHalfMirror>(r2));  // X lanes
    const Fp29<P> X3 = fp29_sub<P, 4>(MM, fp29_add(r2, r2));                         // X lanes: below 6p
    const Fp29<P> W = fp29_add(r2, r2);                                             // Y lanes: below 4p
    // M (S - X3), -W Y | ZZZ3, -
    const Fp29<P> x3 = fp29_select(onX, M, fp29_select(low, fp29_sub<P, 4>(Fp29<P>::zero(), W), a.v));
    const Fp29<P> y3 =
        fp29_select(onX, fp29_sub<P, 6>(r2, X3), fp29_select(low, a.v, fp29_dpp<kHalfMirror>(W)));
    const Fp29<P> r3 = coop_fq2_mul(x3, y3, c1);
    const Fp29<P> Y3 = fp29_add(r3, fp29_dpp<quad_perm(0, 1, 0, 1)>(r3));
    return fp29_select(low, fp29_select(onX, X3, Y3), fp29_select(onZZZ, r3, r2));
}

// a + b, complete (add-2008-s), G1: lanes X, Y, ZZ, ZZZ.
__device__ __forceinline__ Coop<fq_t> coop_add(const Coop<fq_t> &a, const Coop<fq_t> &b)
{
    using P = FqParams;
    const uint32_t q = Coop<fq_t>::lane();
    const bool low = q < 2;
    const uint32_t fa = a.finite(), fb = b.finite();
    // U1 S1 U2 S2, below 2p (8p x 2p)
    const Fp29<P> r1 = fp29_mul(a.v, fp29_dpp<quad_perm(2, 3, 0, 1)>(b.v));
    // -P -R P R, below 4p
    const Fp29<P> d = fp29_sub<P, 2>(r1, fp29_dpp<quad_perm(2, 3, 0, 1)>(r1));
    // PP RR ZZ1ZZ2 ZZZ1ZZZ2 (4p x 4p)
    const Fp29<P> r2 = fp29_mul(fp29_select(low, d, a.v), fp29_select(low, d, b.v));
    // Q - ZZ3 PPP
    const Fp29<P> pd = fp29_dpp<quad_perm(0, 1, 2, 2)>(d);
    const Fp29<P> r3 =
        fp29_mul(fp29_select(q == 0, r1, fp29_select(q == 3, pd, r2)), fp29_dpp<quad_perm(0, 0, 0, 0)>(r2));
    const Fp29<P> Q = fp29_dpp<quad_perm(0, 0, 0, 0)>(r3);
    const Fp29<P> PPP = fp29_dpp<quad_perm(3, 3, 3, 3)>(r3);
    const Fp29<P> RR = fp29_dpp<quad_perm(1, 1, 1, 1)>(r2);
    const Fp29<P> X3 = fp29_sub<P, 4>(fp29_sub<P, 2>(RR, PPP), fp29_add(Q, Q));  // below 8p
    const Fp29<P> T = fp29_sub<P, 8>(Q, X3);                                     // below 10p
    const Fp29<P> N = fp29_sub<P, 2>(Fp29<P>::zero(), PPP);
    // RT S1N - ZZZ3 (4p x 10p)
    const Fp29<P> R = fp29_dpp<quad_perm(3, 1, 2, 3)>(d);
    const Fp29<P> r4 = fp29_mul(fp29_select(q == 0, R, fp29_select(q == 1, r1, r2)),
                                fp29_select(q == 0, T, fp29_select(q == 1, N, PPP)));
    const Fp29<P> Y3 = fp29_add(r4, fp29_dpp<quad_perm(0, 0, 2, 3)>(r4));  // below 4p
    Fp29<P> s = fp29_select(low, fp29_select(q == 0, X3, Y3), fp29_select(q == 2, r3, r4));
    if (__any(q == 0 && fa && fb && fp29_may_be_zero<P, 4>(d))) {
        // b = +-a in some group of the wave: doubling, or infinity
        const uint32_t z = fp29_to_mont(d).is_zero() ? 1u : 0u;
        const bool same_x = dpp_mov<quad_perm(0, 0, 0, 0)>(z, z), same_y = dpp_mov<quad_perm(1, 1, 1, 1)>(z, z);
        const Fp29<P> dbl = coop_double(a);
        s = fp29_select(same_x, fp29_select(same_y, dbl, Fp29<P>::zero()), s);
    }
    return {fp29_select(!fa, b.v, fp29_select(!fb, a.v, s))};
}

// a + b, complete, G2: lanes X0 X1 Y0 Y1 ZZZ1 ZZZ0 ZZ1 ZZ0.
__device__ __forceinline__ Coop<fq2_t> coop_add(const Coop<fq2_t> &a, const Coop<fq2_t> &b)
{
    using P = FqParams;
    const uint32_t q = Coop<fq2_t>::lane();
    const bool low = q < 4, c1 = Coop<fq2_t>::second();
    const bool onX = q < 2, onZZZ = q == 4 || q == 5;
    const uint32_t fa = a.finite(), fb = b.finite();
    // U1 S1 | S2 U2 (8p, 4p x 2p; 2p x 8p)
    const Fp29<P> r1 = coop_fq2_mul(a.v, fp29_dpp<kHalfMirror>(b.v), c1);
    // -P -R | R P, below 4p
    const Fp29<P> d = fp29_sub<P, 2>(r1, fp29_dpp<kHalfMirror>(r1));
    // PP RR | ZZZ1ZZZ2 ZZ1ZZ2 (4p x 4p)
    const Fp29<P> r2 = coop_fq2_mul(fp29_select(low, d, a.v), fp29_select(low, d, b.v), c1);
    // Q - | PPP ZZ3: PP to every lane; P from the ZZ lanes to the ZZZ lanes
    const Fp29<P> pp =
        fp29_dpp2<quad_perm(0, 1, 0, 1), quad_perm(2, 3, 2, 3)>(r2, fp29_dpp<kHalfMirror>(r2));
    const Fp29<P> pd = fp29_dpp<quad_perm(2, 3, 2, 3)>(d);
    const Fp29<P> r3 = coop_fq2_mul(fp29_select(onX, r1, fp29_select(onZZZ, pd, r2)), pp, c1);
    // on the Y lanes m3 is PPP, and from there it goes to the X lanes
    const Fp29<P> m3 = fp29_dpp<kHalfMirror>(r3);
    const Fp29<P> PPP = fp29_dpp<quad_perm(2, 3, 2, 3)>(m3);
    const Fp29<P> RR = fp29_dpp<quad_perm(2, 3, 2, 3)>(r2);
    const Fp29<P> X3 = fp29_sub<P, 4>(fp29_sub<P, 2>(RR, PPP), fp29_add(r3, r3));  // X lanes: below 8p
    const Fp29<P> T = fp29_sub<P, 2>(X3, r3);                                     // X3 - Q, below 10p
    const Fp29<P> N = fp29_sub<P, 2>(Fp29<P>::zero(), m3);                         // Y lanes: -PPP
    const Fp29<P> R = fp29_dpp<quad_perm(2, 3, 2, 3)>(d);                          // X lanes: -R
    // RT S1N | ZZZ3 - (4p x 10p)
    const Fp29<P> r4 = coop_fq2_mul(fp29_select(onX, R, fp29_select(low, r1, r2)),
                                    fp29_select(onX, T, fp29_select(low, N, r3)), c1);
    const Fp29<P> Y3 = fp29_add(r4, fp29_dpp<quad_perm(0, 1, 0, 1)>(r4));  // Y lanes: below 4p
    Fp29<P> s = fp29_select(low, fp29_select(onX, X3, Y3), fp29_select(onZZZ, r4, r3));
    uint32_t z = fp29_may_be_zero<P, 4>(d) ? 1u : 0u;
    z &= dpp_mov<quad_perm(1, 0, 3, 2)>(z, z);
    if (__any(q == 0 && fa && fb && z)) {
        // b = +-a in some group of the wave: doubling, or infinity
        z = fp29_to_mont(d).is_zero() ? 1u : 0u;
        z &= dpp_mov<quad_perm(1, 0, 3, 2)>(z, z);
        const bool same_x = dpp_mov<quad_perm(3, 3, 3, 3), kHighQuads>(dpp_mov<quad_perm(0, 0, 0, 0)>(z, z), z);
        const bool same_y = dpp_mov<quad_perm(0, 0, 0, 0), kHighQuads>(dpp_mov<quad_perm(2, 2, 2, 2)>(z, z), z);
        const Fp29<P> dbl = coop_double(a);
        s = fp29_select(same_x, fp29_select(same_y, dbl, Fp29<P>::zero()), s);
    }
    return {fp29_select(!fa, b.v, fp29_select(!fb, a.v, s))};
}

// The point of the group `groups` groups away (XOR) in the wave.
template <class F>
__device__ __forceinline__ Coop<F> coop_shfl_xor(const Coop<F> &a, uint32_t groups)
{
    Coop<F> r;
#pragma unroll
    for (int i = 0; i < 9; ++i)
        r.v.l[i] = (uint32_t)__shfl_xor((int)a.v.l[i], (int)(groups * Coop<F>::kLanes), 64);
    return r;
}

// Component of partial sum i of an array of partial sums.
template <class F, class T>
__device__ __forceinline__ Coop<F> coop_load(const T *base, size_t i)
{
    static_assert(sizeof(T) == Coop<F>::kLanes * sizeof(Fp29<FqParams>), "partial sum layout");
    return {reinterpret_cast<const Fp29<FqParams> *>(base)[i * Coop<F>::kLanes + Coop<F>::word()]};
}
template <class F, class T>
__device__ __forceinline__ void coop_store(T *base, size_t i, const Coop<F> &a)
{
    static_assert(sizeof(T) == Coop<F>::kLanes * sizeof(Fp29<FqParams>), "partial sum layout");
    reinterpret_cast<Fp29<FqParams> *>(base)[i * Coop<F>::kLanes + Coop<F>::word()] = a.v;
}
// The point as canonical XYZZ coordinates (infinity: all zero).
template <class F>
__device__ __forceinline__ void coop_store_plane(Xyzz<F> *plane, const Coop<F> &a)
{
    static_assert(sizeof(Xyzz<F>) == Coop<F>::kLanes * sizeof(fq_t), "XYZZ layout");
    const fq_t c = a.finite() ? fp29_to_mont(a.v) : fq_t::zero();
    reinterpret_cast<fq_t *>(plane)[Coop<F>::word()] = c;
}

}  // namespace nkr
