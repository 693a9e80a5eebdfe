// One field inversion shared by a workgroup (device code only).
//
// An inversion by Fermat is about 350 dependent products, 140 us on MI355X
// whatever the number of lanes that do it, against 16 products for a tree over
// 256 lanes: the lanes' values are multiplied pairwise up to the root, the
// root is inverted by one wave, and each node hands its two children their
// inverses (Montgomery's simultaneous inversion as a tree).
#pragma once

#include "curve.h"
#include "field29.h"

namespace nkr {

// x^(p-2), 0 for 0: square and multiply by two bits of the exponent, in the
// 29-bit form throughout.
template <class P>
__device__ Fp<P> fp_inv_fermat29(const Fp<P> &x)
{
    Fp29<P> x1 = fp29_reduce_to_2p(fp29_from_mont(x)), acc = Fp29<P>::one();
    // a value every lane shares would be computed on the scalar unit, whose
    // products take four instructions where the vector unit's take one
    fp29_opaque(x1);
    fp29_opaque(acc);
    const Fp29<P> x2 = fp29_sqr(x1), x3 = fp29_mul(x2, x1);
#pragma unroll 1
    for (int i = 127; i >= 0; --i) {
        acc = fp29_sqr(fp29_sqr(acc));
        // selects, not an indexed constant: a load per step would be longer
        // than the step's products.  The modulus is odd and its low word above
        // 2, so p - 2 changes no other word.
        uint32_t word = P::P[0] - 2u;
#pragma unroll
        for (int w = 1; w < 8; ++w) word = (i >> 4) == w ? P::P[w] : word;
        const uint32_t d = (word >> ((i & 15) * 2)) & 3u;
        if (d == 0) continue;
        acc = fp29_mul(acc, d == 1 ? x1 : (d == 2 ? x2 : x3));
    }
    return fp29_to_mont(acc);
}

// 1 / x of every lane of a workgroup of N threads (a power of two, 64 or
// more); 0 gives 0.  All threads take part; `node` is LDS of 2 N elements.
template <uint32_t N, class P>
__device__ Fp<P> block_inverse(const Fp<P> &x, Fp<P> *node)
{
    const uint32_t t = threadIdx.x;
    const bool zero = x.is_zero();
    __syncthreads();  // a previous call's reads
    node[N + t] = zero ? Fp<P>::one() : x;
#pragma unroll 1
    for (uint32_t s = N / 2; s >= 1; s >>= 1) {
        __syncthreads();
        if (t < s) node[s + t] = fp_mul(node[2 * (s + t)], node[2 * (s + t) + 1]);
    }
    __syncthreads();
    if (t < 64) {
        const Fp<P> r = fp_inv_fermat29(node[1]);
        if (t == 0) node[1] = r;
    }
#pragma unroll 1
    for (uint32_t s = 1; s < N; s <<= 1) {
        __syncthreads();
        if (t < s) {
            const uint32_t i = s + t;
            const Fp<P> inv = node[i], l = node[2 * i], r = node[2 * i + 1];
            node[2 * i] = fp_mul(inv, r);
            node[2 * i + 1] = fp_mul(inv, l);
        }
    }
    __syncthreads();
    return zero ? Fp<P>::zero() : node[N + t];
}

// Over Fq2: 1 / (a0 + a1 u) = (a0 - a1 u) / (a0^2 + a1^2).
template <uint32_t N>
__device__ fq2_t block_inverse(const fq2_t &x, fq_t *node)
{
    const fq_t n = block_inverse<N>(fp_add(fp_sqr(x.c0), fp_sqr(x.c1)), node);
    return {fp_mul(x.c0, n), fp_neg(fp_mul(x.c1, n))};
}

// The affine points of a workgroup's XYZZ points with one inversion.
template <uint32_t N, class F>
__device__ Affine<F> block_to_affine(const Xyzz<F> &p, fq_t *node)
{
    using O = FieldOps<F>;
    const F t = block_inverse<N>(O::mul(p.ZZ, p.ZZZ), node);
    if (p.is_inf()) return affine_infinity<F>();
    return {O::mul(p.X, O::mul(t, p.ZZZ)), O::mul(p.Y, O::mul(t, p.ZZ))};
}

}  // namespace nkr
