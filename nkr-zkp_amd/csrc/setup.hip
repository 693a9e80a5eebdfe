// Fixed-base batch scalar multiplication on the GPU: out_i = k_i * P for one
// base P.  This is the building block of Groth16 key generation (the
// reference's FixedBaseMsm, operators/include/nkr/operators/fixed_base_msm.hpp:
// 14-39, and its HIP fixmsm_kernel, operators/hip/include/msm/fixmsm_kernel.hip:
// 6-20) and produces the synthetic proving-key vectors (k_i * G) the
// benchmarks and tests use.
//
// A table T[j][d] = d * 2^(8j) * P (32 windows of 8 bits, affine) is built
// once; a scalar then needs 32 mixed additions and an inversion (shared by the
// workgroup) to emit a normalised point (Z = 1, or (0, 1, 0) for k = 0).
#include "setup.h"

#include "block_inverse.h"
#include "curve29.h"

namespace nkr {

namespace {

constexpr uint32_t kFixedThreads = 256;

// The reduced-radix accumulator of each group (curve29.h).
template <class F>
struct Acc29;
template <>
struct Acc29<fq_t> {
    using type = Xyzz29<FqParams>;
    __device__ static void add(type &a, const Affine<fq_t> &b)
    {
        a = xyzz29_add_affine(a, fp29_from_mont(b.x), fp29_from_mont(b.y));
    }
    __device__ static void add(type &a, const type &b) { a = xyzz29_add(a, b); }
    __device__ static Xyzz<fq_t> to(const type &a) { return xyzz29_to(a); }
};
template <>
struct Acc29<fq2_t> {
    using type = Xyzz2_29<FqParams>;
    __device__ static void add(type &a, const Affine<fq2_t> &b)
    {
        a = xyzz2_29_add_affine(a, fq2_29_from<FqParams>(b.x), fq2_29_from<FqParams>(b.y));
    }
    __device__ static void add(type &a, const type &b) { a = xyzz2_29_add(a, b); }
    __device__ static Xyzz<fq2_t> to(const type &a) { return xyzz2_29_to(a); }
};

// T[j*256 + d] = d * 2^(8j) * P, affine (infinity flagged for d = 0), from the
// powers pow2[i] = 2^i P: workgroup j, thread d, up to 8 additions and one
// inversion for all.  (Doubling up from P in every thread, with an inversion
// each, took 3.4 ms at G1 and 10.6 ms at G2; 0.22 and 0.31 ms now.)
template <class F>
__global__ __launch_bounds__(kFixedThreads) void k_fixed_table(const Affine<F> *__restrict__ pow2,
                                                               Affine<F> *__restrict__ table)
{
    __shared__ fq_t node[2 * kFixedThreads];
    const uint32_t j = blockIdx.x, d = threadIdx.x;
    typename Acc29<F>::type acc = Acc29<F>::type::infinity();
#pragma unroll 1
    for (uint32_t b = 0; b < 8; ++b) {
        const Affine<F> p = pow2[8 * j + b];
        if (((d >> b) & 1u) && !affine_is_inf(p)) Acc29<F>::add(acc, p);
    }
    table[j * 256 + d] = block_to_affine<kFixedThreads>(Acc29<F>::to(acc), node);
}

// out[i] = scalars[i] * P.  `split` threads (1, 2, 4 or 8 neighbours) share a
// scalar's windows and add their sums, so that few scalars do not wait for 32
// additions in a row; the additions stay in the reduced-radix form.
template <class F>
__global__ __launch_bounds__(kFixedThreads) void k_fixed_mul(const Affine<F> *__restrict__ table,
                                                             const fr_t *__restrict__ scalars, uint64_t n,
                                                             uint32_t split, Jacobian<F> *__restrict__ out)
{
    __shared__ fq_t node[2 * kFixedThreads];
    const uint64_t g = blockIdx.x * (uint64_t)kFixedThreads + threadIdx.x;
    const uint64_t i = g / split;
    const uint32_t part = (uint32_t)g & (split - 1);
    const fr_t k = i < n ? fp_from_mont(scalars[i]) : fr_t::zero();
    typename Acc29<F>::type acc = Acc29<F>::type::infinity();
#pragma unroll 1
    for (uint32_t j = part; j < 32; j += split) {
        uint32_t word = 0;
#pragma unroll
        for (uint32_t w = 0; w < 8; ++w) word = (j >> 2) == w ? k.l[w] : word;
        const uint32_t d = (word >> ((j & 3u) * 8)) & 255u;
        const Affine<F> t = table[j * 256 + d];
        if (d != 0 && !affine_is_inf(t)) Acc29<F>::add(acc, t);
    }
#pragma unroll 1
    for (uint32_t off = 1; off < split; off <<= 1) {
        typename Acc29<F>::type o;
        const uint32_t *src = reinterpret_cast<const uint32_t *>(&acc);
        uint32_t *dst = reinterpret_cast<uint32_t *>(&o);
#pragma unroll
        for (uint32_t w = 0; w < sizeof(o) / 4; ++w) dst[w] = (uint32_t)__shfl_xor((int)src[w], (int)off);
        Acc29<F>::add(acc, o);
    }
    const Xyzz<F> p = Acc29<F>::to(acc);
    const Affine<F> a = block_to_affine<kFixedThreads>(part == 0 ? p : Xyzz<F>::infinity(), node);
    if (i >= n || part != 0) return;
    using O = FieldOps<F>;
    out[i] = p.is_inf() ? Jacobian<F>{O::zero(), O::one(), O::zero()} : Jacobian<F>{a.x, a.y, O::one()};
}

}  // namespace

template <class F>
FixedBaseMul<F>::FixedBaseMul(const Jacobian<F> &base, hipStream_t stream)
{
    // 2^i P for i < 256 on the host (a chain of doublings, which a GPU lane
    // takes ten times as long for), normalised with one inversion
    using O = FieldOps<F>;
    constexpr int n = 256;
    std::vector<Xyzz<F>> p(n);
    std::vector<F> prefix(n);
    p[0] = jacobian_to_xyzz(base);
    for (int i = 1; i < n; ++i) p[i] = xyzz_dbl(p[i - 1]);
    F acc = O::one();
    for (int i = 0; i < n; ++i) {
        prefix[i] = acc;
        if (!p[i].is_inf()) acc = O::mul(acc, O::mul(p[i].ZZ, p[i].ZZZ));
    }
    F inv = O::inv(acc);
    pow2_host_.resize(n);
    for (int i = n - 1; i >= 0; --i) {
        if (p[i].is_inf()) {
            pow2_host_[i] = affine_infinity<F>();
            continue;
        }
        const F t = O::mul(inv, prefix[i]);
        inv = O::mul(inv, O::mul(p[i].ZZ, p[i].ZZZ));
        pow2_host_[i] = Affine<F>{O::mul(p[i].X, O::mul(t, p[i].ZZZ)), O::mul(p[i].Y, O::mul(t, p[i].ZZ))};
    }
    pow2_.allocate(n);
    table_.allocate(32 * 256);
    NKR_HIP(hipMemcpyAsync(pow2_.get(), pow2_host_.data(), n * sizeof(Affine<F>), hipMemcpyHostToDevice, stream));
    k_fixed_table<F><<<32, kFixedThreads, 0, stream>>>(pow2_.get(), table_.get());
    NKR_LAUNCH_CHECK();
}

template <class F>
void FixedBaseMul<F>::run(const fr_t *scalars_dev, uint64_t n, Jacobian<F> *out_dev, hipStream_t stream) const
{
    if (n == 0) return;
    // threads per scalar: as many as keep the launch within one wave per SIMD
    // (up to 4 at G1 and 8 at G2, where joining two sums costs half of what
    // halving the windows saves)
    uint32_t split = 1;
    while (split < (std::is_same<F, fq2_t>::value ? 8u : 4u) && n * split * 2 <= 65536) split *= 2;
    k_fixed_mul<F><<<(uint32_t)((n * split + kFixedThreads - 1) / kFixedThreads), kFixedThreads, 0, stream>>>(
        table_.get(), scalars_dev, n, split, out_dev);
    NKR_LAUNCH_CHECK();
}

template <class F>
Xyzz<F> FixedBaseMul<F>::mul_host(const fr_t &k_mont) const
{
    const fr_t k = fp_from_mont(k_mont);
    Xyzz<F> acc = Xyzz<F>::infinity();
    for (int i = 0; i < 256; ++i)
        if (((k.l[i >> 5] >> (i & 31)) & 1u) && !affine_is_inf(pow2_host_[i]))
            acc = xyzz_add_affine(acc, pow2_host_[i].x, pow2_host_[i].y);
    return acc;
}

template <class F>
std::vector<Affine<F>> FixedBaseMul<F>::table_host(hipStream_t stream) const
{
    std::vector<Affine<F>> t(32 * 256);
    NKR_HIP(hipMemcpyAsync(t.data(), table_.get(), t.size() * sizeof(Affine<F>), hipMemcpyDeviceToHost, stream));
    NKR_HIP(hipStreamSynchronize(stream));
    return t;
}

// Host: k * base from a comb table (32 mixed additions, no doublings).
template <class F>
Xyzz<F> fixed_base_mul_host(const std::vector<Affine<F>> &table, const fr_t &k_mont)
{
    const fr_t k = fp_from_mont(k_mont);
    Xyzz<F> acc = Xyzz<F>::infinity();
    for (uint32_t j = 0; j < 32; ++j) {
        const uint32_t d = (k.l[j >> 2] >> ((j & 3u) * 8)) & 255u;
        if (d == 0) continue;
        const Affine<F> &t = table[j * 256 + d];
        if (affine_is_inf(t)) continue;
        acc = xyzz_add_affine(acc, t.x, t.y);
    }
    return acc;
}

template Xyzz<fq_t> fixed_base_mul_host(const std::vector<Affine<fq_t>> &, const fr_t &);
template Xyzz<fq2_t> fixed_base_mul_host(const std::vector<Affine<fq2_t>> &, const fr_t &);

template class FixedBaseMul<fq_t>;
template class FixedBaseMul<fq2_t>;

}  // namespace nkr
