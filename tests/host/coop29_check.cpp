// CPU check of the point additions shared by a group of lanes
// (nkr-zkp_amd/csrc/coop29.h): its device code runs here on a row of 16 lanes,
// each lane a context of its own that is switched at every lane move, and is
// compared with the canonical additions of curve.h.  (The formulas are field
// identities, so coordinates need not lie on the curve.)
//   * operands at the top of what the additions accept (G1: X, Y below 8p; G2: X
//     below 8p, Y below 4p; ZZ, ZZZ below 2p) and anywhere below it, in groups
//     that add, double (equal points in different representations), cancel and
//     pass infinity through, side by side in one row;
//   * every component of a sum has limbs below 2^29, stays below the bounds it
//     has to keep, and is congruent to the canonical sum's.
// Prints "ok <additions> (<doublings>, <cancellations>)", or the first
// mismatches and exit status 1.
#include <ucontext.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <vector>

// ---- 16 lanes in step.  Every lane makes the same lane moves in the same
// order; a move publishes the lane's operand, lets the other lanes come to the
// same move, and reads.  Two sets of slots: a lane may be one move ahead.
constexpr int kRow = 16;
struct LaneIndex {
    uint32_t x;
};
static LaneIndex threadIdx;
static ucontext_t g_lane[kRow], g_main;
static uint32_t g_slot[2][kRow];
static unsigned g_moves[kRow];
static bool g_done[kRow];

static void next_lane()
{
    const uint32_t me = threadIdx.x;
    const uint32_t to = (me + 1) % kRow;
    threadIdx.x = to;
    swapcontext(&g_lane[me], &g_lane[to]);
    threadIdx.x = me;
}
// Publishes v; true slots of all lanes for this move are returned.
static const uint32_t *exchange(uint32_t v)
{
    const uint32_t me = threadIdx.x;
    uint32_t *s = g_slot[g_moves[me]++ & 1];
    s[me] = v;
    next_lane();
    return s;
}
static int emulated_dpp(int old, int src, int ctrl, int row_mask, int bank_mask, bool)
{
    const uint32_t me = threadIdx.x;
    const uint32_t *s = exchange((uint32_t)src);
    if (row_mask != 0xf) std::abort();
    if (!(bank_mask >> (me / 4) & 1)) return old;
    if (ctrl < 0x100) return (int)s[(me & ~3u) | (ctrl >> (2 * (me & 3)) & 3)];  // quad_perm
    if (ctrl == 0x141) return (int)s[(me & ~7u) | (7 - (me & 7))];               // row_half_mirror
    std::abort();
}
static int emulated_any(bool p)
{
    const uint32_t *s = exchange(p);
    int any = 0;
    for (int i = 0; i < kRow; ++i) any |= (int)s[i];
    return any;
}
static int emulated_shfl_xor(int v, int mask, int)
{
    const uint32_t me = threadIdx.x;
    return (int)exchange((uint32_t)v)[me ^ (uint32_t)mask];
}
#define __builtin_amdgcn_update_dpp emulated_dpp
#define __any emulated_any
#define __shfl_xor emulated_shfl_xor
#include "coop29.h"
#undef __any

using namespace nkr;
using P = FqParams;

static uint64_t g_state = 0x243F6A8885A308D3ull;
static uint32_t rnd()
{
    g_state ^= g_state << 13;
    g_state ^= g_state >> 7;
    g_state ^= g_state << 17;
    return (uint32_t)(g_state >> 11);
}
static long g_adds = 0, g_doublings = 0, g_cancels = 0;
static int g_bad = 0;
static void expect(bool ok, const char *what, long at)
{
    if (!ok && g_bad++ < 10) std::printf("mismatch: %s at addition %ld\n", what, at);
}

template <uint32_t K>
static bool is_below(const Fp29<P> &x)
{
    const Fp29<P> y = fp29_sub_if_ge<P, K>(x);
    for (int k = 0; k < 9; ++k)
        if (x.l[k] != y.l[k]) return false;
    return true;
}
// x + k p for a k < K (the largest, or any), x canonical: a value below K p.
template <uint32_t K>
static Fp29<P> represent(const fq_t &x)
{
    const Fp29<P> z = Fp29<P>::zero();
    Fp29<P> v = fp29_sub_if_ge<P, 1>(fp29_reduce_to_2p(fp29_from_mont(x)));
    for (uint32_t k = rnd() % 3 ? K - 1 : rnd() % K; k; --k) v = fp29_sub<P, 1>(v, z);
    return v;
}
// A coordinate: near the modulus in the 29-bit form (K p - 1 - d with a small
// d once represented), or any.
static fq_t coordinate()
{
    fq_t x;
    if (rnd() % 2) {
        Fp29<P> d = Fp29<P>::zero();
        d.l[0] = 1 + rnd() % 4;
        return fp29_to_mont(fp29_sub<P, 1>(Fp29<P>::zero(), d));
    }
    for (int i = 0; i < 8; ++i) x.l[i] = rnd();
    x.l[7] %= P::P[7] + 1;
    return fp_reduce_once(x);
}

// ---- a group's coordinates as the components its lanes hold
struct G1 {
    using F = fq_t;
    static constexpr int kParts = 1;
    static fq_t any() { return coordinate(); }
    static fq_t part(const fq_t &x, int) { return x; }
    static constexpr uint32_t kY = 8;
};
struct G2 {
    using F = fq2_t;
    static constexpr int kParts = 2;
    static fq2_t any() { return {coordinate(), coordinate()}; }
    static fq_t part(const fq2_t &x, int i) { return i ? x.c1 : x.c0; }
    static constexpr uint32_t kY = 4;
};
template <class G>
static void spread(const Xyzz<typename G::F> &p, Fp29<P> *word)
{
    const typename G::F *c[4] = {&p.X, &p.Y, &p.ZZ, &p.ZZZ};
    for (int q = 0; q < 4; ++q)
        for (int i = 0; i < G::kParts; ++i) {
            Fp29<P> &w = word[q * G::kParts + i];
            const fq_t x = G::part(*c[q], i);
            if (p.is_inf()) w = Fp29<P>::zero();
            else if (q == 0) w = represent<8>(x);
            else if (q == 1) w = represent<G::kY>(x);
            else w = represent<2>(x);
        }
}

// What the lanes add: component `word` of group g's operands and sum.
static Fp29<P> g_a[kRow][8], g_b[kRow][8], g_sum[kRow][8];
template <class F>
static void lane_main()
{
    const uint32_t me = threadIdx.x, g = me / Coop<F>::kLanes, w = Coop<F>::word();
    const Coop<F> r = coop_add(Coop<F>{g_a[g][w]}, Coop<F>{g_b[g][w]});
    g_sum[g][w] = r.v;
    g_done[me] = true;
    // on to the next lane, which has the same moves behind it; the last one is done
    for (;;) {
        if (me == kRow - 1) setcontext(&g_main);
        threadIdx.x = me + 1;
        setcontext(&g_lane[me + 1]);
    }
}
template <class F>
static void run_row()
{
    static std::vector<char> stacks(kRow * (256 << 10));
    for (int i = 0; i < kRow; ++i) {
        getcontext(&g_lane[i]);
        g_lane[i].uc_stack.ss_sp = &stacks[(size_t)i * (256 << 10)];
        g_lane[i].uc_stack.ss_size = 256 << 10;
        g_lane[i].uc_link = nullptr;
        makecontext(&g_lane[i], lane_main<F>, 0);
        g_moves[i] = 0;
        g_done[i] = false;
    }
    threadIdx.x = 0;
    swapcontext(&g_main, &g_lane[0]);
    for (int i = 0; i < kRow; ++i)
        if (!g_done[i]) std::abort();
}

template <class G>
static void check(int rows)
{
    using F = typename G::F;
    constexpr int lanes = 4 * G::kParts, groups = kRow / lanes;
    for (int row = 0; row < rows; ++row) {
        Xyzz<F> want[kRow];
        const bool plain = row % 3 == 0;  // no exceptional group in the row
        for (int g = 0; g < groups; ++g) {
            Xyzz<F> a, b;
            for (F *c : {&a.X, &a.Y, &a.ZZ, &a.ZZZ, &b.X, &b.Y, &b.ZZ, &b.ZZZ}) *c = G::any();
            const uint32_t kind = plain ? 9 : rnd() % 8;
            if (kind == 0) a = Xyzz<F>::infinity();
            if (kind == 1) b = Xyzz<F>::infinity();
            if (kind == 2) a = b = Xyzz<F>::infinity();
            if (kind == 3 || kind == 4) b = a;
            if (kind == 4) b.Y = FieldOps<F>::neg(b.Y);
            g_doublings += kind == 3;
            g_cancels += kind == 4;
            want[g] = xyzz_add(a, b);
            spread<G>(a, g_a[g]);
            spread<G>(b, g_b[g]);
        }
        run_row<F>();
        for (int g = 0; g < groups; ++g, ++g_adds) {
            const Fp29<P> *s = g_sum[g];
            bool limbs = true, inf = true, same = true, bounds = true;
            const F *c[4] = {&want[g].X, &want[g].Y, &want[g].ZZ, &want[g].ZZZ};
            for (int w = 0; w < lanes; ++w) {
                const int q = w / G::kParts;
                for (int k = 0; k < 9; ++k) limbs = limbs && (s[w].l[k] >> 29) == 0;
                bounds = bounds && (q == 0 ? is_below<8>(s[w]) : q == 1 ? is_below<G::kY>(s[w]) : is_below<2>(s[w]));
                same = same && (want[g].is_inf() || fp29_to_mont(s[w]) == G::part(*c[q], w % G::kParts));
                if (q == 2) inf = inf && s[w].is_exact_zero();
            }
            expect(limbs, "limbs", g_adds);
            expect(bounds, "bounds", g_adds);
            expect(inf == want[g].is_inf(), "infinity", g_adds);
            expect(same, "sum", g_adds);
        }
    }
}

int main()
{
    check<G1>(1200);
    check<G2>(1200);
    if (g_bad) {
        std::printf("FAILED %d\n", g_bad);
        return 1;
    }
    std::printf("ok %ld additions (%ld doublings, %ld cancellations)\n", g_adds, g_doublings, g_cancels);
    return 0;
}
