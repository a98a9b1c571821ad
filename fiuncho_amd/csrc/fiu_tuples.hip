// gfx950 kernels that count k-combinations on the matrix cores around a fixed
// head of k - 2 SNPs: the scans of order 4, of round-robin shares and of
// datasets with uncalled genotypes, and the tables of lower-order counts that
// the marginal form needs.
//
// For a head h = (s_1 < .. < s_{k-2}) the counts of the combinations
// (h, b, c) are dot products over the samples: row (b, y) times row (c, z)
// masked by the head's genotype rows.  Marginal form (complete coverage):
// genotypes 0 and 1 only, 2^k products per combination; the other cells
// follow by inclusion-exclusion from the counts of fewer SNPs.  All-cells
// form (any dataset): genotypes 0, 1 and 2, 3^k products and no tables.
//
// Counts of a combination travel as one 32-bit word per cell, cases in the
// low half and controls in the high half (datasets with counts16):
// the inclusion-exclusion then runs on both classes with one subtraction,
// since every intermediate value is itself a pair of counts and no half
// borrows from the other.
#include "fiu_kernels.h"

#include <algorithm>

#include "fiu_matrix.h"
#include "fiu_score.h"

namespace fiu {

namespace {

constexpr int ipow(int b, int e) { return e == 0 ? 1 : b * ipow(b, e - 1); }

// kSampleSmall: the sampling pass in tiles of 16 b rows
enum TupleMode { kScore = 0, kSample = 1, kTable = 2, kSampleSmall = 3 };
constexpr bool samples(int mode) { return mode == kSample || mode == kSampleSmall; }

// Shape of one kernel: W waves, NB blocks of 16 b rows against 16 W c columns,
// wave w taking columns c0 + 16 w ..; NB is a power of two, 4 at most, whose
// accumulators (4 registers per product and block) stay at 144 or below, so
// that two waves per SIMD fit (order 2 with uncalled genotypes, 9 products:
// NB = 4 560 us on 4,001 x 8,999, NB = 2 655, whose 18 KB per 72 products outran
// the loads).  Two waves per workgroup where the column range of a head is short
// (order 4 runs on a few hundred SNPs) or the staged c rows outweigh the shared
// b rows (all cells); four where the b rows do.
template <int K, bool ALL, int MODE = kScore> struct Tup {
    static constexpr int G = ALL ? 3 : 2;            // genotype rows per SNP
    static constexpr int H = K - 2;                  // head SNPs
    static constexpr int M = ipow(G, H);             // head cells
    static constexpr int dots = ipow(G, K);
    static constexpr int W = K == 4 || (K == 3 && ALL) ? 2 : 4;
    static constexpr int threads = 64 * W;
    static constexpr int CT = 16 * W;                // c columns per workgroup
    static constexpr int NB = MODE == kSampleSmall ? 1 : dots <= 9 ? 4 : dots == 16 ? 2 : 1;
    static constexpr int BT = 16 * NB;               // b rows per workgroup
    static constexpr int b_rows = G * BT;            // LDS rows (64 bytes) per stage
    static constexpr int c_rows = G * CT;
    static constexpr int a_rows = G * H;             // per wave: every wave has its own copy
    static constexpr int stage = (b_rows + c_rows + W * a_rows) * 64;
    // stages in LDS, ring - 1 in flight: 4, or 3 where two workgroups per CU
    // would not fit
    static constexpr int ring = 2 * 4 * stage <= 160 * 1024 ? 4 : 3;
    static constexpr int b_units = b_rows * 4 / W;   // 16-byte units of the b rows a wave loads
    static constexpr int b_loads = (b_units + 63) / 64;
    static constexpr int loads = b_loads + G + (H > 0 ? 1 : 0);   // per wave and stage
    static constexpr int inst = 4 * NB;              // combinations per lane
    static constexpr int cells = ipow(3, K);
    static constexpr int pairs = (dots + 1) / 2;     // words of one class's packed counts
    static_assert(loads * (ring - 2) < 64, "vmcnt immediate");
};

__device__ __forceinline__ int swz16(int r) { return (r >> 1) & 3; }

// Lexicographic rank of the pair x < y < n among the C(n, 2), below 2^32.
__device__ __forceinline__ uint32_t pair_index_u32(uint32_t x, uint32_t y, uint32_t n)
{
    return (uint32_t)((uint64_t)x * (2u * n - x - 1u) >> 1) + (y - x - 1u);
}

// A workgroup's head and its b progression: SNPs b_first, b_first + step, ..
// (the share's prefixes (head, b)), below n - 1.
template <int H> struct Head {
    int s[H > 0 ? H : 1];
    int b_first;     // above the head; n - 1 or above: no prefix of the share
};

template <int K>
__device__ __forceinline__ Head<K - 2> head_at(const ScanParams &P, int n, uint64_t h)
{
    constexpr int H = K - 2;
    Head<H> r;
    r.b_first = 0;
    if constexpr (H > 0) {
        unrank(h, n, H, P.binom, r.s);
        r.b_first = r.s[H - 1] + 1;
    }
    if (P.step != 1 || P.offset != 0) {
        // rank of the prefix (head, b) = r0 + b
        const uint64_t stride = (uint64_t)n + 1;
        int64_t r0 = (int64_t)P.binom[(uint64_t)(K - 1) * stride + n] - n;
#pragma unroll
        for (int i = 0; i < H; ++i) r0 -= (int64_t)P.binom[(uint64_t)(K - 1 - i) * stride + (n - 1 - r.s[i])];
        const int64_t at = r0 + r.b_first, rel = at - P.offset;
        const int64_t skip = rel < 0 ? -rel : (P.step - rel % P.step) % P.step;
        r.b_first = skip >= n ? n : r.b_first + (int)skip;
    }
    return r;
}

// Positions of a combination: 0 .. K - 3 the head, K - 2 b, K - 1 c.  A proper
// subset s of them (bit i = position i) of m SNPs t_0 < .. < t_{m-1} has its
// counts at entry C(n, m) - 1 - sum_i C(n-1-t_i, m-i) of table m (the
// lexicographic rank), 2^m words each.  Its b and c part is the rank of the
// pair (b, c), or b or c itself, so an entry is a wave-uniform base plus a
// 32-bit offset (the host checks that the largest fits).
template <int K> struct Subsets {
    const char *base[1 << K];
};
// uint4 words of the tables that depend on the instance's b, and their order:
// {b} as one, every other subset with b as 2^m / 4
template <int K> constexpr int subset_loads()
{
    int q = 0;
    for (int s = 1; s < (1 << K) - 1; ++s)
        if (s >> (K - 2) & 1) q += std::max(1, (1 << __builtin_popcount(s)) / 4);
    return q;
}
template <int K> constexpr int subset_slot(int s0)
{
    int q = 0;
    for (int s = 1; s < s0; ++s)
        if (s >> (K - 2) & 1) q += std::max(1, (1 << __builtin_popcount(s)) / 4);
    return q;
}
template <int K>
__device__ __forceinline__ void subsets_at(Subsets<K> &S, const TupleTables &T, const ScanParams &P, int n,
                                           const Head<K - 2> &h)
{
    constexpr int H = K - 2;
    const uint64_t stride = (uint64_t)n + 1;
    static_for<(1 << K) - 1>([&](auto I) __attribute__((always_inline)) {
        constexpr int s = decltype(I)::value;
        if constexpr (s != 0) {
            constexpr int m = __builtin_popcount(s);
            constexpr bool has_b = (s >> (K - 2) & 1) != 0, has_c = (s >> (K - 1) & 1) != 0;
            int64_t r = (int64_t)P.binom[(uint64_t)m * stride + n] - 1;
            int at = 0;
#pragma unroll
            for (int i = 0; i < H; ++i)
                if (s >> i & 1) {
                    r -= (int64_t)P.binom[(uint64_t)(m - at) * stride + (n - 1 - h.s[i])];
                    ++at;
                }
            if constexpr (has_b && has_c) r -= (int64_t)n * (n - 1) / 2 - 1;
            else if constexpr (has_b || has_c) r -= n - 1;
            S.base[s] = (const char *)T.t[m] + (r << (m + 2));
        }
    });
}

// The entry of subset s for (b, c), `pr` the rank of the pair (b, c).
template <int K, int s>
__device__ __forceinline__ const char *subset_entry(const Subsets<K> &S, uint32_t b, uint32_t c, uint32_t pr)
{
    constexpr int m = __builtin_popcount(s);
    constexpr bool has_b = (s >> (K - 2) & 1) != 0, has_c = (s >> (K - 1) & 1) != 0;
    const uint32_t at = has_b && has_c ? pr : has_b ? b : has_c ? c : 0u;
    return S.base[s] + (uint64_t)(at << (m + 2));
}

// Loads of one instance: its packed counts of both classes and the tables'
// words that depend on its b.
template <int K, bool ALL> struct Loaded {
    uint32_t w[2][Tup<K, ALL>::pairs];
    uint4 t[ALL ? 1 : subset_loads<K>()];
};

template <int K>
__device__ __forceinline__ void load_tables(uint4 (&t)[subset_loads<K>()], const Subsets<K> &S, uint32_t b, uint32_t c,
                                            uint32_t n)
{
    const uint32_t pr = pair_index_u32(b, c, n);
    static_for<(1 << K) - 1>([&](auto I) __attribute__((always_inline)) {
        constexpr int s = decltype(I)::value;
        if constexpr (s != 0 && (s >> (K - 2) & 1) != 0) {
            constexpr int m = __builtin_popcount(s), q0 = subset_slot<K>(s);
            const char *p = subset_entry<K, s>(S, b, c, pr);
            if constexpr (m == 1) {
                const uint2 v = *(const uint2 *)p;
                t[q0] = make_uint4(v.x, v.y, 0, 0);
            } else {
                static_for<(1 << m) / 4>([&](auto Q) __attribute__((always_inline)) {
                    t[q0 + decltype(Q)::value] = ((const uint4 *)p)[decltype(Q)::value];
                });
            }
        }
    });
}

// The 3^K cells (word: cases | controls << 16, first SNP most significant)
// of the combination whose 2^K corner counts (genotypes 0 and 1) are
// corner[], with t the words of load_tables; the subsets without b are read
// here (the head's at wave-uniform addresses, c's from L1).
template <int K>
__device__ __forceinline__ void marginal_cells(const Subsets<K> &S, const uint4 (&t)[subset_loads<K>()], uint32_t c,
                                               uint32_t total, const uint32_t (&corner)[1 << K],
                                               uint32_t (&m)[ipow(3, K)])
{
    // entry with "any genotype" (digit 2) outside subset s: the counts of s
    static_for<(1 << K)>([&](auto I) __attribute__((always_inline)) {
        constexpr int s = decltype(I)::value;
        constexpr int sz = __builtin_popcount(s);
        // cell index of entry e of the subset: the digits of its positions
        auto cell_of = [](int e) constexpr {
            int idx = 0, at = 0;
            for (int i = 0; i < K; ++i) {
                int d = 2;
                if (s >> i & 1) {
                    d = e >> (sz - 1 - at) & 1;
                    ++at;
                }
                idx = idx * 3 + d;
            }
            return idx;
        };
        if constexpr (s == 0) {
            m[ipow(3, K) - 1] = total;
        } else if constexpr (s == (1 << K) - 1) {
            static_for<(1 << K)>([&](auto E) __attribute__((always_inline)) {
                constexpr int e = decltype(E)::value, at = cell_of(e);
                m[at] = corner[e];
            });
        } else {
            static_for<(1 << sz) >= 4 ? (1 << sz) / 4 : 1>([&](auto Q) __attribute__((always_inline)) {
                constexpr int q = decltype(Q)::value;
                uint4 v;
                if constexpr ((s >> (K - 2) & 1) != 0) {
                    v = t[subset_slot<K>(s) + q];
                } else {
                    const char *p = subset_entry<K, s>(S, 0, c, 0);
                    if constexpr (sz == 1) {
                        const uint2 u = *(const uint2 *)p;
                        v = make_uint4(u.x, u.y, 0, 0);
                    } else {
                        v = ((const uint4 *)p)[q];
                    }
                }
                constexpr int a0 = cell_of(4 * q), a1 = cell_of(4 * q + 1);
                m[a0] = v.x;
                m[a1] = v.y;
                if constexpr (sz > 1) {
                    constexpr int a2 = cell_of(4 * q + 2), a3 = cell_of(4 * q + 3);
                    m[a2] = v.z;
                    m[a3] = v.w;
                }
            });
        }
    });
    // "any" -> genotype 2, last SNP first
#pragma unroll
    for (int d = 1; d < ipow(3, K); d *= 3)
#pragma unroll
        for (int hi = 0; hi < ipow(3, K); hi += 3 * d)
#pragma unroll
            for (int lo = 0; lo < d; ++lo) m[hi + 2 * d + lo] -= m[hi + lo] + m[hi + d + lo];
}

__device__ __forceinline__ float cases_of(uint32_t w) { return (float)(w & 0xffffu); }
__device__ __forceinline__ float ctrls_of(uint32_t w) { return (float)(w >> 16); }

// Upper bound on the MI of a table of packed cells.  With every sample called
// (P.bounded) the bound of mi_bound_fn.  Otherwise, with M = n_c + n_t called
// samples of N: MI = H(Y) + [n_c ln(n_c/M) + n_t ln(n_t/M)] / N + (M/N) times
// the MI among the called, and that MI is below its own chi2/M; a single
// pass over the cells' sum (packed words add without carry) gives n_c, n_t.
// The added logarithms err by less than 1e-6, inside bound_passes' margin.
struct BoundTerms {
    float frac, scale, base;
};
__device__ __forceinline__ BoundTerms bound_terms(float nc, float nt, const ScanParams &P)
{
    BoundTerms t;
    const float all = nc + nt, r = __builtin_amdgcn_rcpf(fmaxf(all, 1.0f));
    t.frac = nc * r;
    const float lc = __builtin_amdgcn_logf(fmaxf(t.frac, 7.9e-31f));
    const float lt = __builtin_amdgcn_logf(fmaxf(nt * r, 7.9e-31f));
    t.base = fmaf(fmaf(nc, lc, nt * lt), P.inv_n * 0.69314718f, P.hy);
    t.scale = nc > 0.0f && nt > 0.0f ? all * P.inv_n * (all * __builtin_amdgcn_rcpf(nc)) * __builtin_amdgcn_rcpf(nt)
                                     : 0.0f;
    return t;
}

// FIXED: the terms are the same for every table (all cover the samples of `t`).
template <bool FIXED, int CELLS>
__device__ __forceinline__ float packed_bound(const uint32_t (&m)[CELLS], const ScanParams &P, BoundTerms t)
{
    if constexpr (!FIXED) {
        uint32_t sum = 0;
#pragma unroll
        for (int x = 0; x < CELLS; ++x) sum += m[x];
        t = bound_terms(cases_of(sum), ctrls_of(sum), P);
    }
    return t.base + mi_bound_fn<CELLS>(
                        [&](int x, float &fc, float &fx) __attribute__((always_inline)) {
                            fc = cases_of(m[x]);
                            fx = fc + ctrls_of(m[x]);
                        },
                        t.frac, t.scale);
}

template <int CELLS>
__device__ __forceinline__ float packed_screen(const uint32_t (&m)[CELLS], const ScanParams &P)
{
    return fmaf(screen_sum_fn<CELLS>([&](int x, float &fc, float &ft) __attribute__((always_inline)) {
                    fc = cases_of(m[x]);
                    ft = ctrls_of(m[x]);
                }),
                P.inv_n * 0.69314718f, P.hy);
}

// What bounds it: the 2^K (3^K) products per combination, 16 cycles of a SIMD
// each for 256 combinations x 128 samples, and the cells' bound (about 13
// issue slots per cell) beside them; the operands come from L2 through a ring
// of 64-byte LDS rows filled by direct-to-LDS loads.  Why this split: the
// head's masks go on the c operand, of which a wave holds one 16-row block,
// so that a masked fragment (one three-operand AND per word and head cell)
// feeds NB x G products; each wave loads its own c and head rows, reads and
// masks them before the barrier that publishes the shared b rows.  Measured,
// stage loop alone: order 4 on 240 x 16,000 13 ms (matrix pipe busy 67 % of
// the cycles; the products of its 16 x 16 blocks take 8.8), a share of order
// 3 on 2,500 x 16,000 18 ms (9.7).  Counts wait as 16-bit pairs and the
// epilogue loads an instance ahead: the whole order-4 scan 35 -> 21 ms.
// b rows bmin + step * (0 .. BT - 1), of which those from hd.b_first on and
// below the column count; columns c0 + (0 .. CT - 1).
template <int K, bool ALL, int MODE>
__device__ __forceinline__ void tuple_tile(const DevData &D, const ScanParams &P, TopState *st, const TupleArgs &A,
                                           const Head<K - 2> &hd, int bmin, int c0,
                                           int8_t (*lds)[Tup<K, ALL, MODE>::stage], uint32_t *lds_hist)
{
    using Z = Tup<K, ALL, MODE>;
    constexpr int G = Z::G, H = Z::H, NB = Z::NB, R = Z::ring;
    const int n = D.n, np = D.n_pad;
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    // staging offsets within a quad of the image.  b rows: 16-byte units
    // U = b_units w + 64 i + lane of the stage's b part, row U / 4 = (genotype,
    // progression index), stored segment U % 4; rows past the last SNP read
    // the last one and are dropped in the epilogue
    uint32_t vb[Z::b_loads];
#pragma unroll
    for (int i = 0; i < Z::b_loads; ++i) {
        const int u = Z::b_units * w + 64 * i + lane, row = u >> 2;
        const int g = row / Z::BT, j = row % Z::BT;
        const int64_t snp = std::min<int64_t>((int64_t)bmin + (int64_t)P.step * j, n - 1);
        vb[i] = 16u * (uint32_t)(4 * (g * np + (int)snp) + ((u & 3) ^ swz16(row & 15)));
    }
    const int lr = lane >> 2, ls = (lane & 3) ^ swz16(lr);
    const uint32_t vc = 16u * (uint32_t)(4 * std::min(c0 + 16 * w + lr, n - 1) + ls);
    uint32_t va = 0;
    if constexpr (H > 0) {
        int s = hd.s[0];
#pragma unroll
        for (int i = 1; i < H; ++i)
            if (lr >= G * i) s = hd.s[i];
        va = 16u * (uint32_t)(4 * ((lr % G) * np + s) + (lane & 3));
    }
    const bool a_lane = lane < 4 * Z::a_rows;
    const int rr = lane & 15, kc = lane >> 4;
    const int fo = rr * 64 + ((kc ^ swz16(rr)) << 4), ao = kc << 4;
    // the 16-row b blocks [lo, hi) with a combination among the wave's columns:
    // rows from the head's first b on, below the last column (a wave without
    // any stages and waits with the others)
    const int c_top = std::min(c0 + 16 * w + 15, n - 1);
    int lo = 0, hi = 0;
#pragma unroll
    for (int bb = 0; bb < NB; ++bb) {
        const int64_t first = (int64_t)bmin + (int64_t)P.step * (16 * bb);
        if (first + 15 * (int64_t)P.step < hd.b_first) lo = bb + 1;
        if (first < c_top && c0 + 16 * w < n) hi = bb + 1;
    }
    lo = __builtin_amdgcn_readfirstlane(lo);
    hi = __builtin_amdgcn_readfirstlane(hi);
    const bool active = lo < hi, full = lo == 0 && hi == NB;
    v4f acc[Z::dots][NB];
    // per lane: the counts of its combinations as 16-bit pairs of products,
    // [class][instance][pair]; the pointer passes through an empty asm so that
    // they stay in memory
    uint32_t counts_mem[2 * Z::inst * Z::pairs];
    __attribute__((address_space(5))) uint32_t *counts = (__attribute__((address_space(5))) uint32_t *)counts_mem;
    asm volatile("" : "+v"(counts));
#pragma unroll 1
    for (int cls = 0; cls < 2; ++cls) {
#pragma unroll
        for (int e = 0; e < Z::dots; ++e)
#pragma unroll
            for (int bb = 0; bb < NB; ++bb) acc[e][bb] = (v4f){0.f, 0.f, 0.f, 0.f};
        const int iters = D.quads[cls];
        const uint4 *img = A.F.base + A.F.class_off[cls];
        auto issue = [&](int q) __attribute__((always_inline)) {
            const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc(
                (void *)(img + (int64_t)q * 4 * G * np), (short)0, 64 * G * np, 0x00020000);
            int8_t *s = lds[q % R];
#pragma unroll
            for (int i = 0; i < Z::b_loads; ++i) {
                int8_t *to = s + (Z::b_units * w + 64 * i) * 16;
                if (64 * (i + 1) <= Z::b_units) dma16(rq, vb[i], to);
                else if (lane < Z::b_units - 64 * i) dma16(rq, vb[i], to);
            }
#pragma unroll
            for (int g = 0; g < G; ++g)
                dma16(rq, vc + 64u * (uint32_t)(g * np), s + (Z::b_rows + Z::CT * g + 16 * w) * 64);
            if constexpr (H > 0)
                if (a_lane) dma16(rq, va, s + (Z::b_rows + Z::c_rows + Z::a_rows * w) * 64);
        };
#pragma unroll
        for (int q = 0; q < R - 1; ++q)
            if (q < iters) issue(q);
        // steady: at least R - 1 stages follow; FULL: every b block is used
        auto stage = [&](int it, bool steady, auto FULL) __attribute__((always_inline)) {
            // this wave's loads of stage it are complete once at most those
            // of the stages issued after it are pending
            if (steady) wait_vmcnt<Z::loads * (R - 2)>();
            else wait_stages<R - 2, Z::loads>(iters - 1 - it);
            asm volatile("" ::: "memory");
            // its own c and head rows are there: masked c fragments
            const int8_t *sb = lds[it % R];
            v4i mc[Z::M][G];
            {
                v4i fa[H > 0 ? Z::a_rows : 1], fc[G];
                if constexpr (H > 0) {
#pragma unroll
                    for (int r = 0; r < Z::a_rows; ++r)
                        fa[r] = *(const v4i *)(sb + (Z::b_rows + Z::c_rows + Z::a_rows * w + r) * 64 + ao);
                }
#pragma unroll
                for (int g = 0; g < G; ++g) fc[g] = *(const v4i *)(sb + (Z::b_rows + Z::CT * g + 16 * w) * 64 + fo);
#pragma unroll
                for (int mi = 0; mi < Z::M; ++mi)
#pragma unroll
                    for (int z = 0; z < G; ++z) {
                        mc[mi][z] = fc[z];   // nibble 0x2 & 0x2 = 1.0, else 0
#pragma unroll
                        for (int i = 0; i < H; ++i) mc[mi][z] &= fa[i * G + mi / ipow(G, H - 1 - i) % G];
                    }
            }
            // the barrier publishes every wave's b rows and tells that the
            // slot of stage it - 1 is read no more
            stage_barrier();
            __builtin_amdgcn_s_setprio(1);
            v4i fb[G][NB];
#pragma unroll
            for (int bb = 0; bb < NB; ++bb)
#pragma unroll
                for (int g = 0; g < G; ++g) fb[g][bb] = *(const v4i *)(sb + (g * Z::BT + 16 * bb) * 64 + fo);
            if (steady || it + R - 1 < iters) issue(it + R - 1);
#pragma unroll
            for (int bb = 0; bb < NB; ++bb) {
                if (!decltype(FULL)::value && (bb < lo || bb >= hi)) continue;
#pragma unroll
                for (int y = 0; y < G; ++y) {
                    const v8i b8 = {fb[y][bb][0], fb[y][bb][1], fb[y][bb][2], fb[y][bb][3], 0, 0, 0, 0};
#pragma unroll
                    for (int mi = 0; mi < Z::M; ++mi)
#pragma unroll
                        for (int z = 0; z < G; ++z) {
                            const v8i c8 = {mc[mi][z][0], mc[mi][z][1], mc[mi][z][2], mc[mi][z][3], 0, 0, 0, 0};
                            v4f &d = acc[(mi * G + y) * G + z][bb];
                            d = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(b8, c8, d, 4, 4, 0, 0, 0, 0);
                        }
                }
            }
            __builtin_amdgcn_s_setprio(0);
        };
        auto idle = [&](int it) __attribute__((always_inline)) {
            wait_stages<R - 2, Z::loads>(iters - 1 - it);
            stage_barrier();
            if (it + R - 1 < iters) issue(it + R - 1);
        };
        int it = 0;
        if (full) {
            for (; it + R - 1 < iters; ++it) stage(it, true, std::true_type{});
            for (; it < iters; ++it) stage(it, false, std::true_type{});
        } else if (active) {
            for (; it < iters; ++it) stage(it, false, std::false_type{});
        } else {
            for (; it < iters; ++it) idle(it);
        }
        // the ring is filled again by the next class (or tile)
        stage_barrier();
        if (active) {
            __attribute__((address_space(5))) uint32_t *to = counts + cls * (Z::inst * Z::pairs);
#pragma unroll
            for (int bb = 0; bb < NB; ++bb)
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int e = 0; e < Z::pairs; ++e) {
                        const uint32_t v0 = (uint32_t)acc[2 * e][bb][j];
                        const uint32_t v1 = 2 * e + 1 < Z::dots ? (uint32_t)acc[2 * e + 1 < Z::dots ? 2 * e + 1 : 0][bb][j] : 0;
                        to[(bb * 4 + j) * Z::pairs + e] = v0 | v1 << 16;
                    }
        }
    }
    if (!active) return;
    // epilogue: lane holds column c = c0 + 16 w + lane % 16 and rows
    // b = bmin + step (16 bb + 4 (lane / 16) + j), instance i = 4 bb + j; the
    // next instance's counts and tables are loaded while one is scored
    const int c = std::min(c0 + 16 * w + rr, n - 1);
    const bool c_ok = c0 + 16 * w + rr < n;
    const float tau = MODE == kScore ? st->tau : 0.0f;
    const uint64_t tau_combo = MODE == kScore ? st->tau_combo : 0;
    auto b_at = [&](int i) { return (int64_t)bmin + (int64_t)P.step * (16 * (i >> 2) + 4 * kc + (i & 3)); };
    // (an aligned block starts below b_first, and in the head where the share's
    // offset falls, members of the progression above the head lie before it)
    auto valid_at = [&](int64_t b) { return c_ok && b < c && b >= hd.b_first; };
    // columns up to the first b (aligned tiles) read a valid one's tables
    const uint32_t c_tab = (uint32_t)std::max(c, hd.b_first + 1);
    const uint32_t total = D.total[0] | D.total[1] << 16;
    Subsets<K> S;
    if constexpr (!ALL && MODE != kTable) subsets_at<K>(S, A.T, P, n, hd);
    auto load = [&](int i, Loaded<K, ALL> &x) __attribute__((always_inline)) {
#pragma unroll
        for (int cls = 0; cls < 2; ++cls)
#pragma unroll
            for (int e = 0; e < Z::pairs; ++e) x.w[cls][e] = counts[(cls * Z::inst + i) * Z::pairs + e];
        if constexpr (!ALL && MODE != kTable) {
            // a combination outside the scan reads a valid one's tables
            const int64_t b = b_at(i);
            const bool ok = b < c && b >= hd.b_first;
            load_tables<K>(x.t, S, ok ? (uint32_t)b : (uint32_t)hd.b_first, c_tab, (uint32_t)n);
        }
    };
    // both classes' counts of each product, cases | controls << 16
    auto words = [&](const Loaded<K, ALL> &x, uint32_t (&v)[Z::dots]) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < Z::dots; ++e)
            v[e] = e & 1 ? __builtin_amdgcn_perm(x.w[1][e / 2], x.w[0][e / 2], 0x07060302u)
                         : __builtin_amdgcn_perm(x.w[1][e / 2], x.w[0][e / 2], 0x05040100u);
    };
    auto cells_of = [&](const Loaded<K, ALL> &x, uint32_t (&m)[Z::cells]) __attribute__((always_inline)) {
        if constexpr (ALL) {
            words(x, m);
        } else {
            uint32_t v[Z::dots];
            words(x, v);
            marginal_cells<K>(S, x.t, c_tab, total, v, m);
        }
    };
    uint32_t pend = 0;
    const int i1 = 4 * hi;
    Loaded<K, ALL> cur;
    if constexpr (MODE == kScore) {
        // U instances at a time, without a branch, so that their chains overlap
        constexpr int U = K <= 3 ? 2 : 1;
        const BoundTerms fixed = P.bounded ? BoundTerms{P.frac_c, P.chi_scale, 0.0f}
                                           : bound_terms(cases_of(total), ctrls_of(total), P);
#pragma unroll 1
        for (int i = 4 * lo; i < i1; i += U) {
            Loaded<K, ALL> x[U];
#pragma unroll
            for (int u = 0; u < U; ++u) load(i + u, x[u]);
            uint32_t marks = 0;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                uint32_t m[Z::cells];
                cells_of(x[u], m);
                const float bound = packed_bound<!ALL>(m, P, fixed);
                const bool pass = bound_passes(bound, tau, P.delta), valid = valid_at(b_at(i + u));
                marks |= ((uint32_t)pass & (uint32_t)valid) << u;   // no branch
            }
            pend |= marks << i;
        }
    } else {
        Loaded<K, ALL> nxt;
        load(4 * lo, cur);
#pragma unroll 1
        for (int i = 4 * lo; i < i1; ++i) {
            load(std::min(i + 1, i1 - 1), nxt);
            const int64_t bi = b_at(i);
            const bool valid = valid_at(bi);
            if constexpr (MODE == kTable) {
                if (valid) {
                    const uint64_t stride = (uint64_t)n + 1;
                    int64_t r = (int64_t)P.binom[(uint64_t)K * stride + n] - 1;
#pragma unroll
                    for (int q = 0; q < H; ++q) r -= (int64_t)P.binom[(uint64_t)(K - q) * stride + (n - 1 - hd.s[q])];
                    const int64_t v = n - 1 - bi;
                    r -= v * (v - 1) / 2 + (n - 1 - c);
                    uint4 *to = (uint4 *)(A.out + (r << K));
                    uint32_t x[Z::dots];
                    words(cur, x);
#pragma unroll
                    for (int e = 0; e < Z::dots; e += 4) to[e / 4] = make_uint4(x[e], x[e + 1], x[e + 2], x[e + 3]);
                }
            } else {
                uint32_t m[Z::cells];
                cells_of(cur, m);
                const float ms = packed_screen<Z::cells>(m, P);
                if (valid) atomicAdd(&lds_hist[hist_bin(ms)], 1u);
            }
            cur = nxt;
        }
    }
    if constexpr (MODE == kScore) {
        // one marked combination per lane and round: screen, exact MI, push
        while (__ballot(pend != 0)) {
            bool need = false;
            int pre[K - 1] = {};
            uint32_t m[Z::cells];
            if (pend) {
                const int i = __builtin_ctz(pend);
                pend &= pend - 1;
                load(i, cur);
                cells_of(cur, m);
#pragma unroll
                for (int q = 0; q < H; ++q) pre[q] = hd.s[q];
                pre[H] = (int)b_at(i);
                need = packed_screen<Z::cells>(m, P) >= tau - P.delta;
            }
            exact_push<Z::cells>(
                need,
                [&](int x, uint32_t &n0, uint32_t &n1) __attribute__((always_inline)) {
                    n0 = m[x] & 0xffffu;
                    n1 = m[x] >> 16;
                },
                [&] { return prefix_key(P.binom, n, pre, K - 1) + (uint64_t)c; }, tau, tau_combo, P, st);
        }
    }
}

// Work: unit u of [j0, j1), u = j0 + i * stride, is a head (K >= 3) or a block
// of BT b's (K = 2, no head).  Workgroup L runs on XCD L % 8.
// Free tiles: a head's tiles (b blocks from its first b on, and for each the
// column tiles past the block's first b) are dealt to 8 * `rounds`
// workgroups; for 64 units in a row an XCD takes the same tile number, then
// the next, so that the XCDs' shares of units with few tiles even out.
// Sampling takes every tile_stride-th tile of a unit, starting elsewhere in
// each.
// Aligned tiles (A.aligned, shares of order 3): blocks of BT members of the
// progression b = b_first mod step, and columns in multiples of CT, so that
// the heads whose progressions agree -- first SNPs 2 step apart -- use the
// same rows; they run back to back on one XCD, a tile at a time.  Costs half
// a block more per head, but an XCD's L2 holds the rows its workgroups read:
// on 2,500 x 16,000, step 8, the scan fetched 129 GB beyond L2 with free
// tiles and 4.3 with aligned ones, 39 -> 26 ms.
template <int K, bool ALL, int MODE>
__global__ void __launch_bounds__((Tup<K, ALL, MODE>::threads)) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_tuples(const DevData D, const ScanParams P, TopState *st, const TupleArgs A)
{
    using Z = Tup<K, ALL, MODE>;
    // one array: beside a second one the compiler waits for every pending
    // direct-to-LDS load ahead of each stage's reads (a sampling pass of
    // 5,003 x 9,001: 76 us so, 29 with the histogram behind the ring)
    __shared__ __attribute__((aligned(1024))) int8_t lds_all[Z::ring * Z::stage + (samples(MODE) ? 4 * kHistBins : 0)];
    int8_t(*const lds)[Z::stage] = (int8_t(*)[Z::stage])lds_all;
    uint32_t *const lds_hist = (uint32_t *)(lds_all + (samples(MODE) ? Z::ring * Z::stage : 0));
    const int64_t L = blockIdx.x, s = L >> 3;
    if constexpr (K == 3 && MODE == kScore) {
        if (A.aligned) {
            // unit i of class i / per: heads j0 + class + 2 step k
            const int64_t i = s % A.units, tile = s / A.units * 8 + (L & 7);
            const int64_t period = 2 * P.step, per = (P.j1 - P.j0 + period - 1) / period;
            const int64_t u = P.j0 + i % per * period + i / per;
            if (u >= P.j1 || tile >= (int64_t)A.nb * A.nc) return;
            const Head<Z::H> hd = head_at<K>(P, D.n, (uint64_t)u);
            const int64_t ib = tile / A.nc, c0 = tile % A.nc * Z::CT, span = (int64_t)Z::BT * P.step;
            const int64_t bmin = ib * span + hd.b_first % P.step;
            // first and last b of the block in the share
            const int64_t b0 = std::max<int64_t>(bmin, hd.b_first), b1 = bmin + span - P.step;
            if (b1 < hd.b_first || b0 >= D.n - 1 || c0 + Z::CT - 1 <= b0 || c0 >= D.n) return;
            tuple_tile<K, ALL, MODE>(D, P, st, A, hd, (int)bmin, (int)c0, lds, lds_hist);
            return;
        }
    }
    // (a sample has few tiles per unit: the XCDs take turns sooner)
    constexpr int turn = !samples(MODE) ? 6 : K == 2 ? 3 : 0;
    const int64_t i = s % A.units, first = s / A.units * 8 + ((L + (i >> turn)) & 7);
    const int64_t u = P.j0 + i * A.stride;
    const Head<Z::H> hd = head_at<K>(P, D.n, K == 2 ? 0 : (uint64_t)u);
    // sampling: the unit's tiles at multiples of tile_stride, from its own first
    const int64_t ts = samples(MODE) ? A.tile_stride : 1;
    int64_t tile = first * ts;
    int64_t bmin = hd.b_first;
    if constexpr (K == 2) bmin += u * Z::BT * P.step;
    // an order-2 sample takes whole column tiles of the table, the same ones
    // for eight units in a row, which one XCD runs: their c rows stay in its L2
    // (50,000 x 32,000: 1.4 -> 0.8 ms)
    const int64_t skip = K == 2 && samples(MODE) ? (bmin + 1) / Z::CT : 0;
    if constexpr (samples(MODE)) {
        const int64_t at = (K == 2 ? u / 8 : u) % ts * 5 + skip;
        tile += (ts - at % ts) % ts;
    }
    bool any = false;   // a workgroup without a tile leaves the histogram alone
    while (bmin < D.n - 1) {
        // column tiles past bmin
        const int64_t from = K == 2 && samples(MODE) ? skip * Z::CT : bmin + 1;
        const int ct = (int)(D.n - from + Z::CT - 1) / Z::CT;
        if (tile < ct) {
            if (!any) hist_begin<samples(MODE)>(lds_hist);
            any = true;
            tuple_tile<K, ALL, MODE>(D, P, st, A, hd, (int)bmin, (int)from + Z::CT * (int)tile, lds, lds_hist);
            tile += 8 * (int64_t)A.rounds * ts;
        } else {
            if constexpr (K == 2) break;
            tile -= ct;
            bmin += (int64_t)Z::BT * P.step;
        }
    }
    if (!any) return;
    hist_end<samples(MODE)>(lds_hist, P.hist);
}

// fp4 image of genotype rows 0 .. G - 1, as the two-row image of the pair
// and triple scans: quad q, genotype g, SNP s of a class at 4 ((G q + g)
// n_pad + s) past the class's offset.
__global__ void k_tuple_image(const uint4 *__restrict__ bits, DevData D, uint4 *__restrict__ out, uint64_t off1)
{
    const uint64_t id = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t per0 = 3ull * D.quads[0] * D.n_pad, total = per0 + 3ull * D.quads[1] * D.n_pad;
    if (id >= total) return;
    const int cls = id < per0 ? 0 : 1;
    const uint64_t v = cls ? id - per0 : id;
    const uint4 w = bits[D.class_off[cls] + v];
    uint4 *dst = out + (cls ? off1 : 0) + 4 * v;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t x = comp(w, e);
        dst[e] = make_uint4(byte_fp4(x & 255u), byte_fp4(x >> 8 & 255u), byte_fp4(x >> 16 & 255u), byte_fp4(x >> 24));
    }
}

// Table of one SNP: words (genotype 0, genotype 1), cases | controls << 16.
__global__ void k_tuple_singles(DevData D, uint32_t *out)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 2 * D.n) return;
    const uint32_t *sp = D.singles + (size_t)(i >> 1) * 6 + (i & 1);
    out[i] = sp[0] | sp[3] << 16;
}

template <int K, bool ALL, int MODE>
hipError_t launch_tuples_as(const DevData &D, ScanParams P, TopState *st, TupleArgs A, hipStream_t s)
{
    using Z = Tup<K, ALL, MODE>;
    // a dispatch holds at most 2^32 - 1 work-items
    constexpr int64_t max_blocks = (int64_t)(0xffffffffu / (uint32_t)Z::threads);
    int64_t units = (P.j1 - P.j0 + A.stride - 1) / A.stride;
    if (units <= 0) return hipSuccess;
    const int64_t span = Z::BT * P.step;
    A.nb = (int32_t)((D.n + span - 1) / span);
    A.nc = (D.n + Z::CT - 1) / Z::CT;
    A.aligned = K == 3 && MODE == kScore && P.step > 1;
    const int64_t most = K == 2 ? A.nc : (int64_t)std::max(A.nb, 1) * A.nc;   // tiles of the largest unit
    if (A.aligned) {
        // one workgroup per unit and tile; units padded to whole classes
        A.rounds = (int32_t)((most + 7) / 8);
    } else {
        // a unit's (sampled) tiles dealt in rounds of 8: no more rounds than
        // fill the device
        const int64_t want = std::max<int64_t>(1, (int64_t)A.fill / std::max<int64_t>(1, 8 * units));
        const int64_t taken = samples(MODE) ? (most + A.tile_stride - 1) / A.tile_stride : most;
        A.rounds = (int32_t)std::min<int64_t>((taken + 7) / 8, want);
    }
    const int64_t per_launch = std::max<int64_t>(1, max_blocks / (8 * (int64_t)A.rounds) / 2);
    for (int64_t i = 0; i < units; i += per_launch) {
        ScanParams Q = P;
        TupleArgs B = A;
        const int64_t count = std::min(per_launch, units - i);
        Q.j0 = P.j0 + i * A.stride;
        Q.j1 = std::min(P.j1, P.j0 + (i + count) * A.stride);
        B.units = count;
        if (A.aligned) {
            const int64_t period = 2 * P.step, per = (Q.j1 - Q.j0 + period - 1) / period;
            B.units = per * std::min(period, Q.j1 - Q.j0);
        }
        hipLaunchKernelGGL((k_tuples<K, ALL, MODE>), dim3((unsigned)(B.units * 8 * B.rounds)), dim3(Z::threads), 0, s,
                           D, Q, st, B);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <int K, bool ALL>
hipError_t launch_tuples_k(const DevData &D, const ScanParams &P, TopState *st, const TupleArgs &A, hipStream_t s)
{
    if constexpr (!ALL && K <= 3)
        if (A.out) return launch_tuples_as<K, ALL, kTable>(D, P, st, A, s);
    if (P.hist && A.small) return launch_tuples_as<K, ALL, kSampleSmall>(D, P, st, A, s);
    if (P.hist) return launch_tuples_as<K, ALL, kSample>(D, P, st, A, s);
    return launch_tuples_as<K, ALL, kScore>(D, P, st, A, s);
}

}  // namespace

int tuple_b_block(int order, bool all_cells, bool small)
{
    if (small) return 16;
    if (all_cells) return order == 2 ? Tup<2, true>::BT : Tup<3, true>::BT;
    return order == 2 ? Tup<2, false>::BT : order == 3 ? Tup<3, false>::BT : Tup<4, false>::BT;
}

hipError_t launch_tuples(int order, bool all_cells, const DevData &D, const ScanParams &P, TopState *st,
                         const TupleArgs &A, hipStream_t s)
{
    if (all_cells) {
        if (order == 2) return launch_tuples_k<2, true>(D, P, st, A, s);
        if (order == 3) return launch_tuples_k<3, true>(D, P, st, A, s);
        return hipErrorInvalidValue;
    }
    if (order == 2) return launch_tuples_k<2, false>(D, P, st, A, s);
    if (order == 3) return launch_tuples_k<3, false>(D, P, st, A, s);
    if (order == 4) return launch_tuples_k<4, false>(D, P, st, A, s);
    return hipErrorInvalidValue;
}

hipError_t launch_tuple_singles(const DevData &D, uint32_t *out, hipStream_t s)
{
    if (D.n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_tuple_singles, dim3((unsigned)((2 * D.n + 255) / 256)), dim3(256), 0, s, D, out);
    return hipGetLastError();
}

hipError_t launch_tuple_image(const DevData &D, uint4 *out, hipStream_t s)
{
    const uint64_t total = 3ull * (D.quads[0] + D.quads[1]) * D.n_pad;
    if (!total) return hipSuccess;
    hipLaunchKernelGGL(k_tuple_image, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, D.bits, D, out,
                       12ull * D.quads[0] * D.n_pad);
    return hipGetLastError();
}

}  // namespace fiu
