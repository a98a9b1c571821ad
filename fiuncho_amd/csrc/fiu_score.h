// Device code shared by the scan kernels: bit-table loads, unranking and
// combination keys, the MI bound, screen and exact value, candidate pushes and
// the threshold sampling histogram.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>

#include <type_traits>
#include <utility>

#include "fiu_device.h"

namespace fiu {

template <int N> struct Pow3 { static constexpr int v = 3 * Pow3<N - 1>::v; };
template <> struct Pow3<0> { static constexpr int v = 1; };

__device__ __forceinline__ uint32_t comp(const uint4 &v, int w)
{
    return w == 0 ? v.x : w == 1 ? v.y : w == 2 ? v.z : v.w;
}

// Buffer resource over the three genotype rows of one quad (all SNPs of one
// class); loads through it are in-order vector loads whose offset can live in
// an SGPR (wave-uniform prefix rows) or a VGPR (the lanes' own SNPs), with no
// 64-bit address arithmetic, and reads past the rows return zero.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t quad_rsrc(const uint4 *row, int np)
{
    return __builtin_amdgcn_make_buffer_rsrc((void *)row, (short)0, 3 * np * 16, 0x00020000);
}

// Row z of SNP s (wave-uniform s): 16 bytes broadcast to every lane.
__device__ __forceinline__ uint4 ld_uniform(__amdgpu_buffer_rsrc_t r, int np, int z, int s)
{
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, 0, (z * np + s) * 16, 0);
    return make_uint4(v[0], v[1], v[2], v[3]);
}

// Row z of each lane's SNP (voff = 16 * SNP index).
__device__ __forceinline__ uint4 ld_lane(__amdgpu_buffer_rsrc_t r, int np, int z, int voff)
{
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, voff, z * np * 16, 0);
    return make_uint4(v[0], v[1], v[2], v[3]);
}

// acc_k += popcount(x_k & y_k & z_k) for four independent cells: one
// v_bitop3_b32 (3-input AND) and one accumulating v_bcnt_u32_b32 per cell,
// the four ANDs issued before the four popcounts.
__device__ __forceinline__ void and3_bcnt4(uint32_t &a0, uint32_t &a1, uint32_t &a2, uint32_t &a3, uint32_t x0,
                                           uint32_t y0, uint32_t z0, uint32_t x1, uint32_t y1, uint32_t z1,
                                           uint32_t x2, uint32_t y2, uint32_t z2, uint32_t x3, uint32_t y3,
                                           uint32_t z3)
{
    uint32_t t0, t1, t2, t3;
    asm("v_bitop3_b32 %0, %4, %5, %6 bitop3:0x80\n\t"
        "v_bitop3_b32 %1, %7, %8, %9 bitop3:0x80\n\t"
        "v_bitop3_b32 %2, %10, %11, %12 bitop3:0x80\n\t"
        "v_bitop3_b32 %3, %13, %14, %15 bitop3:0x80"
        : "=&v"(t0), "=&v"(t1), "=&v"(t2), "=&v"(t3)
        : "v"(x0), "v"(y0), "v"(z0), "v"(x1), "v"(y1), "v"(z1), "v"(x2), "v"(y2), "v"(z2), "v"(x3), "v"(y3),
          "v"(z3));
    asm("v_bcnt_u32_b32 %0, %4, %0\n\t"
        "v_bcnt_u32_b32 %1, %5, %1\n\t"
        "v_bcnt_u32_b32 %2, %6, %2\n\t"
        "v_bcnt_u32_b32 %3, %7, %3"
        : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3)
        : "v"(t0), "v"(t1), "v"(t2), "v"(t3));
}

// acc_k += popcount(x_k & y_k), four independent cells, VGPR operands.
__device__ __forceinline__ void and2_bcnt4(uint32_t &a0, uint32_t &a1, uint32_t &a2, uint32_t &a3, uint32_t x0,
                                           uint32_t y0, uint32_t x1, uint32_t y1, uint32_t x2, uint32_t y2,
                                           uint32_t x3, uint32_t y3)
{
    uint32_t t0, t1, t2, t3;
    asm("v_and_b32 %0, %4, %5\n\t"
        "v_and_b32 %1, %6, %7\n\t"
        "v_and_b32 %2, %8, %9\n\t"
        "v_and_b32 %3, %10, %11"
        : "=&v"(t0), "=&v"(t1), "=&v"(t2), "=&v"(t3)
        : "v"(x0), "v"(y0), "v"(x1), "v"(y1), "v"(x2), "v"(y2), "v"(x3), "v"(y3));
    asm("v_bcnt_u32_b32 %0, %4, %0\n\t"
        "v_bcnt_u32_b32 %1, %5, %1\n\t"
        "v_bcnt_u32_b32 %2, %6, %2\n\t"
        "v_bcnt_u32_b32 %3, %7, %3"
        : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3)
        : "v"(t0), "v"(t1), "v"(t2), "v"(t3));
}

// Lexicographic unranking of an m-combination of [0, n) (wave-uniform).
// rank(c) = C(n,m) - 1 - sum_i C(n-1-c_i, m-i), so the complement is written
// greedily in the combinatorial number system.
__device__ inline void unrank(uint64_t r, int n, int m, const uint64_t *binom, int *out)
{
    const uint64_t stride = (uint64_t)n + 1;
    uint64_t x = binom[(uint64_t)m * stride + n] - 1 - r;
    int hi = n - 1;
    for (int i = 0; i < m; ++i) {
        const int j = m - i;
        int lo = 0, h = hi;
        while (lo < h) {
            const int mid = (lo + h + 1) >> 1;
            if (binom[(uint64_t)j * stride + mid] <= x) lo = mid;
            else h = mid - 1;
        }
        x -= binom[(uint64_t)j * stride + lo];
        out[i] = n - 1 - lo;
        hi = lo - 1;
    }
}

// Lexicographic rank of the k-combination (pre[0] < ... < pre[k-2] < c) of
// [0, n), the key of a candidate: rank = C(n,k) - 1 - sum_i C(n-1-c_i, k-i),
// whose last term is C(n-1-c, 1) = n-1-c, so the rank is a constant of the
// prefix plus c.  Needs the binomial table up to row k and C(n, k) < 2^64
// (checked on the host).  Ranks keep the lexicographic order of the
// combinations, so comparing keys compares combinations.
__device__ __forceinline__ uint64_t prefix_key(const uint64_t *binom, int n, const int *pre, int M)
{
    const uint64_t stride = (uint64_t)n + 1;
    uint64_t s = binom[(uint64_t)(M + 1) * stride + n] - (uint64_t)n;   // C(n,k) - 1 - (n - 1)
    for (int i = 0; i < M; ++i) s -= binom[(uint64_t)(M + 1 - i) * stride + (n - 1 - pre[i])];
    return s;
}

// Screening MI in FP32 from exact counts, in the conditional-entropy form
// MI = H(Y) + (1/N) sum_x [n_cx ln(n_cx/n_x) + n_tx ln(n_tx/n_x)], whose terms
// all have one sign (no cancellation inside the sum).  Error < 2e-6 nats for
// N < 2^24; only used to decide which combinations get the exact value.
// Counts as uint32_t or as FP32 holding the same integers (exact below 2^24).
// The sum over cells, in log2 units (the screen of a table split over
// several lanes adds their sums).
// Cells come from cell(x, fc, ft) (counts as FP32), x < CELLS.
template <int CELLS, class F>
__device__ __forceinline__ float screen_sum_fn(F &&cell)
{
    // hardware v_rcp_f32 / v_log_f32 (log2) on normal arguments: every ratio
    // is clamped to >= 2^-100, and a zero count multiplies its log by zero
    float s = 0.0f;
#pragma unroll
    for (int x = 0; x < CELLS; ++x) {
        float fc, ft;
        cell(x, fc, ft);
        const float r = __builtin_amdgcn_rcpf(fmaxf(fc + ft, 1.0f));
        const float lc = __builtin_amdgcn_logf(fmaxf(fc * r, 7.9e-31f));
        const float lt = __builtin_amdgcn_logf(fmaxf(ft * r, 7.9e-31f));
        s = fmaf(fc, lc, s);
        s = fmaf(ft, lt, s);
    }
    return s;
}

template <int CELLS, class T>
__device__ __forceinline__ float screen_sum(const T *a0, const T *a1)
{
    return screen_sum_fn<CELLS>([&](int x, float &fc, float &ft) __attribute__((always_inline)) {
        fc = (float)a0[x];
        ft = (float)a1[x];
    });
}

template <int CELLS, class T>
__device__ __forceinline__ float mi_screen(const T *a0, const T *a1, float hy, float inv_n)
{
    return fmaf(screen_sum<CELLS>(a0, a1), inv_n * 0.69314718f, hy);
}

// v_mul_legacy_f32: the product, with 0 times anything 0 (the compiler's own
// intrinsic, which has no builtin name).
__device__ float fmul_legacy(float a, float b) __asm("llvm.amdgcn.fmul.legacy");

// Upper bound on the MI in nats, one reciprocal per cell and no logarithm:
// MI = KL(P_XY || P_X P_Y) <= ln(1 + chi2/N) <= chi2/N (Jensen's inequality
// on E_P[P_XY / (P_X P_Y)]), and with two classes
//   chi2/N = N/(n_c n_t) sum_x d_x^2 / n_x,  d_x = n_cx - n_x n_c/N.
// FP32 error: below 2e-6 relative plus 5e-7 absolute (each |d_x| error is
// under 1.2e-7 (n_x n_c/N + |d_x|), and sum_x |d_x| <= 2 min(n_c, n_t)).
// Cells from cell(x, fc, fx): case count and case + control count, FP32.
template <int CELLS, class F>
__device__ __forceinline__ float mi_bound_fn(F &&cell, float frac_c, float chi_scale)
{
    float s = 0.0f;
#pragma unroll
    for (int x = 0; x < CELLS; ++x) {
        float fc, fx;
        cell(x, fc, fx);
        // an empty cell has d = 0, and 0 times its infinite reciprocal is 0 in
        // the legacy product: no clamp of fx
        const float d = fmaf(-fx, frac_c, fc);
        s = fmaf(fmul_legacy(d, __builtin_amdgcn_rcpf(fx)), d, s);
    }
    return s * chi_scale;
}

template <int CELLS, class T>
__device__ __forceinline__ float mi_bound(const T *a0, const T *a1, float frac_c, float chi_scale)
{
    return mi_bound_fn<CELLS>(
        [&](int x, float &fc, float &fx) __attribute__((always_inline)) {
            fx = (float)(a0[x] + a1[x]);
            fc = (float)a0[x];
        },
        frac_c, chi_scale);
}

// The bound rejects a combination when even its bound, raised by far more
// than the bound's own FP32 error plus the screen's (2e-6), stays below the
// screening threshold: the screen would then reject it as well, so the set
// of combinations that reach the exact MI is unchanged.
__device__ __forceinline__ bool bound_passes(float bound, float tau, float delta)
{
    return fmaf(bound, 1.0001f, 4e-6f) >= tau - delta;
}

// p*ln(p) in FP64 for p > 0, else 0 (kept out of line: it is only reached for
// the few combinations that pass the FP32 screen).
__device__ __noinline__ double plogp(double p)
{
#pragma clang fp contract(off)
    return p > 0.0 ? p * log(p) : 0.0;
}

// Exact MI: H(X) + H(Y) - H(X,Y) in FP64 from the integer counts, summed in
// cell order with no fused multiply-add, so that the value depends only on
// the counts (not on tiling, batching or launch shape).
// The running sums continue over CELLS consecutive cells (a table split over
// lanes in cell order is one chain through them).
// Cells from cell(x, n0, n1) (integer counts).
template <int CELLS, class F>
__device__ __forceinline__ void mi_exact_part_fn(F &&cell, double n, double &hx, double &hall)
{
#pragma clang fp contract(off)
#pragma unroll
    for (int x = 0; x < CELLS; ++x) {
        uint32_t n0, n1;
        cell(x, n0, n1);
        const double pc = (double)n0 / n, pt = (double)n1 / n, pa = pc + pt;
        hall -= plogp(pc);
        hall -= plogp(pt);
        hx -= plogp(pa);
    }
}

__device__ __forceinline__ bool better(float ma, uint64_t ca, float mb, uint64_t cb)
{
    return ma > mb || (ma == mb && ca < cb);
}

// Wave-aggregated push of candidates (all 64 lanes must call).
__device__ __forceinline__ void push_candidates(bool want, float mi, uint64_t combo,
                                                const ScanParams &P, TopState *st)
{
    const uint64_t m = __ballot(want);
    if (m == 0) return;
    const int lane = threadIdx.x & 63;
    const int leader = __ffsll((long long)m) - 1;
    uint32_t base = 0;
    if (lane == leader) base = atomicAdd(&st->cand_count, (uint32_t)__popcll(m));
    base = __shfl(base, leader);
    if (want) {
        const uint32_t idx = base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
        if (idx < P.cand_cap) {
            Cand c;
            c.mi = mi;
            c.tag = P.tag;
            c.combo = combo;
            P.cand[idx] = c;
        } else {
            atomicOr(&st->overflow, 1u);
        }
    }
}

__device__ __forceinline__ double readlane64(double v, int lane)
{
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(u >> 32), lane);
    return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

// The exact MI of lane src's table by the whole wave: lane 3 x + k computes
// term k of cell x (cases, controls, both; 21 cells at a time), then every lane
// runs the same chain over them in cell order, so the value is
// mi_exact_part_fn's bit for bit.  One logarithm deep for 21 cells, a third of
// what a lane per cell takes.  cell(x, n0, n1) gives the calling lane's own
// counts.
template <int CELLS, class F>
__device__ __forceinline__ double mi_exact_wave(F &&cell, int src, double n, double hy)
{
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63, mine = lane / 3, k = lane - 3 * mine;
    double hx = 0.0, hall = 0.0;
#pragma unroll
    for (int base = 0; base < CELLS; base += 21) {
        const int m = CELLS - base < 21 ? CELLS - base : 21;
        uint32_t c = 0, t = 0;
#pragma unroll
        for (int x = 0; x < m; ++x) {
            uint32_t n0, n1;
            cell(base + x, n0, n1);
            n0 = (uint32_t)__builtin_amdgcn_readlane((int)n0, src);
            n1 = (uint32_t)__builtin_amdgcn_readlane((int)n1, src);
            if (mine == x) c = n0, t = n1;
        }
        const double pc = (double)c / n, pt = (double)t / n, pa = pc + pt;
        const double term = plogp(k == 0 ? pc : k == 1 ? pt : pa);
#pragma unroll 1
        for (int x = 0; x < 3 * m; x += 3) {
            hall -= readlane64(term, x);
            hall -= readlane64(term, x + 1);
            hx -= readlane64(term, x + 2);
        }
    }
    return hx + hy - hall;
}

// Exact MI and the key test of the lanes that `need` them, and the push (all
// 64 lanes call).  A lane alone takes 3 CELLS FP64 logarithms one after the
// other, the wave three per table: up to kExactWave lanes are taken one by one
// by the wave, more of them side by side.  What a small search waits for:
// pairs of 1,000 x 4,000, scan 106 -> 47 us; triples of 151 x 1,203, 145 -> 73.
constexpr int kExactWave = 12;
template <int CELLS, class F, class K>
__device__ __forceinline__ void exact_push(bool need, F &&cell, K &&key, float tau, uint64_t tau_combo,
                                           const ScanParams &P, TopState *st)
{
    const uint64_t mask = __ballot(need);
    if (mask == 0) return;
    const int lane = threadIdx.x & 63;
    float mf = 0.0f;
    if (__popcll(mask) <= kExactWave) {
        for (uint64_t m = mask; m; m &= m - 1) {
            const int src = __builtin_ctzll(m);
            const float v = (float)mi_exact_wave<CELLS>(cell, src, P.n64, P.hy64);
            if (lane == src) mf = v;
        }
    } else if (need) {
#pragma clang fp contract(off)
        double hx = 0.0, hall = 0.0;
        mi_exact_part_fn<CELLS>(cell, P.n64, hx, hall);
        mf = (float)(hx + P.hy64 - hall);
    }
    uint64_t combo = ~0ull;
    bool want = false;
    if (need) {
        combo = key();
        want = better(mf, combo, tau, tau_combo);
    }
    push_candidates(want, mf, combo, P, st);
}

// exact_push on tables held as two arrays (integers, or FP32 integers).
template <int CELLS, class T, class K>
__device__ __forceinline__ void exact_push_arrays(bool need, const T *a0, const T *a1, K &&key, float tau,
                                                  uint64_t tau_combo, const ScanParams &P, TopState *st)
{
    exact_push<CELLS>(
        need,
        [&](int x, uint32_t &n0, uint32_t &n1) __attribute__((always_inline)) {
            n0 = (uint32_t)a0[x];
            n1 = (uint32_t)a1[x];
        },
        key, tau, tau_combo, P, st);
}

// Whether a valid combination passes the bound (always, without it).
template <int CELLS, class T>
__device__ __forceinline__ bool bound_ok(const T *a0, const T *a1, float tau, const ScanParams &P)
{
    return !P.bounded || bound_passes(mi_bound<CELLS>(a0, a1, P.frac_c, P.chi_scale), tau, P.delta);
}

// Epilogue shared by every scan kernel: screening MI, exact MI for the
// survivors, key test against the current N-th best, push.  key() gives the
// combination's key; it is only called for the few combinations that reach
// the exact MI.
template <int CELLS, class T, class K>
__device__ __forceinline__ void score_and_push(bool valid, const T *a0, const T *a1, K &&key, float tau,
                                               uint64_t tau_combo, const ScanParams &P, TopState *st)
{
    const bool need = valid && bound_ok<CELLS>(a0, a1, tau, P) &&
                      mi_screen<CELLS>(a0, a1, P.hy, P.inv_n) >= tau - P.delta;
    exact_push_arrays<CELLS>(need, a0, a1, key, tau, tau_combo, P, st);
}

// Uniform lookup of prefix j < j1: rank -> SNP indices, or an empty marker.
template <int M>
__device__ __forceinline__ bool prefix_at(const ScanParams &P, int n, int64_t j, int64_t j1, int *pre)
{
    if (j >= j1) return false;
    const uint64_t rank = (uint64_t)P.offset + (uint64_t)j * (uint64_t)P.step;
    if (rank >= P.total_prefixes) return false;
    unrank(rank, n, M, P.binom, pre);
    return true;
}

// Either the normal epilogue, or (threshold sampling pass) one count in the
// workgroup's LDS histogram of screening MI values.
template <bool HIST, int CELLS, class K>
__device__ __forceinline__ void score_or_sample(bool valid, const uint32_t *a0, const uint32_t *a1, K &&key,
                                                float tau, uint64_t tau_combo, const ScanParams &P, TopState *st,
                                                uint32_t *lds_hist)
{
    if constexpr (HIST) {
        if (valid) atomicAdd(&lds_hist[hist_bin(mi_screen<CELLS>(a0, a1, P.hy, P.inv_n))], 1u);
    } else {
        score_and_push<CELLS>(valid, a0, a1, key, tau, tau_combo, P, st);
    }
}

template <bool HIST>
__device__ __forceinline__ void hist_begin(uint32_t *lds_hist)
{
    if constexpr (HIST) {
        for (int b = threadIdx.x; b < kHistBins; b += blockDim.x) lds_hist[b] = 0;
        __syncthreads();
    }
}

template <bool HIST>
__device__ __forceinline__ void hist_end(uint32_t *lds_hist, uint32_t *hist)
{
    if constexpr (HIST) {
        __syncthreads();
        for (int b = threadIdx.x; b < kHistBins; b += blockDim.x)
            if (lds_hist[b]) atomicAdd(&hist[b], lds_hist[b]);
    }
}

}  // namespace fiu
