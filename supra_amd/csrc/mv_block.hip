// Minimum variance for well-loaded systems: the per-sample covariances are
// accumulated on the FP64 matrix cores and every system is factorised by 16
// lanes.
//
// Same per-sample mathematics as mv_kernels.hip (which keeps the forms this
// one does not have: FP64 refinement of weakly loaded systems and conjugate
// gradients); the references are the same: RxBeamformerMV.cu:44-113 apertures
// and sub-arrays, :115-195 covariance, :197-228 temporal sum, :239-305
// loading, :558-586 solve, :307-378 output.
//
// One workgroup takes nb consecutive output depths of one scanline:
//
//   1. stage x[channel][tau] of the nb depths and their +-T halo in LDS, find
//      the apertures (mv_stage.hpp);
//   2. the window sums R~(t) = sum_{|tau-t| <= T} sum_k x_k x_k^T of the nb
//      outputs, as 16 x 16 blocks of the lower triangle with
//      v_mfma_f64_16x16x4 (products of floats are exact in FP64).  The
//      outputs go in sub-blocks of at most 2T + 1: their windows share a core
//      of samples, so the accumulator is filled with the core, then extended
//      downwards (one sample per output, stored as it grows) and a second one
//      upwards (added to what was stored).  No sum is ever subtracted from,
//      so a weak window next to a strong echo keeps its precision, and about
//      2 evaluations per output replace the 2T + 1 additions of stored
//      covariances;
//   3. sixteen lanes per system, row 16 r + q in slot r of lane q: diagonal
//      loading, then a right-looking Cholesky factorisation whose column is
//      broadcast inside the FMAs (DPP row_newbcast), FP64 pivots and
//      diagonal, with the two right-hand sides 1 and the sub-array sums xs as
//      extra columns.  With z = G^-1 1 and u = G^-1 xs the output is
//      xs^T R~^-1 1 / 1^T R~^-1 1 = u.z / z.z: no backward substitution and
//      no factor kept.
//
// Bound by the FP64 pipe at L = 32: the matrix instructions (26 % of the time)
// and the vector instructions (49 %) of the waves of a SIMD add up.  At L = 64
// the matrices fill the LDS and one wave per SIMD waits for itself.
// 128 x 2080 samples, L = 32, T = 5: 0.66 ms against 2.01 ms of
// mv_kernels.hip; pre-delay + 128 x 1750 samples, L = 64: 0.90 ms against
// 9.51 ms (in both, windows of few terms take the short way below);
// relative error of the image against FP64 1.3e-6 against 2.1e-6.
// Summing the blocks off the first column by differences along the block
// diagonals (fewer matrix instructions, but longer serial chains) and running
// the two accumulations of a sub-block side by side were slower (2.49 and
// 2.58 ms at L = 64).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdint>

#include "bf_internal.hpp"
#include "das_device.hpp"
#include "mv_launch.hpp"
#include "mv_stage.hpp"

namespace supra_amd {
namespace {

typedef double double4v __attribute__((ext_vector_type(4)));

// Waves per workgroup: the matrix blocks are dealt to the waves (3 blocks for
// 32 rows, 10 for 64), for 16 rows the sub-blocks of outputs are.
template <int LMAX> struct Cfg {
    static constexpr int kBlocks = LMAX / 16;
    static constexpr int kWaves = LMAX == 32 ? 3 : 4;
    static constexpr int kThreads = 64 * kWaves;
    // floats of one stored lower triangle: full 16 x 16 blocks below the
    // diagonal, 160 floats per diagonal block (its 4-column chunks without
    // the rows above them)
    static constexpr int kMatrix = kBlocks * 160 + kBlocks * (kBlocks - 1) / 2 * 256;
};

// First float of block (r, c), c <= r.  Blocks are stored by chunks of 4
// columns, [chunk][row][4], so that 16 rows of a chunk are 256 contiguous
// bytes for the solver's 16-byte reads.
__device__ constexpr int block_at(int r, int c) { return r * 160 + r * (r - 1) / 2 * 256 + c * 256; }
// First float of a diagonal block's chunk (rows 4 chunk .. 15).
__device__ constexpr int diag_chunk(int chunk) { return chunk == 0 ? 0 : (chunk == 1 ? 64 : (chunk == 2 ? 112 : 144)); }

struct Gram {
    const float* xs;
    const uint32_t* code;  // per staged sample: first | active sub-arrays << 10, or 0 for one left out
    const float* mean;     // [h][16 kBlocks], nullptr without mean removal
    float* mats;
    int rs, mean_stride, matrix;
    int T, n_d, h_lo;
    uint32_t zero_row;     // first of 16 kBlocks + 4 zeros in xs: row 0's padding
    uint32_t codes;        // lane l: code[l] (the first 64 samples without a wait for LDS)
    __device__ inline uint32_t code_of(int h) const {
        return static_cast<uint32_t>(h < 64 ? __builtin_amdgcn_readlane(static_cast<int>(codes), h)
                                            : __builtin_amdgcn_readfirstlane(static_cast<int>(code[h])));
    }
};

__device__ inline double4v mfma64(float a, float b, double4v c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(a), static_cast<double>(b), c, 0, 0, 0);
}

// The matrix blocks (row block, column block) that one wave accumulates;
// chosen so that the blocks of a wave share operands.
template <int LMAX, int WAVE> struct Deal;
template <int WAVE> struct Deal<16, WAVE> {
    static constexpr int n = 1, r[3] = {0, 0, 0}, c[3] = {0, 0, 0};
};
template <> struct Deal<32, 0> { static constexpr int n = 1, r[3] = {0, 0, 0}, c[3] = {0, 0, 0}; };
template <> struct Deal<32, 1> { static constexpr int n = 1, r[3] = {1, 0, 0}, c[3] = {0, 0, 0}; };
template <> struct Deal<32, 2> { static constexpr int n = 1, r[3] = {1, 0, 0}, c[3] = {1, 0, 0}; };
template <> struct Deal<64, 0> { static constexpr int n = 3, r[3] = {0, 1, 1}, c[3] = {0, 0, 1}; };
template <> struct Deal<64, 1> { static constexpr int n = 3, r[3] = {2, 2, 2}, c[3] = {0, 1, 2}; };
template <> struct Deal<64, 2> { static constexpr int n = 2, r[3] = {3, 3, 0}, c[3] = {0, 1, 0}; };
template <> struct Deal<64, 3> { static constexpr int n = 2, r[3] = {3, 3, 0}, c[3] = {2, 3, 0}; };

// Accumulators of a wave's blocks.  Matrix-core operands: lane = (row or
// column, term); D[j][i] holds row i of the block in lane % 16 and column
// j = lane / 16 + 4 v in register v.
template <typename D>
struct Blocks {
    double4v acc[D::n];
    __device__ inline void clear() {
#pragma unroll
        for (int b = 0; b < D::n; b++) acc[b] = double4v{0.0, 0.0, 0.0, 0.0};
    }
    // acc += the covariance of sample tau: 16 terms at a time, all loads of a
    // group before its first matrix instruction, then 4; the last step reads
    // up to 3 terms past the aperture (in the zeroed padding) and masks them.
    __device__ inline void add(const Gram& g, int tau) {
        const int h = tau - g.h_lo;
        const uint32_t code = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(g.code[h])));
        const int kact = static_cast<int>(code >> 10);
        const int lane = static_cast<int>(threadIdx.x % 64), i = lane % 16, kq = lane / 16;
        const float* x = g.xs + h * g.rs + static_cast<int>(code & 1023u) + i + kq;
        int k = 0;
        for (; k + 16 <= kact; k += 16, x += 16) {
            float v[4][4];       // [step][row block] (unused ones drop out)
#pragma unroll
            for (int u = 0; u < 4; u++)
#pragma unroll
                for (int r = 0; r < 4; r++) v[u][r] = used(r) ? x[4 * u + 16 * r] : 0.0f;
#pragma unroll
            for (int u = 0; u < 4; u++)
#pragma unroll
                for (int b = 0; b < D::n; b++) acc[b] = mfma64(v[u][D::c[b]], v[u][D::r[b]], acc[b]);
        }
#pragma unroll 1
        for (; k < kact; k += 4, x += 4) {
            const bool in = k + kq < kact;
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; r++) v[r] = used(r) ? x[16 * r] : 0.0f;
#pragma unroll
            for (int b = 0; b < D::n; b++) acc[b] = mfma64(in ? v[D::c[b]] : 0.0f, v[D::r[b]], acc[b]);
        }
        if (g.mean && kact) {   // - K m m^T
            const float* mu = g.mean + h * g.mean_stride + i;
#pragma unroll
            for (int b = 0; b < D::n; b++)
                acc[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                    kq == 0 ? -static_cast<double>(kact) * static_cast<double>(mu[16 * D::c[b]]) : 0.0,
                    static_cast<double>(mu[16 * D::r[b]]), acc[b], 0, 0, 0);
        }
    }
    static constexpr bool used(int r) {
        for (int b = 0; b < D::n; b++)
            if (D::r[b] == r || D::c[b] == r) return true;
        return false;
    }
    // Stores (ADD: adds) the blocks to output matrix o.
    template <bool ADD>
    __device__ inline void store(const Gram& g, int o) const {
        const int lane = static_cast<int>(threadIdx.x % 64), i = lane % 16, e = lane / 16;
#pragma unroll
        for (int b = 0; b < D::n; b++) {
            const bool diagonal = D::r[b] == D::c[b];
            float* blk = g.mats + o * g.matrix + block_at(D::r[b], D::c[b]);
#pragma unroll
            for (int v = 0; v < 4; v++) {
                float* p = diagonal ? blk + diag_chunk(v) + (i - 4 * v) * 4 + e : blk + v * 64 + i * 4 + e;
                const float x = static_cast<float>(acc[b][v]);
                if (!diagonal || i >= 4 * v) *p = ADD ? *p + x : x;
            }
        }
    }
};

// Window sums of the outputs [ta, ta + n) into matrices o, o + 1, ...; n <=
// 2T + 1: the core of samples common to all windows and, output by output
// downwards, what lies below it; then what lies above it, upwards.
template <typename D>
__device__ inline void window_sums(const Gram& g, int ta, int n, int o) {
    Blocks<D> s;
    s.clear();
    for (int tau = max(0, ta + n - 1 - g.T); tau <= min(g.n_d - 1, ta + g.T); tau++) s.add(g, tau);
    s.template store<false>(g, o + n - 1);
    for (int j = n - 2; j >= 0; j--) {
        if (ta + j - g.T >= 0) s.add(g, ta + j - g.T);
        s.template store<false>(g, o + j);
    }
    s.clear();
    for (int j = 1; j < n; j++) {
        if (ta + j + g.T < g.n_d) s.add(g, ta + j + g.T);   // else the window ends with the last sample
        s.template store<true>(g, o + j);
    }
}

template <int LMAX>
__device__ inline void all_window_sums(const Gram& g, int t0, int n_out, int sub, int wave) {
    if constexpr (LMAX == 16) {
        for (int b = wave * sub; b < n_out; b += Cfg<LMAX>::kWaves * sub)
            window_sums<Deal<16, 0>>(g, t0 + b, min(sub, n_out - b), b);
    } else {
        for (int b = 0; b < n_out; b += sub) {
            const int ta = t0 + b, n = min(sub, n_out - b);
            if (wave == 0) window_sums<Deal<LMAX, 0>>(g, ta, n, b);
            else if (wave == 1) window_sums<Deal<LMAX, 1>>(g, ta, n, b);
            else if (wave == 2) window_sums<Deal<LMAX, 2>>(g, ta, n, b);
            else if constexpr (LMAX == 64) window_sums<Deal<64, 3>>(g, ta, n, b);
        }
    }
}

// ---- the solver: 16 lanes per system -------------------------------------------

// a[k] -= (lane k's lk of this row of 16 lanes) * l for k = START .. 15, one
// v_fmac_f32_dpp row_newbcast each.  The leading s_nop covers the two wait
// states between a VALU write of lk and its DPP read.
#define SUPRA_FM(K) "v_fmac_f32_dpp %" #K ", %16, -%17 row_newbcast:" #K " row_mask:0xf bank_mask:0xf\n\t"
#define SUPRA_FM_15 SUPRA_FM(15)
#define SUPRA_FM_14 SUPRA_FM(14) SUPRA_FM_15
#define SUPRA_FM_13 SUPRA_FM(13) SUPRA_FM_14
#define SUPRA_FM_12 SUPRA_FM(12) SUPRA_FM_13
#define SUPRA_FM_11 SUPRA_FM(11) SUPRA_FM_12
#define SUPRA_FM_10 SUPRA_FM(10) SUPRA_FM_11
#define SUPRA_FM_9 SUPRA_FM(9) SUPRA_FM_10
#define SUPRA_FM_8 SUPRA_FM(8) SUPRA_FM_9
#define SUPRA_FM_7 SUPRA_FM(7) SUPRA_FM_8
#define SUPRA_FM_6 SUPRA_FM(6) SUPRA_FM_7
#define SUPRA_FM_5 SUPRA_FM(5) SUPRA_FM_6
#define SUPRA_FM_4 SUPRA_FM(4) SUPRA_FM_5
#define SUPRA_FM_3 SUPRA_FM(3) SUPRA_FM_4
#define SUPRA_FM_2 SUPRA_FM(2) SUPRA_FM_3
#define SUPRA_FM_1 SUPRA_FM(1) SUPRA_FM_2
#define SUPRA_FM_0 SUPRA_FM(0) SUPRA_FM_1

template <int START>
__device__ __attribute__((always_inline)) inline void fmac16(float* a, float lk, float l) {
#define SUPRA_FM_CASE(S)                                                                                               \
    if constexpr (START == S)                                                                                         \
        asm("s_nop 1\n\t" SUPRA_FM_##S                                                                                \
            : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5]), "+v"(a[6]), "+v"(a[7]),         \
              "+v"(a[8]), "+v"(a[9]), "+v"(a[10]), "+v"(a[11]), "+v"(a[12]), "+v"(a[13]), "+v"(a[14]), "+v"(a[15])    \
            : "v"(lk), "v"(l))
    SUPRA_FM_CASE(0);
    SUPRA_FM_CASE(1);
    SUPRA_FM_CASE(2);
    SUPRA_FM_CASE(3);
    SUPRA_FM_CASE(4);
    SUPRA_FM_CASE(5);
    SUPRA_FM_CASE(6);
    SUPRA_FM_CASE(7);
    SUPRA_FM_CASE(8);
    SUPRA_FM_CASE(9);
    SUPRA_FM_CASE(10);
    SUPRA_FM_CASE(11);
    SUPRA_FM_CASE(12);
    SUPRA_FM_CASE(13);
    SUPRA_FM_CASE(14);
    SUPRA_FM_CASE(15);
#undef SUPRA_FM_CASE
}

// Lane N's value in each row of 16 lanes.
template <int N> __device__ inline float row_bcast(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + N, 0xf, 0xf, true));
}

// Sum over each row of 16 lanes, in every lane (DPP row_ror 8, 4, 2, 1).
__device__ inline float row_sum(float v) {
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xf, 0xf, true));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xf, 0xf, true));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x122, 0xf, 0xf, true));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x121, 0xf, 0xf, true));
    return v;
}

// 1/sqrt in FP64: hardware estimate and one Newton step (NaN for v <= 0)
__device__ inline double rsqrt64(double v) {
    const double r = __builtin_amdgcn_rsq(v);
    return r * (1.5 - (0.5 * v) * (r * r));
}

template <int LMAX> struct System {
    static constexpr int kB = LMAX / 16;
    float a[kB][LMAX];       // row 16 r + q in slot r; entries beyond column 16 r + 15 unused
    double dd[kB];           // running diagonal of the slot's row
    float b1[kB], b2[kB];    // right-hand sides
    float invg;              // 1 / pivot of the next step
};

// 1/sqrt of row J's diagonal, in every lane of the system.
template <int LMAX, int J>
__device__ __attribute__((always_inline)) inline float inverse_pivot(const System<LMAX>& s) {
    return row_bcast<J % 16>(static_cast<float>(rsqrt64(s.dd[J / 16])));
}

// Elimination step J: column J scaled by 1/pivot, then subtracted from the
// rows below.  Rows at or above the pivot take a zero multiplier; entries
// right of a row's own column are its unused upper part.  The diagonals do
// not wait for the rows' updates, so the next pivot's FP64 chain runs beside
// them.
template <int LMAX, int J>
__device__ __attribute__((always_inline)) inline void eliminate(System<LMAX>& s, int q) {
    constexpr int rj = J / 16, qj = J % 16, kB = LMAX / 16;
    const float invg = s.invg;
    float l[kB];
#pragma unroll
    for (int r = rj; r < kB; r++) {
        l[r] = s.a[r][J] * invg;
        if (r == rj) l[r] = q > qj ? l[r] : 0.0f;
        s.dd[r] = fma(-static_cast<double>(l[r]), static_cast<double>(l[r]), s.dd[r]);
    }
    if constexpr (J + 1 < LMAX) s.invg = inverse_pivot<LMAX, J + 1>(s);
    const float z1 = row_bcast<qj>(s.b1[rj] * invg), z2 = row_bcast<qj>(s.b2[rj] * invg);
#pragma unroll
    for (int r = rj; r < kB; r++) {
        if constexpr (qj < 15) fmac16<(qj + 1) % 16>(&s.a[r][16 * rj], l[rj], l[r]);
#pragma unroll
        for (int c = rj + 1; c <= r; c++) fmac16<0>(&s.a[r][16 * c], l[c], l[r]);
        // (a select, not the zero multiplier: a step past the system's last
        // row may have a NaN pivot)
        const float n1 = fmaf(-l[r], z1, s.b1[r]), n2 = fmaf(-l[r], z2, s.b2[r]);
        s.b1[r] = r > rj || q > qj ? n1 : s.b1[r];
        s.b2[r] = r > rj || q > qj ? n2 : s.b2[r];
    }
}

// Steps J .. LMAX-1; steps past the wave's largest system are left out four
// at a time (they would change unused rows only).
template <int LMAX, int J>
__device__ __attribute__((always_inline)) inline void eliminate_from(System<LMAX>& s, int q, int nmax) {
    if constexpr (J < LMAX) {
        if (J < nmax) {   // uniform
            eliminate<LMAX, J>(s, q);
            eliminate<LMAX, J + 1>(s, q);
            eliminate<LMAX, J + 2>(s, q);
            eliminate<LMAX, J + 3>(s, q);
        }
        eliminate_from<LMAX, J + 4>(s, q, nmax);
    }
}

// ---- few terms: the system in the space of the terms ---------------------------

// Where the apertures are hardly longer than the sub-arrays, a window holds
// only a few sub-array vectors: with T = 5 and one sub-array per sample, 11.
// For R~ = delta I + X X^T with the M <= 15 vectors x as columns of X,
//     R~^-1 1 = (1 - X y) / delta,   (delta I + X^T X) y = X^T 1,
// so with the Cholesky factor G of the M x M matrix, w = G^-1 X^T 1 and
// u = G^-1 c (c marks the columns of the output's own sample, xs = X c)
//     xs^T R~^-1 1 = c^T y = u.w,   1^T R~^-1 1 = (n - w.w) / delta.
// Everything is FP64: X^T X comes from the matrix cores with the ones as 16th
// column (its products are X^T 1), 16 lanes factorise a system, and n - w.w is
// at least n delta / (delta + trace), 1e-4 n for the loadings that come here.
constexpr int kTerms = 15;

template <int N> __device__ inline double row_bcast(double v) {
    const uint64_t b = __double_as_longlong(v);
    const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(b), 0x150 + N, 0xf, 0xf, true));
    const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(b >> 32), 0x150 + N, 0xf, 0xf, true));
    return __longlong_as_double(static_cast<int64_t>(static_cast<uint64_t>(hi) << 32 | lo));
}
template <int CTRL> __device__ inline double row_ror(double v) {
    const uint64_t b = __double_as_longlong(v);
    const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(b), CTRL, 0xf, 0xf, true));
    const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(b >> 32), CTRL, 0xf, 0xf, true));
    return __longlong_as_double(static_cast<int64_t>(static_cast<uint64_t>(hi) << 32 | lo));
}
__device__ inline double row_sum(double v) {
    v += row_ror<0x128>(v);
    v += row_ror<0x124>(v);
    v += row_ror<0x122>(v);
    v += row_ror<0x121>(v);
    return v;
}

// a -= (lane C's lk of this row of 16 lanes) * l.  The s_nop covers the wait
// states between a VALU write of lk and its DPP read.
template <int C> __device__ inline void fmac_bcast(double& a, double lk, double l) {
    asm("s_nop 1\n\tv_fmac_f64_dpp %0, %1, -%2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(a) : "v"(lk), "v"(l), "n"(C));
}

template <bool HALF> __device__ inline void swap_rows(double& x, double& y) {
    uint64_t a = __double_as_longlong(x), b = __double_as_longlong(y);
    uint32_t a0 = static_cast<uint32_t>(a), a1 = static_cast<uint32_t>(a >> 32);
    uint32_t b0 = static_cast<uint32_t>(b), b1 = static_cast<uint32_t>(b >> 32);
    const auto lo = HALF ? __builtin_amdgcn_permlane32_swap(a0, b0, false, false) : __builtin_amdgcn_permlane16_swap(a0, b0, false, false);
    const auto hi = HALF ? __builtin_amdgcn_permlane32_swap(a1, b1, false, false) : __builtin_amdgcn_permlane16_swap(a1, b1, false, false);
    x = __longlong_as_double(static_cast<int64_t>(static_cast<uint64_t>(hi[0]) << 32 | lo[0]));
    y = __longlong_as_double(static_cast<int64_t>(static_cast<uint64_t>(hi[1]) << 32 | lo[1]));
}

// Row q = lane % 16 of the system of lane / 16: columns 0 .. 14 and X^T 1.
struct TermSystem {
    double a[16];
    double own;         // 1 / pivot of the lane's own row
    double b1, b2;      // right-hand sides X^T 1 and c
};

template <int J, int C>
__device__ __attribute__((always_inline)) inline void eliminate_terms(TermSystem& s, double l) {
    if constexpr (C < kTerms) {
        fmac_bcast<C>(s.a[C], l, l);
        eliminate_terms<J, C + 1>(s, l);
    }
}
template <int J>
__device__ __attribute__((always_inline)) inline void factor_terms(TermSystem& s, int q, int terms) {
    if constexpr (J < kTerms) {
        if (J < terms) {   // uniform
            const double inv = rsqrt64(row_bcast<J>(s.a[J]));
            if (q == J) s.own = inv;
            const double l = q > J ? s.a[J] * inv : 0.0;
            const double z1 = row_bcast<J>(s.b1) * inv, z2 = row_bcast<J>(s.b2) * inv;
            s.b1 = fma(-l, z1, s.b1);
            s.b2 = fma(-l, z2, s.b2);
            eliminate_terms<J, J + 1>(s, l);
            factor_terms<J + 1>(s, q, terms);
        }
    }
}

// The outputs of the tile, if each of their windows has at most kTerms terms;
// false without any work otherwise.  One tile of 16 outputs of 64 rows takes
// 13 k cycles here and 75 to 98 k with window sums and 64 x 64 systems
// (pre-delay + 128 x 1750 samples, L = 64, T = 5: 0.95 ms against 2.00).
template <int LMAX>
__device__ inline bool solve_few_terms(const MvArgs& a, const Gram& g, const SampleMeta* meta, int t0, int n_out, float2* res,
                                       int wave) {
    const int lane = static_cast<int>(threadIdx.x % 64), q = lane % 16, e = lane / 16;
    if (g.mean || 2 * g.T + 1 > kTerms || n_out > 64) return false;
    // lane o looks at output o
    const int ht = t0 + min(lane, n_out - 1) - g.h_lo;
    const int lo = max(0, ht - g.T), hi = min(g.n_d - 1 - g.h_lo, ht + g.T);
    int terms = 0;
    bool bad = false, single = true;
#pragma unroll
    for (int j = 0; j < kTerms; j++) {
        const uint32_t own = g.code[min(lo + j, hi)] >> 10;    // sub-arrays of the sample; 0: a bad one
        if (lo + j <= hi) {
            terms += static_cast<int>(own);
            bad |= own == 0;
            single &= own == 1;
        }
    }
    const int n_rows = meta[ht].lt;
    if (__builtin_amdgcn_ballot_w64(terms > kTerms) != 0) return false;
    const uint64_t bad_outputs = __builtin_amdgcn_ballot_w64(bad);       // output 0
    const bool all_single = __builtin_amdgcn_ballot_w64(!single) == 0;   // one sub-array in every sample
    for (int o0 = wave * 4; o0 < n_out; o0 += 4 * Cfg<LMAX>::kWaves) {
        // column q of X for the four systems: where its samples are
        const float* x[4];
        int n[4], n_max = 0, m_max = 0;
        double mark = 0.0;      // c of the lane's own system (lane / 16)
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const int o = min(o0 + s, n_out - 1);    // a spare system repeats the last sample
            n[s] = __builtin_amdgcn_readlane(n_rows, o);
            n_max = max(n_max, n[s]);
            m_max = max(m_max, __builtin_amdgcn_readlane(terms, o));
            const int h1 = __builtin_amdgcn_readlane(hi, o);
            int at = static_cast<int>(g.zero_row), before = 0;      // unused columns read zeros
            if (all_single) {
                const int h = __builtin_amdgcn_readlane(lo, o) + q;
                if (h <= h1) {
                    at = h * g.rs + static_cast<int>(g.code[h] & 1023u);
                    if (e == s && t0 + o - g.h_lo == h) mark = 1.0;
                }
            } else for (int h = __builtin_amdgcn_readlane(lo, o); h <= h1; h++) {
                const uint32_t code = g.code_of(h);
                const int k = q - before, own = static_cast<int>(code >> 10);
                if (k >= 0 && k < own) {
                    at = h * g.rs + static_cast<int>(code & 1023u) + k;
                    if (e == s && t0 + o - g.h_lo == h) mark = 1.0;
                }
                before += own;
            }
            x[s] = g.xs + at + e;
        }
        double4v acc[4];
#pragma unroll
        for (int s = 0; s < 4; s++) acc[s] = double4v{0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
        for (int i0 = 0; i0 < n_max; i0 += 16) {
            float v[4][4];
#pragma unroll
            for (int s = 0; s < 4; s++)
#pragma unroll
                for (int u = 0; u < 4; u++) v[s][u] = x[s][i0 + 4 * u];
#pragma unroll
            for (int u = 0; u < 4; u++)
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    const float w = i0 + 4 * u + e < n[s] ? (q == kTerms ? 1.0f : v[s][u]) : 0.0f;
                    acc[s] = mfma64(w, w, acc[s]);
                }
        }
        // lane (e, q) holds columns e, e + 4, .. of row q of all four systems:
        // transposed to all columns of row q of system e
        TermSystem sys;
#pragma unroll
        for (int v = 0; v < 4; v++) {
            double c[4] = {acc[0][v], acc[1][v], acc[2][v], acc[3][v]};
            swap_rows<true>(c[0], c[2]);
            swap_rows<true>(c[1], c[3]);
            swap_rows<false>(c[0], c[1]);
            swap_rows<false>(c[2], c[3]);
#pragma unroll
            for (int k = 0; k < 4; k++) sys.a[4 * v + k] = c[k];
        }
        double diag = 0.0;
#pragma unroll
        for (int c = 0; c < kTerms; c++) diag = q == c ? sys.a[c] : diag;
        const int rows = e == 0 ? n[0] : (e == 1 ? n[1] : (e == 2 ? n[2] : n[3]));
        const double delta = row_sum(diag) / static_cast<double>(rows) * static_cast<double>(a.alpha);
#pragma unroll
        for (int c = 0; c < kTerms; c++) sys.a[c] = q == c ? sys.a[c] + delta : sys.a[c];
        sys.b1 = sys.a[kTerms];
        sys.b2 = mark;
        sys.own = 0.0;
        factor_terms<0>(sys, q, m_max);
        const bool term = q < m_max;
        const double w = term ? sys.b1 * sys.own : 0.0, u = term ? sys.b2 * sys.own : 0.0;
        const double ww = row_sum(w * w), uw = row_sum(u * w);
        if (q == 0 && o0 + e < n_out)
            res[o0 + e] = (bad_outputs >> (o0 + e)) & 1 ? make_float2(0.0f, 0.0f)
                                                        : make_float2(static_cast<float>(uw), static_cast<float>((static_cast<double>(rows) - ww) / delta));
    }
    return true;
}

// The samples of outputs [t0, t0 + n_out) of scanline s.
template <int LMAX>
__device__ inline void solve_outputs(const MvArgs& a, int t0, int n_out, int h_lo, const float* xs,
                                     const SampleMeta* meta, const float* mats, float2* res, int wave) {
    constexpr int kB = LMAX / 16;
    const int lane = static_cast<int>(threadIdx.x % 64), q = lane % 16;
    const int rs = static_cast<int>(a.rs);
    for (int o0 = wave * 4; o0 < n_out; o0 += 4 * Cfg<LMAX>::kWaves) {
        const int o = min(o0 + lane / 16, n_out - 1);    // a spare row of lanes repeats the last sample
        const int t = t0 + o, ht = t - h_lo;
        const SampleMeta m = meta[ht];
        const int n = m.lt;
        const float* mat = mats + o * Cfg<LMAX>::kMatrix;
        System<LMAX> s;
        float diag[kB], tr = 0.0f;
#pragma unroll
        for (int r = 0; r < kB; r++) {
#pragma unroll
            for (int c = 0; c < r; c++)
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const float4 x = *reinterpret_cast<const float4*>(mat + block_at(r, c) + v * 64 + q * 4);
                    float* p = &s.a[r][16 * c + 4 * v];
                    p[0] = x.x, p[1] = x.y, p[2] = x.z, p[3] = x.w;
                }
#pragma unroll
            for (int v = 0; v < 4; v++) {   // (rows above the chunk read its first row: unused entries)
                const float4 x = *reinterpret_cast<const float4*>(mat + block_at(r, r) + diag_chunk(v) + max(q - 4 * v, 0) * 4);
                float* p = &s.a[r][16 * r + 4 * v];
                p[0] = x.x, p[1] = x.y, p[2] = x.z, p[3] = x.w;
            }
            const int dc = q / 4;
            diag[r] = mat[block_at(r, r) + dc * 64 - (dc * (dc - 1) / 2) * 16 + (q % 4) * 4 + q % 4];
            tr += 16 * r + q < n ? diag[r] : 0.0f;
        }
        const float trace = row_sum(tr);
        const float delta = ((1.0f / static_cast<float>(n)) * trace) * a.alpha;
        int bad = 0;             // a window with a bad sample: output 0
        for (int h = max(0, ht - static_cast<int>(a.T)); h <= min(static_cast<int>(a.n_d) - 1 - h_lo, ht + static_cast<int>(a.T)); h++)
            bad |= meta[h].bad;
#pragma unroll
        for (int r = 0; r < kB; r++) {
            s.dd[r] = static_cast<double>(diag[r] + delta);
            s.b1[r] = 1.0f;
            s.b2[r] = 0.0f;
        }
        // sub-array sums x_i = sum_k x[f+k+i] (applyWeights, RxBeamformerMV.cu:342-376)
        const float* x = xs + ht * rs + m.first + q;
        int k = 0;
        for (; k + 8 <= m.kact; k += 8, x += 8) {
            float v[kB][8];
#pragma unroll
            for (int r = 0; r < kB; r++)
#pragma unroll
                for (int u = 0; u < 8; u++) v[r][u] = x[u + 16 * r];
#pragma unroll
            for (int u = 0; u < 8; u++)
#pragma unroll
                for (int r = 0; r < kB; r++) s.b2[r] += v[r][u];
        }
        for (; k < m.kact; k++, x++)
#pragma unroll
            for (int r = 0; r < kB; r++) s.b2[r] += x[16 * r];
        int nmax = n;
#pragma unroll
        for (int p = 16; p < 64; p += 16) nmax = max(nmax, __shfl_xor(nmax, p, 64));
        s.invg = inverse_pivot<LMAX, 0>(s);
        eliminate_from<LMAX, 0>(s, q, __builtin_amdgcn_readfirstlane(nmax));
        float zz = 0.0f, uz = 0.0f;
#pragma unroll
        for (int r = 0; r < kB; r++) {
            // row 16 r + q's right-hand sides and diagonal are final
            const float ginv = static_cast<float>(rsqrt64(s.dd[r]));
            const float z = s.b1[r] * ginv, u = s.b2[r] * ginv;
            if (16 * r + q < n) {
                zz = fmaf(z, z, zz);
                uz = fmaf(u, z, uz);
            }
        }
        zz = row_sum(zz);
        uz = row_sum(uz);
        if (q == 0 && o0 + lane / 16 < n_out) res[o] = make_float2(uz, bad ? 0.0f : zz);   // zz 0: output 0
    }
}

// The images' samples from (xs^T R~^-1 1, 1^T R~^-1 1): one lane each (the power
// and the division once per workgroup).
__device__ inline void write_outputs(const MvArgs& a, uint32_t scan, int t0, int n_out, int h_lo, const SampleMeta* meta,
                                     const float2* res) {
    if (static_cast<int>(threadIdx.x) < n_out) {
        const int t = t0 + static_cast<int>(threadIdx.x);
        const float2 r = res[threadIdx.x];
        const float kact = static_cast<float>(meta[t - h_lo].kact);
        float y = r.x / (r.y * powf(kact, a.p));
        if (!(fabsf(y) <= 1e7f) || r.y == 0.0f) y = 0.0f;
        y *= static_cast<float>(a.n_ch);
        const uint64_t at = static_cast<uint64_t>(t) * a.n_rx + scan;
        if (a.out_i16) static_cast<int16_t*>(a.out)[at] = clamp_out<int16_t>(y);
        else static_cast<float*>(a.out)[at] = clamp_out<float>(y);
    }
}

// Marks the samples whose covariance is not finite in single precision (e.g.
// from a -FLT_MAX pre-delayed value): by Cauchy-Schwarz those with a
// non-finite diagonal entry.  Only samples that find_apertures marked kHuge
// are looked at.  Also packs what the covariance needs of each sample.
template <int LMAX>
__device__ inline void find_bad(const MvArgs& a, const float* xs, const float* mean, int H, SampleMeta* meta, uint32_t* code) {
    constexpr int kWaves = Cfg<LMAX>::kWaves;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / 64));
    const int lane = static_cast<int>(threadIdx.x % 64);
    const int rs = static_cast<int>(a.rs);
    for (int h0 = 0; h0 < H; h0 += 64) {
        const int hl = h0 + lane;
        const SampleMeta ml = hl < H ? meta[hl] : SampleMeta{0, 0, 0, 0};
        if (wave == 0 && hl < H && ml.bad == 0) code[hl] = static_cast<uint32_t>(ml.first) | static_cast<uint32_t>(ml.kact) << 10;
        for (uint64_t left = __builtin_amdgcn_ballot_w64(ml.bad != 0); left != 0; left &= left - 1) {
            const int h = h0 + __builtin_ctzll(left);
            if (h % kWaves != wave) continue;
            const SampleMeta m = meta[h];
            double r = 0.0;
            if (lane < m.lt) {
                for (int k = 0; k < m.kact; k++) {
                    const double x = static_cast<double>(xs[h * rs + m.first + k + lane]);
                    r = fma(x, x, r);
                }
                if (mean) {
                    const double mu = static_cast<double>(mean[h * LMAX + lane]);
                    r -= static_cast<double>(m.kact) * mu * mu;
                }
            }
            const uint64_t over = __ballot(!(fabsf(static_cast<float>(r)) <= FLT_MAX));
            if (lane == 0) {
                meta[h].bad = over != 0 ? 1 : 0;
                code[h] = over != 0 ? 0u : static_cast<uint32_t>(m.first) | static_cast<uint32_t>(m.kact) << 10;
            }
        }
    }
}

template <typename InT, int LMAX, bool FUSED>
__device__ inline void mv_block_tile(const MvArgs& a, const float* lut, uint32_t scan, uint32_t tile, unsigned char* lds) {
    constexpr int kThreads = Cfg<LMAX>::kThreads;
    float* xs = reinterpret_cast<float*>(lds);
    SampleMeta* meta = reinterpret_cast<SampleMeta*>(lds + a.off_meta);
    float* mean = a.means ? reinterpret_cast<float*>(lds + a.off_mean) : nullptr;
    float* mats = reinterpret_cast<float*>(lds + a.off_r);
    float2* res = reinterpret_cast<float2*>(lds + a.off_wave);
    const uint32_t t0 = tile * a.tile, t1 = min(t0 + a.tile, a.n_d);
    const uint32_t h_lo = t0 >= a.T ? t0 - a.T : 0;
    const int H = static_cast<int>(min(a.n_d - 1, t1 - 1 + a.T) - h_lo + 1);
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / 64));

    if (FUSED) stage_delayed<InT, kThreads>(a, lut, scan, h_lo, H, xs, lds);
    else stage_read<InT, kThreads>(a, scan, h_lo, H, xs);
    find_apertures<kThreads, true>(a, xs, H, meta);
    __syncthreads();
    if (mean) {
        for (int idx = threadIdx.x; idx < H * LMAX; idx += kThreads) {
            const int h = idx / LMAX, i = idx % LMAX;
            const SampleMeta m = meta[h];
            float acc = 0.0f;
            if (i < m.lt) {
                for (int k = 0; k < m.kact; k++) acc += xs[h * a.rs + m.first + k + i];
                acc = acc / static_cast<float>(m.kact);
            }
            mean[idx] = acc;
        }
        __syncthreads();
    }
    uint32_t* code = reinterpret_cast<uint32_t*>(lds + a.off_code);
    find_bad<LMAX>(a, xs, mean, H, meta, code);
    __syncthreads();
    Gram g;
    g.xs = xs;
    g.code = code;
    g.mean = mean;
    g.mats = mats;
    g.rs = static_cast<int>(a.rs);
    g.mean_stride = LMAX;
    g.matrix = Cfg<LMAX>::kMatrix;
    g.T = static_cast<int>(a.T);
    g.n_d = static_cast<int>(a.n_d);
    g.h_lo = static_cast<int>(h_lo);
    const int n_out = static_cast<int>(t1 - t0);
    g.codes = code[min(static_cast<int>(threadIdx.x % 64), H - 1)];
    g.zero_row = a.n_ch;
    if (!solve_few_terms<LMAX>(a, g, meta, static_cast<int>(t0), n_out, res, wave)) {   // uniform
        all_window_sums<LMAX>(g, static_cast<int>(t0), n_out, static_cast<int>(a.sub), wave);
        __syncthreads();
        solve_outputs<LMAX>(a, static_cast<int>(t0), n_out, g.h_lo, xs, meta, mats, res, wave);
    }
    __syncthreads();
    write_outputs(a, scan, static_cast<int>(t0), n_out, g.h_lo, meta, res);
}

// Renumbers the workgroups as mv_logical_wg in mv_kernels.hip does: 32
// consecutive tiles (which share halos) on one XCD, XCDs rotated per round.
constexpr uint32_t kXcdTile = 32;

template <typename InT, int LMAX, bool FUSED>
__global__ __launch_bounds__(Cfg<LMAX>::kThreads) void mv_block_kernel(const MvArgs a) {
    extern __shared__ __align__(16) unsigned char lds[];
    const uint32_t b = blockIdx.x, xcd = b % 8u, local = b / 8u;
    const uint32_t round = local / kXcdTile, k = local % kXcdTile;
    const uint32_t wg = (round * 8u + (xcd + round) % 8u) * kXcdTile + k;
    if (wg >= a.n_rx * a.n_tiles) return;   // whole workgroup: the padded grid
    mv_block_tile<InT, LMAX, FUSED>(a, a.g.lut, wg / a.n_tiles, wg % a.n_tiles, lds);
}

// Persistent work queue over many frames (fused pre-delay), as mv_batch_kernel.
template <typename InT, int LMAX>
__global__ __launch_bounds__(Cfg<LMAX>::kThreads) void mv_block_batch_kernel(const MvBatchArgs b) {
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ uint32_t s_item;
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0) s_item = atomicAdd(b.sync.head, 1u);
        __syncthreads();
        const uint32_t item = s_item;
        if (item >= b.n_items) break;
        const uint32_t code = b.items[item];
        const MvBatchFrame& fr = b.frames[code >> 24];
        const MvArgs a = fr.a;     // scalars of the frame (the LUT is read from fr)
        const uint32_t local = code & 0xffffffu;
        mv_block_tile<InT, LMAX, true>(a, fr.a.g.lut, local / a.n_tiles, local % a.n_tiles, lds);
        __syncthreads();
        if (threadIdx.x == 0) {
            __threadfence();
            if (atomicAdd(&b.sync.done[fr.frame], 1u) + 1u == fr.n_items) b.sync.stamp[fr.frame] = wall_clock64();
        }
    }
}

size_t plan_lds(MvArgs& a, uint32_t lmax, uint32_t tile, bool with_delay) {
    const uint32_t H = tile + 2 * a.T, blocks = lmax / 16;
    a.tile = tile;
    size_t off = (static_cast<size_t>(H) * a.rs * 4 + 15) & ~static_cast<size_t>(15);
    a.off_meta = static_cast<uint32_t>(off);
    off += static_cast<size_t>(H) * sizeof(SampleMeta);
    a.off_mean = static_cast<uint32_t>(off);
    off += a.means ? static_cast<size_t>(H) * lmax * 4 : 0;
    a.off_wave = static_cast<uint32_t>(off);     // (u.z, z.z) of the outputs
    off += static_cast<size_t>(tile + 1) / 2 * 16;
    a.off_code = static_cast<uint32_t>(off);
    off += static_cast<size_t>(H + 3) / 4 * 16;
    a.off_r = static_cast<uint32_t>(off);
    // the pre-delay tables are only read before the matrices are written
    const size_t mats = static_cast<size_t>(tile) * (blocks * 160 + blocks * (blocks - 1) / 2 * 256) * 4;
    a.off_fused = static_cast<uint32_t>(off);
    const size_t fused = with_delay ? delay_table_floats(a.n_ch, H) * 4 : 0;
    return off + std::max(mats, fused);
}

}  // namespace

uint32_t mv_block_lmax(uint32_t L) { return L <= 16 ? 16 : (L <= 32 ? 32 : 64); }

bool mv_block_plan(MvArgs& a, size_t full, size_t budget, size_t* lds) {
    const uint32_t lmax = mv_block_lmax(a.L), w = 2 * a.T + 1;
    // zero padding: the last step and the unused rows read past the aperture
    a.rs = a.n_ch + lmax + 4;
    // Of the tiles that fit into all of the LDS, the one with the least modelled
    // time per output.  (Not of those that fit into the budget: the order of a
    // window's sum and the way that a tile is solved depend on the tile, so a
    // batch that plans for a share of the LDS would give other bits than the
    // single call, and smaller tiles do not pay: 6 of the uneven stream's
    // acquisitions with L = 64 take 31.8 ms with this one, 50 to 101 ms with what
    // fits two to four times.  For the same reason the pre-delay's tables count
    // in calls that do without.)  The time: subs (w - 1) + tile covariance evaluations on the busiest wave (9 matrix
    // instructions of 64 cycles with 32 rows, up to 51 with 64, fewer where the
    // aperture is small; with 16 rows the waves share the outputs) and rounds of
    // 4 systems per wave (one, but for tall tiles).
    // Tall tiles: with 16 rows a wave would sum w - 1 + 4 covariances for 4 outputs, so long
    // windows take 8, 12 or 16 outputs per wave, as far as the frame still makes
    // 384 workgroups (128 lines x 1024 depths, 128 channels, L = 4: T = 24 0.90 ms
    // with 64, 1.82 with 16, 1.08 in mv_kernels.hip; T = 8 474 us with 32, 713
    // with 16, 631 there; T = 3 410 and 403; 16 lines x 600 depths,
    // 32 channels, T = 5: 24.4 us with 32 and 23.3 with 16).
    const uint32_t waves = lmax == 32 ? 3 : 4;
    const double eval = lmax == 64 ? 1400.0 : (lmax == 32 ? 580.0 : 320.0);
    const double solve = lmax == 64 ? 23000.0 : (lmax == 32 ? 6000.0 : 2000.0);
    uint32_t longest = 4 * waves;
    if (lmax == 16 && a.T >= 4) {
        const uint32_t tall = a.T < 10 ? 32 : (a.n_ch < 160 && a.T < 20 ? 48 : 64);
        if (static_cast<uint64_t>(a.n_rx) * ((a.n_d + tall - 1) / tall) >= 384) longest = tall;
    }
    double best = 0;
    uint32_t pick = 0;
    for (uint32_t tile = 1; tile <= longest; tile++) {
        if (plan_lds(a, lmax, tile, true) > full) break;
        const uint32_t per_wave = lmax == 16 ? (tile + waves - 1) / waves : tile;
        const uint32_t subs = (per_wave + w - 1) / w;
        const uint32_t rounds = (tile + 4 * waves - 1) / (4 * waves);
        const double cost = ((subs * (w - 1) + per_wave) * eval + rounds * solve) / tile;
        if (pick && cost >= best) continue;
        best = cost;
        pick = tile;
        a.sub = (per_wave + subs - 1) / subs;
    }
    if (!pick) return false;
    if (pick > a.n_d) {
        pick = a.n_d;
        a.sub = std::min(a.sub, pick);
    }
    *lds = plan_lds(a, lmax, pick, a.g.rf != nullptr);
    a.n_tiles = (a.n_d + pick - 1) / pick;
    return *lds <= budget;
}

template <typename InT, bool FUSED>
static hipError_t launch_in(const MvArgs& a, size_t lds, hipStream_t stream) {
    const uint32_t round = 8u * kXcdTile;
    const dim3 grid((a.n_rx * a.n_tiles + round - 1) / round * round);
    switch (mv_block_lmax(a.L)) {
        case 16: hipLaunchKernelGGL((mv_block_kernel<InT, 16, FUSED>), grid, dim3(Cfg<16>::kThreads), lds, stream, a); break;
        case 32: hipLaunchKernelGGL((mv_block_kernel<InT, 32, FUSED>), grid, dim3(Cfg<32>::kThreads), lds, stream, a); break;
        default: hipLaunchKernelGGL((mv_block_kernel<InT, 64, FUSED>), grid, dim3(Cfg<64>::kThreads), lds, stream, a); break;
    }
    return hipGetLastError();
}

hipError_t launch_mv_block(const MvArgs& a, int32_t in_dtype, bool fused, size_t lds, hipStream_t stream) {
    if (in_dtype == SUPRA_INT16)
        return fused ? launch_in<int16_t, true>(a, lds, stream) : launch_in<int16_t, false>(a, lds, stream);
    return fused ? launch_in<float, true>(a, lds, stream) : launch_in<float, false>(a, lds, stream);
}

template <typename InT>
static hipError_t launch_batch_in(const MvBatchArgs& b, uint32_t lmax, uint32_t workgroups, size_t lds, hipStream_t stream) {
    const dim3 grid(workgroups);
    if (lmax == 16) hipLaunchKernelGGL((mv_block_batch_kernel<InT, 16>), grid, dim3(Cfg<16>::kThreads), lds, stream, b);
    else if (lmax == 32) hipLaunchKernelGGL((mv_block_batch_kernel<InT, 32>), grid, dim3(Cfg<32>::kThreads), lds, stream, b);
    else hipLaunchKernelGGL((mv_block_batch_kernel<InT, 64>), grid, dim3(Cfg<64>::kThreads), lds, stream, b);
    return hipGetLastError();
}

hipError_t launch_mv_block_batch(const MvBatchArgs& b, uint32_t lmax, int32_t rf_dtype, uint32_t workgroups, size_t lds,
                                 hipStream_t stream) {
    return rf_dtype == SUPRA_INT16 ? launch_batch_in<int16_t>(b, lmax, workgroups, lds, stream)
                                   : launch_batch_in<float>(b, lmax, workgroups, lds, stream);
}

}  // namespace supra_amd
