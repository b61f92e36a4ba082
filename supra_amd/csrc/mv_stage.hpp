// Staging shared by the minimum-variance kernels: the pre-delayed samples of
// a depth tile and its temporal halo in LDS, and each sample's aperture.
#pragma once

#include <hip/hip_runtime.h>

#include <cfloat>
#include <cmath>
#include <cstdint>

#include "bf_internal.hpp"
#include "das_device.hpp"
#include "mv_launch.hpp"

namespace supra_amd {
namespace {

template <typename T> __device__ inline float in_f(T v) { return static_cast<float>(v); }

template <typename T> __device__ inline T clamp_out(float x);
template <> __device__ inline float clamp_out<float>(float x) { return fminf(fmaxf(x, -FLT_MAX), FLT_MAX); }
template <> __device__ inline int16_t clamp_out<int16_t>(float x) {
    return static_cast<int16_t>(fminf(fmaxf(x, -32767.0f), 32767.0f));
}

struct SampleMeta {
    int32_t first, lt, kact;
    int32_t bad;    // a non-finite covariance: every window holding it ends as NaN -> 0
};

// LDS floats set aside for the pre-delay tables of a tile of H staged samples
// (it decides the sizes that fit at all; stage_delayed uses 3 n_ch and 2 H).
__host__ __device__ inline size_t delay_table_floats(size_t n_ch, size_t H) { return kWindowEntries + 4 * n_ch + 6 * H; }

// The thread's index, as a value that the compiler does not know: what is
// derived from it is computed where it is used, not once before the work loop of
// a batch kernel.  Kept over the solve it cost mv_batch_kernel with 64 rows 8
// registers, 258 in all, and with them the second workgroup of a CU (8 frames of
// 140 x 900, 96 channels, L = 40, weakly loaded: 29.9 ms, 20.6 with 248).
__device__ inline int opaque_tid() {
    int t = static_cast<int>(threadIdx.x);
    asm volatile("" : "+v"(t));
    return t;
}

// Fused mode: the pre-delayed samples of scanline s, depths [h_lo, h_lo+H),
// computed from the RF exactly as the pre-delay kernel writes them
// (rawdelay2d_kernel in das_kernels.hip; RawDelay.cu:221-312, 404-468):
// highest-weight transmit, aperture element c = e - first, w * interp * n/W
// through clampCast<float>, 0 for c >= last - first.  Same operations in the
// same order, so the values are bit-identical to the two-kernel path.
//
// Half-waves take one element each, lanes = depths: a lane keeps its depth's
// geometry in registers and no index is divided.  The window weights go to
// xs first and are added up from there, one lane per depth in element order
// (the sum is a serial chain, but of additions only); then the samples take
// their place.  26 depths x 128 elements with 4 waves: 31.7 k cycles with one
// lane per depth for geometry and weights, 15.5 k now (half of it memory latency).
template <typename RFT, int NT>
__device__ inline void stage_delayed(const MvArgs& a, const float* lut, uint32_t s, uint32_t h_lo, int H,
                                     float* xs, unsigned char* lds) {
    const int tid = opaque_tid();
    constexpr int kRows = NT / 32, kBatch = 8;
    const DasArgs& g = a.g;
    const int n_ch = static_cast<int>(a.n_ch), rs = static_cast<int>(a.rs);
    const int hstride = static_cast<int>(a.tile + 2 * a.T);
    float* s_lut = reinterpret_cast<float*>(lds + a.off_fused);
    float* s_xe = s_lut + kWindowEntries;
    float* s_dx = s_xe + n_ch;
    uint32_t* s_off = reinterpret_cast<uint32_t*>(s_dx + n_ch);
    int* s_count = reinterpret_cast<int*>(s_off + n_ch);
    float* s_scale = reinterpret_cast<float*>(s_count + hstride);

    const int hl = tid % 32, cl = tid / 32;
    // the first 32 depths stay in registers over the passes (all of them, mostly)
    const float d_first = g.depths[h_lo + min(hl, H - 1)];
    const auto aperture = [&](float d) { return (((d * g.dt) * g.c) / (2.0f * g.F)) / g.c / g.dt; };
    const float aDT_first = aperture(d_first);
    const ScanView sc = scan_view(g.scans, s);
    const int k = sc.sel();
    TxDT tx{};
    int cnt = 0;
    if (k >= 0) {
        tx = sc.tx(k);
        cnt = tx.last_x > tx.first_x ? static_cast<int>(tx.last_x - tx.first_x) : 0;
    }
    for (int i = tid; i < kWindowEntries; i += NT) s_lut[i] = lut[i];
    for (int i = tid; i < H; i += NT) s_count[i] = 0;
    for (int j = tid; j < cnt; j += NT) {
        const int e = static_cast<int>(tx.first_x) + j;
        const float xe = g.ex[e];
        s_xe[j] = xe;
        s_dx[j] = xe - sc.x();
        s_off[j] = (static_cast<uint32_t>(e) % g.n_ch) * g.n_s;
    }
    __syncthreads();
    for (int h0 = 0; h0 < H; h0 += 32) {
        const int h = h0 + hl;
        const float aDT = h0 == 0 ? aDT_first : aperture(g.depths[h_lo + min(h, H - 1)]);
        const float inv = 1.0f / fminf(aDT, sc.max_ed_x());
        int n = 0;
#pragma unroll 4
        for (int c = cl; c < cnt; c += kRows) {
            const float dx = s_dx[c];
            const float w = s_lut[window_index(dx * inv)];
            const bool in = fabsf(dx) <= aDT;
            if (h < H) xs[h * rs + c] = in ? w : 0.0f;     // (0 leaves a sum of weights as it is)
            n += in ? 1 : 0;
        }
        if (h < H && n != 0) atomicAdd(&s_count[h], n);
    }
    __syncthreads();
    for (int h = tid; h < H; h += NT) {
        const float* w = xs + h * rs;
        const int nadd = s_count[h];
        float wsum = 0.0f;
        int c = 0;
        for (; c + 16 <= cnt; c += 16) {
            float v[16];
#pragma unroll
            for (int u = 0; u < 16; u++) v[u] = w[c + u];
#pragma unroll
            for (int u = 0; u < 16; u++) wsum += v[u];
        }
        for (; c < cnt; c++) wsum += w[c];
        s_scale[h] = nadd > 0 ? 1.0f / wsum * static_cast<float>(nadd) : 1.0f;
    }
    __syncthreads();
    const bool vertical = (sc.dir_x() == 0.0f);
    const RFT* rf_tx = static_cast<const RFT*>(g.rf) + static_cast<uint64_t>(tx.tx_idx) * g.n_ch * g.n_s;
    const __amdgpu_buffer_rsrc_t rsrc = rf_resource(rf_tx, g.n_ch * g.n_s * sizeof(RFT));
    const uint32_t last_bits = last_sample_bits(g.n_s);
    const bool nan = nan_delays<RFT, false>(g.nan_lines, sc, tx.t0, g.n_s);
    for (int h0 = 0; h0 < H; h0 += 32) {
        const int h = h0 + hl;
        if (h >= H) continue;
        const float d = h0 == 0 ? d_first : g.depths[h_lo + h];
        const float aDT = h0 == 0 ? aDT_first : aperture(d);
        const float px = sc.x() + sc.dir_x() * d;
        const float py = sc.dir_y() * d;
        const float py2 = py * py;
        const float scale = s_scale[h];
        float* row = xs + h * rs;
        for (int c0 = cl; c0 < cnt; c0 += kBatch * kRows) {
            float w[kBatch], f[kBatch], v0[kBatch], v1[kBatch];
            bool add[kBatch], edge[kBatch];
#pragma unroll
            for (int u = 0; u < kBatch; u++) {
                const int c = min(c0 + u * kRows, cnt - 1);
                const float dx = s_dx[c];
                const float e = vertical ? dx : s_xe[c] - px;
                const float tau = tx.t0 + (sqrt_rn(e * e + py2) + d);
                const uint32_t ui = static_cast<uint32_t>(tau), off = s_off[c];
                w[u] = row[c];
                f[u] = __builtin_amdgcn_fractf(tau);
                v0[u] = load_rf<RFT>(rsrc, off + ui);
                v1[u] = load_rf<RFT>(rsrc, off + ui + 1u);
                add[u] = (fabsf(dx) <= aDT) & ((__float_as_uint(tau) <= last_bits) | nan);
                edge[u] = !std::is_same_v<RFT, int16_t> && __float_as_uint(tau) == last_bits;
            }
#pragma unroll
            for (int u = 0; u < kBatch; u++) {
                const int c = c0 + u * kRows;
                const float val = edge[u] ? v0[u] : ((1.0f - f[u]) * v0[u] + f[u] * v1[u]);
                const float sample = 0.0f + (add[u] ? w[u] * val : 0.0f);
                if (c < cnt) row[c] = clamp_cast<float>(sample * scale);
            }
        }
        for (int c = cnt + cl; c < rs; c += kRows) row[c] = 0.0f;
    }
    __syncthreads();
}

// Reads the pre-delayed samples of scanline s, depths [h_lo, h_lo + H), into
// xs[h * rs + channel], zero for channels n_ch .. rs-1.  Half-waves take one
// channel each (lanes = depths, no index division); 8 channels per half-wave
// are in flight before the LDS stores (past the last channel it is read again: a
// load under a condition of its own waits for the one before, which cost
// conjugate gradients 14 us of the 320 of a workgroup with 64 rows).
template <typename InT, int NT>
__device__ inline void stage_read(const MvArgs& a, uint32_t s, uint32_t h_lo, int H, float* xs) {
    const InT* xin = static_cast<const InT*>(a.x) + static_cast<uint64_t>(s) * a.n_ch * a.n_d + h_lo;
    constexpr int kBatch = 8, kRows = NT / 32;
    const int rs = static_cast<int>(a.rs), n_ch = static_cast<int>(a.n_ch);
    const int hl = static_cast<int>(threadIdx.x % 32), cl = static_cast<int>(threadIdx.x / 32);
    for (int h0 = 0; h0 < H; h0 += 32) {
        const int h = h0 + hl;
        if (h >= H) continue;
        float* row = xs + h * rs;
        for (int c0 = cl; c0 < n_ch; c0 += kBatch * kRows) {
            float v[kBatch];
#pragma unroll
            for (int u = 0; u < kBatch; u++)
                v[u] = in_f(xin[static_cast<uint64_t>(min(c0 + u * kRows, n_ch - 1)) * a.n_d + h]);
#pragma unroll
            for (int u = 0; u < kBatch; u++)
                if (c0 + u * kRows < n_ch) row[c0 + u * kRows] = v[u];
        }
        for (int c = n_ch + cl; c < rs; c += kRows) row[c] = 0.0f;
    }
    __syncthreads();
}

// First / last channel with a non-zero sample (0 when there is none), the
// sub-array length and the number of active sub-arrays
// (RxBeamformerMV.cu:44-113): one wave per sample, 64 channels per ballot.
// `bad` is set to 0, or to kHuge for a sample with a NaN or a value whose
// square may leave single precision.
constexpr int32_t kHuge = 2;

template <int NT, bool HUGE>
__device__ inline void find_apertures(const MvArgs& a, const float* xs, int H, SampleMeta* meta) {
    const int wv = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / 64)), ln = threadIdx.x % 64;
    const int n_ch = static_cast<int>(a.n_ch), L = static_cast<int>(a.L), rs = static_cast<int>(a.rs);
    constexpr int kSamples = 4, kStep = NT / 64;   // samples of a wave in flight at once
    for (int h0 = wv; h0 < H; h0 += kSamples * kStep) {
        int f[kSamples], l[kSamples];
        bool huge[kSamples];
#pragma unroll
        for (int u = 0; u < kSamples; u++) f[u] = -1, l[u] = 0, huge[u] = false;
        for (int cb = 0; cb < n_ch; cb += 64) {
            const int c = cb + ln;
            float v[kSamples];
#pragma unroll
            for (int u = 0; u < kSamples; u++)
                v[u] = c < n_ch && h0 + u * kStep < H ? xs[(h0 + u * kStep) * rs + c] : 0.0f;
#pragma unroll
            for (int u = 0; u < kSamples; u++) {
                const uint64_t nz = __builtin_amdgcn_ballot_w64(v[u] != 0.0f);
                if (HUGE) huge[u] |= __builtin_amdgcn_ballot_w64(!(fabsf(v[u]) <= 5e17f)) != 0;   // 256 squares of it stay below 1e38
                if (nz != 0) {
                    if (f[u] < 0) f[u] = cb + __builtin_ctzll(nz);
                    l[u] = cb + 63 - __builtin_clzll(nz);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < kSamples; u++) {
            const int h = h0 + u * kStep;
            if (h >= H) break;
            if (f[u] < 0) f[u] = 0;
            if (ln == 0) {
                SampleMeta m;
                m.first = f[u];
                m.lt = min(L, l[u] - f[u] + 1);
                m.kact = min(static_cast<int>(a.K), l[u] - f[u] - m.lt + 2);
                m.bad = huge[u] ? kHuge : 0;
                meta[h] = m;
            }
        }
    }
}

}  // namespace
}  // namespace supra_amd
