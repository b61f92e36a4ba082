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

// Fused mode: the pre-delayed samples of scanline s, depths [h_lo, h_lo+H),
// computed from the RF exactly as the pre-delay kernel writes them
// (rawdelay2d_kernel in das_kernels.hip; RawDelay.cu:221-312, 404-468):
// highest-weight transmit, aperture element c = e - first, w * interp * n/W
// through clampCast<float>, 0 for c >= last - first.  Same operations in the
// same order, so the values are bit-identical to the two-kernel path.
template <typename RFT, int NT>
__device__ inline void stage_delayed(const MvArgs& a, const float* lut, uint32_t s, uint32_t h_lo, int H,
                                     float* xs, unsigned char* lds) {
    const DasArgs& g = a.g;
    const int n_ch = static_cast<int>(a.n_ch);
    const int hstride = static_cast<int>(a.tile + 2 * a.T);
    float* s_lut = reinterpret_cast<float*>(lds + a.off_fused);
    float* s_xe = s_lut + kWindowEntries;
    float* s_dx = s_xe + n_ch;
    float* s_dx2 = s_dx + n_ch;
    uint32_t* s_off = reinterpret_cast<uint32_t*>(s_dx2 + n_ch);
    float* p_d = reinterpret_cast<float*>(s_off + n_ch);
    float* p_adt = p_d + hstride;
    float* p_inv = p_adt + hstride;
    float* p_px = p_inv + hstride;
    float* p_py2 = p_px + hstride;
    float* p_scale = p_py2 + hstride;

    const ScanView sc = scan_view(g.scans, s);
    const int k = sc.sel();
    TxDT tx{};
    int cnt = 0;
    if (k >= 0) {
        tx = sc.tx(k);
        cnt = tx.last_x > tx.first_x ? static_cast<int>(tx.last_x - tx.first_x) : 0;
    }
    for (int i = threadIdx.x; i < kWindowEntries; i += NT) s_lut[i] = lut[i];
    for (int j = threadIdx.x; j < cnt; j += NT) {
        const int e = static_cast<int>(tx.first_x) + j;
        const float xe = g.ex[e];
        const float dx = xe - sc.x();
        s_xe[j] = xe;
        s_dx[j] = dx;
        s_dx2[j] = dx * dx;
        s_off[j] = (static_cast<uint32_t>(e) % g.n_ch) * g.n_s;
    }
    __syncthreads();
    // per-sample geometry and the aperture's weight sum and count
    for (int h = threadIdx.x; h < H; h += NT) {
        const float d = g.depths[h_lo + h];
        const float aDT = (((d * g.dt) * g.c) / (2.0f * g.F)) / g.c / g.dt;
        const float inv = 1.0f / fminf(aDT, sc.max_ed_x());
        const float py = sc.dir_y() * d;
        float wsum = 0.0f;
        int nadd = 0;
        for (int j = 0; j < cnt; j++) {
            const float dx = s_dx[j];
            if (fabsf(dx) <= aDT) {
                wsum += s_lut[window_index(dx * inv)];
                nadd++;
            }
        }
        float scale = 1.0f;
        if (nadd > 0) scale = 1.0f / wsum * static_cast<float>(nadd);
        p_d[h] = d;
        p_adt[h] = aDT;
        p_inv[h] = inv;
        p_px[h] = sc.x() + sc.dir_x() * d;
        p_py2[h] = py * py;
        p_scale[h] = scale;
    }
    __syncthreads();
    const bool vertical = (sc.dir_x() == 0.0f);
    const RFT* rf_tx = static_cast<const RFT*>(g.rf) + static_cast<uint64_t>(tx.tx_idx) * g.n_ch * g.n_s;
    const __amdgpu_buffer_rsrc_t rsrc = rf_resource(rf_tx, g.n_ch * g.n_s * sizeof(RFT));
    const int rs = static_cast<int>(a.rs);
#pragma unroll 4
    for (int idx = threadIdx.x; idx < H * rs; idx += NT) {
        const int c = idx / H, h = idx % H;
        float v = 0.0f;
        if (c < cnt) {
            float sample = 0.0f;
            const float dx = s_dx[c];
            if (fabsf(dx) <= p_adt[h]) {
                const float w = s_lut[window_index(dx * p_inv[h])];
                float q;
                if (vertical) {
                    q = s_dx2[c] + p_py2[h];
                } else {
                    const float e = s_xe[c] - p_px[h];
                    q = e * e + p_py2[h];
                }
                const float tau = tx.t0 + (sqrt_rn(q) + p_d[h]);
                gather<RFT, false>(rsrc, s_off[c], g.n_s, tau, w, sample);
            }
            v = clamp_cast<float>(sample * p_scale[h]);
        }
        xs[h * rs + c] = v;
    }
    __syncthreads();
}

// Reads the pre-delayed samples of scanline s, depths [h_lo, h_lo + H), into
// xs[h * rs + channel], zero for channels n_ch .. rs-1.  Half-waves take one
// channel each (lanes = depths, no index division); 8 channels per half-wave
// are in flight before the LDS stores.
template <typename InT, int NT>
__device__ inline void stage_read(const MvArgs& a, uint32_t s, uint32_t h_lo, int H, float* xs) {
    const InT* xin = static_cast<const InT*>(a.x) + static_cast<uint64_t>(s) * a.n_ch * a.n_d + h_lo;
    constexpr int kBatch = 8, kRows = NT / 32;
    const int rs = static_cast<int>(a.rs), n_ch = static_cast<int>(a.n_ch);
    const int hl = static_cast<int>(threadIdx.x % 32), cl = static_cast<int>(threadIdx.x / 32);
    for (int h0 = 0; h0 < H; h0 += 32) {
        const int h = h0 + hl;
        if (h >= H) continue;
        for (int c0 = cl; c0 < rs; c0 += kBatch * kRows) {
            float v[kBatch];
#pragma unroll
            for (int u = 0; u < kBatch; u++) {
                const int c = c0 + u * kRows;
                v[u] = c < n_ch ? in_f(xin[static_cast<uint64_t>(c) * a.n_d + h]) : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < kBatch; u++) {
                const int c = c0 + u * kRows;
                if (c < rs) xs[h * rs + c] = v[u];
            }
        }
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
