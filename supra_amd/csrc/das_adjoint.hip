// Differentiable 2D delay-and-sum: per-frame dt-space tables built on the GPU
// for a device array of speeds of sound, and the adjoint of the beamformer
// with respect to the RF and to the speed of sound.
//
// No reference counterpart: SUPRA beamforms with one speed of sound per call
// and never differentiates (RxBeamformerCuda.cu:539-663).  The forward is the
// 2D kernel of das_kernels.hip (RxBeamformerCuda.cu:230-323 with
// RxSampleBeamformerDelayAndSum.h:122-208); for a fixed speed of sound its
// output is linear in the RF,
//     y(s,r) = sum_k a_k (n_k / W_k) sum_e w_e [(1-f) rf_k,ch(e)[i] + f rf_k,ch(e)[i+1]],
// with i = floor(tau), f = tau - i, a_k = txWeight_k (transmit interpolation)
// or 1 (the selected transmit).  The forward optionally writes
// norm = a_k n_k / W_k per pixel and slot; the adjoint scatters
// beta = dL/dy * norm times w_e (1-f) and w_e f back into the two samples.
//
// Speed of sound: every dt-space length is millimetres / (c dt), while the
// transmit delay t0 (seconds / dt) and the additional offset are fixed, so
// tau = t0 + G / c + offset and dtau/dc = -geo / c with geo = sqrt(q) + d,
// the geometric part the kernel evaluates anyway.  Aperture membership, the
// window argument and n/W are ratios of dt-space lengths: independent of c up
// to rounding, piecewise constant, derivative 0.  Hence
//     dL/dc = -(1/c) sum beta w_e (rf[i+1] - rf[i]) geo        (interpolated samples)
// and the delay tables are recomputed here, never stored by the forward.
//
// Launch layout (MI355X): one wave64 per (frame, scanline, slot, pair of
// aperture elements), 4 waves per workgroup.  A wave walks the depths of its
// elements, lanes = 64 consecutive depths, and accumulates each element's RF
// line in a ring of 256 samples in LDS: the delays grow with depth, so the
// lanes of one instruction touch ~64 neighbouring samples, and samples more
// than a guard below the delay of the chunk's first depth are final.  Those
// leave the ring in order, 64 at a time, as coalesced stores when no other
// wave writes that (transmit, channel) line (each focused transmit feeds one
// scanline), else as global float atomics; a target outside the ring's window
// (delays not sorted, or a chunk wider than the ring) is handled exactly by
// moving the ring or adding to the flushed output.  A sample's slot keeps the
// lower shares of that sample and the upper shares of the one before, so the
// lanes' delays meet only where two share a sample; the upper lane adds for
// both, and one LDS read-add-write per lane does.  d/dc partial sums go to a
// per-wave slot and are reduced per frame in a fixed order, so the result does
// not depend on scheduling.  The depth-only quantities (the F-number aperture
// aDT and 1/aDT, four IEEE divisions per depth) come from per-frame planes
// built once.
//
// What bounds it: 16 frames of 128 lines x 2080 depths x 64 elements take
// 0.56 ms (0.75 ms with one element per wave, a share handed from lane to
// lane and an 8 + 4 byte depth entry): the address unit is busy 90 % and the
// VALU 85 % of that time, HBM (0.86 GB read, 1.07 GB written) 43 %.  Two
// elements per wave share a depth's position, aperture and beta; 3 and 4 cost
// waves (their rings) and time the same and 7 % more.  Loads and stores
// complete in one order, so the depth loop keeps a fixed number of stores per
// chunk and uses its d/dc loads after them: a wait for loads then never
// includes the chunk's own stores.  A window of the RF in LDS for d/dc waited
// for its own loads in the loop and took 1.05 ms.
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cmath>
#include <cstddef>
#include <cstdint>

#include "bf_internal.hpp"
#include "das_device.hpp"
#include "das_launch.hpp"

namespace supra_amd {

namespace {

constexpr int kTableThreads = 256;
constexpr uint32_t kThrParts = 4;                // element strides per transmit slot
constexpr uint32_t kScanLanes = 4 * kThrParts;   // lanes per scanline in frame_tables_kernel

__host__ __device__ inline uint32_t scan_items_start(uint32_t n_d, uint32_t n_el) {
    return (n_d + n_el + 63u) / 64u * 64u;
}
constexpr int kBetaTile = 32;
constexpr int kWave = 64;
// Elements of one adjoint wave, waves per workgroup.
constexpr uint32_t kAdjointElements = 2;
constexpr uint32_t kAdjointWaves = 4;
// Each adjoint wave accumulates its RF lines in rings of kRing samples of LDS;
// samples more than kRingGuard below the delay of the chunk's first depth are
// final and leave the ring.
constexpr uint32_t kRing = 256;
// Planes of the per-frame depth table.
constexpr uint32_t kDepthPlanes = 3;
constexpr uint32_t kRingWords = 2 * kRing + 2;
constexpr int32_t kRingGuard = 32;

// ---- per-frame tables --------------------------------------------------------

// The same double-precision expressions and float casts as build_dt_tables
// (bf_context.hip), which restates RxBeamformerCuda::convertToDtSpace
// (RxBeamformerCuda.cu:58-107) with the first-call factors.
__global__ __launch_bounds__(kTableThreads) void frame_tables_kernel(const FrameTablesArgs a) {
    const uint32_t f = blockIdx.y;
    const uint32_t i = blockIdx.x * kTableThreads + threadIdx.x;
    const double c = a.c[f];
    const double factor = 1 / 1.0 / (c * a.dt);
    const double factor_time = 1 / 1.0 / a.dt;
    if (i == 0) a.frame_c[f] = static_cast<float>(c);
    if (i < a.n_d) {
        a.depths[static_cast<size_t>(f) * a.n_d + i] = static_cast<float>(a.depths_mm[i] * factor);
        return;
    }
    uint32_t j = i - a.n_d;
    if (j < a.n_el) {
        a.ex[static_cast<size_t>(f) * a.n_el + j] = static_cast<float>(a.ex_mm[j] * factor);
        return;
    }
    // Scanlines: kScanLanes consecutive lanes per scanline (4 transmit slots x
    // kThrParts element strides), from the first item at a multiple of the
    // wave size, so that each group is one aligned shuffle segment; the
    // far-field threshold of a slot is the largest |ex - x| over its
    // connected elements, a max, so the parts reduce in any order.
    const uint32_t s0 = scan_items_start(a.n_d, a.n_el);
    if (i < s0) return;
    j = i - s0;
    const uint32_t sub = j % kScanLanes;
    j /= kScanLanes;
    if (j >= a.n_rx) return;   // whole groups of kScanLanes lanes
    const supra_scanline_rx& s = a.scan_mm[j];
    ScanlineDT o = a.scan_fixed[j];
    o.x = static_cast<float>(s.position[0] * factor);
    o.z = static_cast<float>(s.position[2] * factor);
    o.max_ed_x = static_cast<float>(s.max_element_distance[0] * factor);
    o.max_ed_y = static_cast<float>(s.max_element_distance[1] * factor);
    const uint32_t kk = sub / kThrParts, part = sub % kThrParts;
    float thr = 0.0f;
    {
        const TxDT& t = o.tx[kk];
        for (uint32_t e = t.first_x + part; e < t.last_x; e += kThrParts) {
            if (a.e2c && a.e2c[e] < 0) continue;
            const float v = fabsf(static_cast<float>(a.ex_mm[e] * factor) - o.x);
            // (a NaN position: no depth is far)
            thr = (thr < v) ? v : (v != v ? INFINITY : thr);
        }
    }
    for (uint32_t m = 1; m < kThrParts; m <<= 1) {
        const float v = __shfl_xor(thr, static_cast<int>(m), kScanLanes);
        thr = (thr < v) ? v : thr;
    }
    float thr_k[4];
    for (int k = 0; k < 4; k++) thr_k[k] = __shfl(thr, k * static_cast<int>(kThrParts), kScanLanes);
    if (sub != 0) return;
    for (int k = 0; k < 4; k++) {
        TxDT& t = o.tx[k];
        t.t0 = static_cast<float>(s.tx[k].initial_delay * factor_time);
        t.far_thr = (thr_k[k] < o.max_ed_x) ? o.max_ed_x : thr_k[k];
    }
    a.scans[static_cast<size_t>(f) * a.n_rx + j] = o;
}

// ---- per-frame depth table ----------------------------------------------------

// Planes of depth, aDT and 1/aDT per (frame, depth), aDT with the same single-precision
// operations as the forward kernel (das_kernels.hip, after
// RxSampleBeamformerDelayAndSum.h:167 and RxBeamformerCommon.h:27-33).
__global__ __launch_bounds__(256) void depth_table_kernel(const float* depths, const float* frame_c, float dt,
                                                          float f_number, uint32_t n_d, float* dtab) {
    const uint32_t f = blockIdx.y;
    const uint32_t r = blockIdx.x * 256 + threadIdx.x;
    if (r >= n_d) return;
    const size_t i = static_cast<size_t>(f) * n_d + r;
    const float d = depths[i];
    const float c = frame_c[f];
    const float aDT = (((d * dt) * c) / (2.0f * f_number)) / c / dt;
    float* const o = dtab + static_cast<size_t>(f) * kDepthPlanes * n_d + r;
    o[0] = d;
    o[n_d] = aDT;
    o[2 * static_cast<size_t>(n_d)] = 1.0f / aDT;
}

// ---- beta = dL/dy * norm, transposed to [frame][slot][scanline][depth] -------

__global__ __launch_bounds__(256) void beta_kernel(const float* grad_image, const float* norm, float* beta,
                                                   uint32_t n_rx, uint32_t n_d, uint32_t slots) {
    __shared__ float tile[kBetaTile][kBetaTile + 1];
    const uint32_t s0 = blockIdx.x * kBetaTile, r0 = blockIdx.y * kBetaTile, f = blockIdx.z;
    const uint32_t tx = threadIdx.x % kBetaTile, ty = threadIdx.x / kBetaTile;
    const float* g = grad_image + static_cast<size_t>(f) * n_d * n_rx;
    for (uint32_t rr = ty; rr < kBetaTile; rr += 256 / kBetaTile) {
        const uint32_t r = r0 + rr, s = s0 + tx;
        tile[rr][tx] = (r < n_d && s < n_rx) ? g[static_cast<size_t>(r) * n_rx + s] : 0.0f;
    }
    __syncthreads();
    for (uint32_t q = 0; q < slots; q++) {
        const size_t base = (static_cast<size_t>(f) * slots + q) * n_rx;
        for (uint32_t ss = ty; ss < kBetaTile; ss += 256 / kBetaTile) {
            const uint32_t s = s0 + ss, r = r0 + tx;
            if (s < n_rx && r < n_d) {
                const size_t idx = (base + s) * n_d + r;
                const float nv = norm[idx];
                // Saturated pixels (norm 0) pass no gradient, whatever dL/dy is.
                beta[idx] = (nv == 0.0f) ? 0.0f : tile[tx][ss] * nv;
            }
        }
    }
}

// ---- the adjoint ---------------------------------------------------------------

__device__ inline double wave_sum(double v) {
    for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
    return v;
}

// Whole-wave DPP shift by one lane (wave_shr:1): lane i reads lane i - 1,
// lane 0 reads 0.  Called with every lane of the wave active.
__device__ inline int32_t from_prev(int32_t v) { return __builtin_amdgcn_update_dpp(0, v, 0x138, 0xf, 0xf, true); }
__device__ inline float from_prev(float v) {
    return __uint_as_float(static_cast<uint32_t>(from_prev(static_cast<int32_t>(__float_as_uint(v)))));
}

__device__ inline uint64_t ballot(bool v) { return __builtin_amdgcn_ballot_w64(v); }

// Largest v of the wave (rare paths only).
__device__ inline uint32_t wave_max(uint32_t v, uint32_t lane) {
    for (uint32_t o = kWave / 2; o > 0; o >>= 1)
        v = max(v, static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(static_cast<int>((lane ^ o) * 4u), static_cast<int>(v))));
    return v;
}

// Takes the kWave samples from base on (a multiple of kWave) out of a ring and
// clears them.  Sample u's slot holds the upper shares of u - 1 and the lower
// shares of u; the upper shares of the last slot's sample are behind it, and
// belong to the first slot's sample.  Samples at or beyond base + kRing - 1
// were never added to, and the slots read for them hold 0 by then.
__device__ inline float ring_take(float* ring, uint32_t lane, int32_t base) {
    const uint32_t first = static_cast<uint32_t>(base) & (kRing - 1u);   // (uniform)
    float2& at = reinterpret_cast<float2*>(ring)[first + lane];
    float v = at.x + at.y;
    at = make_float2(0.0f, 0.0f);
    if (first == 0 && lane == 0) {
        v += ring[2 * kRing];
        ring[2 * kRing] = 0.0f;
    }
    return v;
}

// The line's sample u: a store where the wave is its only writer (past the
// line's end the buffer drops it), else a global atomic.
template <bool EXCLUSIVE>
__device__ inline void put_sample(__amdgpu_buffer_rsrc_t line, float* out, int32_t u, int32_t n_s, float v) {
    if (EXCLUSIVE) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), line, u * 4, 0, 0);
    else if (v != 0.0f && u < n_s) atomicAdd(&out[u], v);
}

// NANS: the geometry has scanlines whose delays are NaN (nan_lines).
template <bool GRAD, bool DC, bool EXCLUSIVE, bool NANS>
__global__ __launch_bounds__(kAdjointWaves * kWave) void das2d_adjoint_kernel(const AdjointArgs a) {
    __shared__ float s_lut[kWindowEntries];
    __shared__ __align__(8) float s_rings[GRAD ? kAdjointWaves * kAdjointElements * kRingWords : 1];
    const uint32_t wave = uniform_u32(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    float* const s_ring = s_rings + (GRAD ? wave * kAdjointElements * kRingWords : 0);
    for (uint32_t i = threadIdx.x; i < kWindowEntries; i += blockDim.x) s_lut[i] = a.lut[i];
    if (GRAD)
        for (uint32_t i = lane; i < kAdjointElements * kRingWords; i += kWave) s_ring[i] = 0.0f;
    __syncthreads();

    uint32_t b = blockIdx.x;
    const uint32_t eg = b % a.egroups;
    b /= a.egroups;
    const uint32_t q = b % a.n_slots;
    b /= a.n_slots;
    const uint32_t s = b % a.n_rx;
    const uint32_t f = b / a.n_rx;

    const ScanView sc = scan_view(a.scans + static_cast<size_t>(f) * a.scan_frame_stride, s);
    int k;
    bool active;
    if (a.interp_tx) {
        k = static_cast<int>(q);
        active = ((sc.active_mask() >> k) & 1) != 0;
    } else {
        k = sc.sel();
        active = k >= 0;
    }
    TxDT tx{};
    if (active) tx = sc.tx(k);
    const uint32_t first = tx.first_x + (eg * kAdjointWaves + wave) * kAdjointElements;

    // The wave's elements.  One that is past the aperture or not connected has
    // a NaN distance, so that no lane takes it (an F-number so small that the
    // aperture is infinite would take an infinite one), and no lines.
    float xe[kAdjointElements], dx[kAdjointElements], dc[kAdjointElements];
    int32_t base[kAdjointElements];   // samples below it are final and in out[]; the ring holds the next kRing - 1
    size_t line[kAdjointElements];
    bool on[kAdjointElements];
    __amdgpu_buffer_rsrc_t rf[kAdjointElements], grad[kAdjointElements];
    float near = INFINITY;
    bool any = false;
    const float x = sc.x();
#pragma unroll
    for (uint32_t n = 0; n < kAdjointElements; n++) {
        const uint32_t e = first + n;
        on[n] = active && e < tx.last_x;
        uint32_t ch = 0;
        if (on[n]) {
            const int32_t m = a.e2c ? a.e2c[e] : static_cast<int32_t>(e % a.n_ch);
            on[n] = m >= 0;
            ch = on[n] ? static_cast<uint32_t>(m) : 0u;
        }
        xe[n] = on[n] ? a.ex[static_cast<size_t>(f) * a.el_frame_stride + e] : 0.0f;
        dx[n] = on[n] ? xe[n] - x : NAN;
        near = fminf(near, fabsf(dx[n]));
        any = any || on[n];
        line[n] = a.rf_frame_stride * f + (static_cast<size_t>(tx.tx_idx) * a.n_ch + ch) * a.n_s;
        if (GRAD) grad[n] = rf_resource(a.grad_rf + line[n], on[n] ? a.n_s * 4u : 0u);
        if (DC) rf[n] = rf_resource(a.rf + line[n], on[n] ? a.n_s * 4u : 0u);
        base[n] = 0;
        dc[n] = 0.0f;
    }
    if (any && a.n_depths > 0u) {
        // (reads past the last depth give 0: no aperture, no beta)
        const float* const planes = a.dtab + static_cast<size_t>(f) * kDepthPlanes * a.n_depths;
        const __amdgpu_buffer_rsrc_t depth = rf_resource(planes, a.n_depths * 4u);
        const __amdgpu_buffer_rsrc_t aperture = rf_resource(planes + a.n_depths, a.n_depths * 4u);
        const __amdgpu_buffer_rsrc_t inverse =
            rf_resource(planes + 2 * static_cast<size_t>(a.n_depths), a.n_depths * 4u);
        const __amdgpu_buffer_rsrc_t beta = rf_resource(
            a.beta + ((static_cast<size_t>(f) * a.n_slots + q) * a.n_rx + s) * a.n_depths, a.n_depths * 4u);
        const float dir_x = sc.dir_x(), dir_y = sc.dir_y(), med = sc.max_ed_x();
        // 1 / fminf(aDT, med) is 1/aDT below med and 1/med from there on.
        const float inv_med = 1.0f / med;
        const int32_t n_s = static_cast<int32_t>(a.n_s);
        const uint32_t last_bits = last_sample_bits(a.n_s);
        const uint64_t nan = NANS && nan_delays<float, false>(1, sc, tx.t0, a.n_s) ? ~0ull : 0ull;   // (uniform)
        float w_far[kAdjointElements];
        bool empty[kAdjointElements];   // nothing was added to the ring yet
#pragma unroll
        for (uint32_t n = 0; n < kAdjointElements; n++) {
            w_far[n] = s_lut[window_index(dx[n] * inv_med)];
            empty[n] = true;
        }
        // The first chunk with a depth whose aperture reaches the wave's nearest
        // element, where the depths do not decrease: the chunks above add
        // nothing.  (Not a test in the loop: a chunk that is passed over there
        // would leave the loop without its stores, and with their number open
        // every wait for a load would be a wait for the stores as well.)
        uint32_t chunk = 0;
        if (a.depths_sorted) {
            const uint32_t chunks = (a.n_depths + kWave - 1u) / kWave;
            for (; chunk < chunks; chunk += kWave) {
                const uint32_t r = min((chunk + lane) * kWave + kWave, a.n_depths) - 1u;
                const uint64_t reached = ballot(near <= load_rf<float>(aperture, r));
                if (reached != 0) {
                    chunk += static_cast<uint32_t>(__builtin_ctzll(reached));
                    break;
                }
            }
        }
        // This iteration's depth entry and beta; the next iteration's are
        // loaded at the top of each iteration.
        using Quad = uint32_t __attribute__((ext_vector_type(4)));
        uint32_t r0 = chunk * kWave;
        float next_d = load_rf<float>(depth, r0 + lane), next_aDT = load_rf<float>(aperture, r0 + lane);
        float next_inv = load_rf<float>(inverse, r0 + lane), next_beta = load_rf<float>(beta, r0 + lane);
        // (waited for here: inside the loop they are older than the d/dc loads
        // and need no wait of their own, which would reach the stores)
        asm volatile("" ::"v"(next_d), "v"(next_aDT), "v"(next_inv), "v"(next_beta));
        for (; r0 < a.n_depths; r0 += kWave) {
            float d = next_d;
            const float aDT = next_aDT, inv_aDT = next_inv, bt = next_beta;
            const uint32_t rn = r0 + kWave + lane;
            next_d = load_rf<float>(depth, rn);
            next_aDT = load_rf<float>(aperture, rn);
            next_inv = load_rf<float>(inverse, rn);
            next_beta = load_rf<float>(beta, rn);
            const uint64_t has_beta = ballot(bt != 0.0f);
            if (r0 + kWave > a.n_depths) {   // (uniform)
                // lanes past the last depth go on in steps of two samples, so
                // that their samples stay sorted and apart; they add nothing
                const uint32_t last = a.n_depths - 1u - r0;
                const float d_last = __uint_as_float(
                    static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(__float_as_uint(d)), last)));
                if (lane > last) d = d_last + 2.0f * static_cast<float>(lane - last);
            }
            // (uniform) every lane's aperture is at its largest: one weight per element
            const bool far = ballot(aDT < med) == 0;
            const float inv = aDT < med ? inv_aDT : inv_med;
            // Same single-precision operations as the forward kernel.
            const float px = x + dir_x * d;
            const float py = dir_y * d;
            const float py2 = py * py;
            float bw[kAdjointElements], fr[kAdjointElements], geo[kAdjointElements];
            float g0[kAdjointElements], g1[kAdjointElements];
            int32_t idx[kAdjointElements];
            uint64_t act[kAdjointElements];   // lanes that have the element in their aperture and their delay in the RF
            int32_t i_first[kAdjointElements], i_last[kAdjointElements];
            uint64_t same_prev[kAdjointElements];
            bool sorted[kAdjointElements];
#pragma unroll
            for (uint32_t n = 0; n < kAdjointElements; n++) {
                const float w = far ? w_far[n] : s_lut[window_index(dx[n] * inv)];
                const float ee = xe[n] - px;
                geo[n] = sqrt_rn(ee * ee + py2) + d;
                float tau = tx.t0 + geo[n];
                tau = tau + a.offset;
                act[n] = has_beta & ballot(fabsf(dx[n]) <= aDT) & (ballot(__float_as_uint(tau) <= last_bits) | nan);
                const int32_t i = static_cast<int32_t>(tau);   // (a delay in the RF is not negative: its floor)
                idx[n] = i;
                fr[n] = __builtin_amdgcn_fractf(tau);
                bw[n] = bt * w;
                const int32_t prev = from_prev(i);
                same_prev[n] = ballot(i == prev) & ~1ull;
                sorted[n] = (ballot(i < prev) & ~1ull) == 0;
                i_first[n] = __builtin_amdgcn_readfirstlane(i);
                i_last[n] = __builtin_amdgcn_readlane(i, kWave - 1);
                if (DC) {
                    g0[n] = load_rf<float>(rf[n], static_cast<uint32_t>(i));
                    g1[n] = load_rf<float>(rf[n], static_cast<uint32_t>(i) + 1u);
                }
            }
#pragma unroll
            for (uint32_t n = 0; GRAD && n < kAdjointElements; n++) {
                float* const ring = s_ring + n * kRingWords;
                float* const out = a.grad_rf + line[n];
                const int32_t i = idx[n];
                const float lo = bw[n] * (1.0f - fr[n]), hi = bw[n] * fr[n];
                // Samples more than a guard below lane 0's (this chunk's
                // smallest delay) are final: flush them, kWave at a time, one
                // store in every chunk (outside the line where there is
                // nothing to flush).
                const int32_t final_to = min(max(i_first[n], 0), n_s) - kRingGuard;
                if (EXCLUSIVE && empty[n]) {   // (uniform) the samples above the aperture's first: 0
                    for (; base[n] + 5 * kWave <= final_to; base[n] += 4 * kWave)
                        __builtin_amdgcn_raw_buffer_store_b128(
                            Quad{0, 0, 0, 0}, grad[n],
                            static_cast<int>((static_cast<uint32_t>(base[n]) + 4u * lane) * 4u), 0, 0);
                    empty[n] = false;
                }
                for (; base[n] + 2 * kWave <= final_to; base[n] += kWave)
                    put_sample<EXCLUSIVE>(grad[n], out, base[n] + static_cast<int32_t>(lane), n_s,
                                          ring_take(ring, lane, base[n]));
                float v = 0.0f;
                int32_t u = n_s;
                if (base[n] + kWave <= final_to) {
                    v = ring_take(ring, lane, base[n]);
                    u = base[n] + static_cast<int32_t>(lane);
                    base[n] += kWave;
                }
                put_sample<EXCLUSIVE>(grad[n], out, u, n_s, v);
                // Delays do not decrease with depth, so the lanes' samples are
                // sorted and, where a depth step is at least half a sample, no
                // three lanes share one: of two lanes with one sample the
                // upper one adds for both, and one plain LDS read-add-write
                // per lane holds the sums.
                const uint64_t pair = same_prev[n] & act[n] & (act[n] << 1);   // takes the lane below's share
                const float lo_pair = lo + from_prev(lo), hi_pair = hi + from_prev(hi);
                const bool in_ring = sorted[n] && i_first[n] >= base[n] && i_last[n] - base[n] <= static_cast<int32_t>(kRing) - 2;
                if (in_ring && (same_prev[n] & (same_prev[n] >> 1)) == 0) {
                    if (__builtin_amdgcn_inverse_ballot_w64(act[n] & ~(pair >> 1))) {
                        float* const at = ring + 2u * (static_cast<uint32_t>(i) & (kRing - 1u));
                        const bool both = __builtin_amdgcn_inverse_ballot_w64(pair);
                        const float lo_sum = at[1], hi_sum = at[2];
                        at[1] = lo_sum + (both ? lo_pair : lo);
                        at[2] = hi_sum + (both ? hi_pair : hi);
                    }
                } else {
                    // Any other chunk: the ring moves up to the largest target
                    // (wide apertures per chunk only), a target that is then
                    // below it is added to the flushed output, and the rest
                    // goes to the ring with LDS atomics.
                    const bool add = __builtin_amdgcn_inverse_ballot_w64(act[n]);
                    const int32_t top = static_cast<int32_t>(
                        uniform_u32(wave_max(add ? static_cast<uint32_t>(i) : 0u, lane)));
                    for (; top - base[n] > static_cast<int32_t>(kRing) - 2; base[n] += kWave)
                        put_sample<EXCLUSIVE>(grad[n], out, base[n] + static_cast<int32_t>(lane), n_s,
                                              ring_take(ring, lane, base[n]));
                    if (ballot(add && i < base[n]) != 0) {
                        __threadfence();
                        if (add && i < base[n]) atomicAdd(&out[i], lo);
                        if (add && i + 1 < min(base[n], n_s)) atomicAdd(&out[i + 1], hi);
                    }
                    if (add) {
                        float* const at = ring + 2u * (static_cast<uint32_t>(i) & (kRing - 1u));
                        if (i >= base[n]) atomicAdd(&at[1], lo);
                        if (i + 1 >= base[n]) atomicAdd(&at[2], hi);
                    }
                }
            }
#pragma unroll
            for (uint32_t n = 0; DC && n < kAdjointElements; n++) {
                // (the last sample, with zero fraction, has no slope)
                const float slope = (bw[n] * (g1[n] - g0[n])) * geo[n];
                dc[n] += __builtin_amdgcn_inverse_ballot_w64(act[n] & ballot(idx[n] < n_s - 1)) ? slope : 0.0f;
            }
        }
#pragma unroll
        for (uint32_t n = 0; GRAD && n < kAdjointElements; n++)
            for (; on[n] && base[n] < n_s; base[n] += kWave)
                put_sample<EXCLUSIVE>(grad[n], a.grad_rf + line[n], base[n] + static_cast<int32_t>(lane), n_s,
                                      ring_take(s_ring + n * kRingWords, lane, base[n]));
    }
    if (DC) {
        double v = 0.0;
#pragma unroll
        for (uint32_t n = 0; n < kAdjointElements; n++) v += static_cast<double>(dc[n]);
        v = wave_sum(v);
        if (lane == 0) a.dc_part[static_cast<size_t>(blockIdx.x) * kAdjointWaves + wave] = v;
    }
}

// dL/dc per frame: fixed-order sum of the waves' partial sums, times -1/c.
constexpr uint32_t kReduceThreads = 1024;

__global__ __launch_bounds__(kReduceThreads) void dc_reduce_kernel(const double* part, uint32_t per_frame,
                                                                   const double* c, double* grad_c) {
    __shared__ double red[kReduceThreads];
    const uint32_t f = blockIdx.x;
    double acc = 0.0;
    for (uint32_t i = threadIdx.x; i < per_frame; i += kReduceThreads)
        acc += part[static_cast<size_t>(f) * per_frame + i];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (uint32_t w = kReduceThreads / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) grad_c[f] = -red[0] / c[f];
}

// Zero the listed (transmit, channel) lines of every frame (lines no wave writes).
__global__ __launch_bounds__(256) void zero_lines_kernel(float* grad_rf, const uint32_t* lines, uint32_t n_s,
                                                         uint64_t frame_stride) {
    float* p = grad_rf + frame_stride * blockIdx.y + static_cast<size_t>(lines[blockIdx.x]) * n_s;
    for (uint32_t i = threadIdx.x; i < n_s; i += 256) p[i] = 0.0f;
}

__global__ __launch_bounds__(256) void fill_zero_kernel(float* p, uint64_t n) {
    for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x; i < n;
         i += static_cast<uint64_t>(gridDim.x) * 256)
        p[i] = 0.0f;
}

}  // namespace

hipError_t launch_frame_tables(const FrameTablesArgs& a, hipStream_t stream) {
    const uint32_t items = scan_items_start(a.n_d, a.n_el) + a.n_rx * kScanLanes;
    dim3 grid((items + kTableThreads - 1) / kTableThreads, a.n_frames), block(kTableThreads);
    hipLaunchKernelGGL(frame_tables_kernel, grid, block, 0, stream, a);
    return hipGetLastError();
}

hipError_t launch_depth_table(const float* depths, const float* frame_c, float dt, float f_number, uint32_t n_d,
                              uint32_t frames, float* dtab, hipStream_t stream) {
    dim3 grid((n_d + 255) / 256, frames), block(256);
    hipLaunchKernelGGL(depth_table_kernel, grid, block, 0, stream, depths, frame_c, dt, f_number, n_d, dtab);
    return hipGetLastError();
}

hipError_t launch_beta(const float* grad_image, const float* norm, float* beta, uint32_t n_rx, uint32_t n_d,
                       uint32_t slots, uint32_t frames, hipStream_t stream) {
    dim3 grid((n_rx + kBetaTile - 1) / kBetaTile, (n_d + kBetaTile - 1) / kBetaTile, frames), block(256);
    hipLaunchKernelGGL(beta_kernel, grid, block, 0, stream, grad_image, norm, beta, n_rx, n_d, slots);
    return hipGetLastError();
}

uint32_t das_adjoint_groups(uint32_t aperture) {
    constexpr uint32_t per_group = kAdjointElements * kAdjointWaves;
    return aperture == 0 ? 1u : (aperture + per_group - 1u) / per_group;
}
uint32_t das_adjoint_waves() { return kAdjointWaves; }

template <bool NANS>
static auto adjoint_kernel(const AdjointArgs& a) {
    if (!a.grad_rf) return das2d_adjoint_kernel<false, true, true, NANS>;
    if (a.dc_part) return a.exclusive ? das2d_adjoint_kernel<true, true, true, NANS> : das2d_adjoint_kernel<true, true, false, NANS>;
    return a.exclusive ? das2d_adjoint_kernel<true, false, true, NANS> : das2d_adjoint_kernel<true, false, false, NANS>;
}

hipError_t launch_das_adjoint(const AdjointArgs& a, uint32_t frames, hipStream_t stream) {
    const uint64_t blocks = static_cast<uint64_t>(frames) * a.n_rx * a.n_slots * a.egroups;
    dim3 grid(static_cast<uint32_t>(blocks)), block(kAdjointWaves * kWave);
    if (!a.grad_rf && !a.dc_part) return hipSuccess;
    const auto kernel = a.nan_lines ? adjoint_kernel<true>(a) : adjoint_kernel<false>(a);
    hipLaunchKernelGGL(kernel, grid, block, 0, stream, a);
    return hipGetLastError();
}

hipError_t launch_dc_reduce(const double* part, uint32_t per_frame, const double* c, double* grad_c, uint32_t frames,
                            hipStream_t stream) {
    hipLaunchKernelGGL(dc_reduce_kernel, dim3(frames), dim3(kReduceThreads), 0, stream, part, per_frame, c, grad_c);
    return hipGetLastError();
}

hipError_t launch_zero_lines(float* grad_rf, const uint32_t* lines, uint32_t n_lines, uint32_t n_s,
                             uint64_t frame_stride, uint32_t frames, hipStream_t stream) {
    if (n_lines == 0) return hipSuccess;
    hipLaunchKernelGGL(zero_lines_kernel, dim3(n_lines, frames), dim3(256), 0, stream, grad_rf, lines, n_s,
                       frame_stride);
    return hipGetLastError();
}

hipError_t launch_fill_zero(float* p, uint64_t n, hipStream_t stream) {
    const uint64_t want = (n + 255) / 256;
    const uint32_t blocks = static_cast<uint32_t>(want < 8192 ? (want ? want : 1) : 8192);
    hipLaunchKernelGGL(fill_zero_kernel, dim3(blocks), dim3(256), 0, stream, p, n);
    return hipGetLastError();
}

}  // namespace supra_amd
