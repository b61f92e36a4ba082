// Envelope detection and log compression of beamformed images, the stages
// after the beamformer in SUPRA's B-mode chain:
//   HilbertFirEnvelope (src/SupraLib/Beamformer/HilbertFirEnvelope.cu:28-104,
//     the FIR Hilbert transformer of FirFilterFactory.h:55-200, filter length
//     65 by default, HilbertFirEnvelopeNode.cpp:42)
//   LogCompressor (src/SupraLib/Beamformer/LogCompressor.cu:20-64,
//     LogCompressorNode.cpp:42-45).
//
// Envelope layout: one workgroup per (64 scanlines, ROWS output samples,
// frame) of images [frame][sample][scanline]; lane = scanline, so every row of
// the window is one coalesced 256-byte load.  The workgroup stages the column
// window (ROWS + N - 1 rows) in LDS, loads issued eight rows at a time per
// wave before they are written.  Samples outside the image are staged as 0,
// which adds +-0 to the FIR sum where the reference skips them (the same
// value).  The FIR sum runs over the taps in ascending order in single
// precision without contraction, as the host restatement does, so the envelope
// is bit for bit the oracle's.
//
// Every second tap of a Hilbert transformer is 0.  It adds +-0 to the sum of a
// window of finite samples, so it is left out there: a lane takes 8 output
// rows of one parity, reads each input row of the other parity once and adds
// it to the up to 8 sums it belongs to, half the multiplications and a sixth
// of the LDS reads of a sum per row.  A workgroup whose window holds an
// infinity or a NaN (0 times it is NaN), and filters whose other taps are not
// all 0, sum every tap.  Bound by VALU: 64 multiplications and additions of a
// 65-tap filter per sample, about as many instructions again for the square
// root and the logarithm.  32 frames of 2080 x 128 to uint8: 28.3 us, 48.1 us with
// every tap and one sum per row.  ROWS is 64 where that leaves at least two
// workgroups per CU (fewer halo rows staged per output) and taps are left out,
// else 32.  The fused variant applies the log compression to the float envelope in
// registers (the same operations as the two-step path with a float intermediate).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdint>
#include <cstring>

#include "status.hpp"
#include "supra_bf.h"

namespace supra_amd {
namespace {

constexpr int kEnvOut = 8;            // output rows per lane, every second row of 16
constexpr int kEnvPadRows = 14;       // zero rows after the window: padded taps read them
constexpr int kMaxTaps = 257;         // HilbertFirEnvelopeNode's filterLength range (1..257)

struct EnvArgs {
    const void* in;
    void* out;
    uint32_t n_rx, n_s, n_taps, half;  // half = n_taps / 2 (window t - half .. t + half)
    uint32_t used_taps;               // taps that exist: min(n_taps, 2 half + 1)
    uint32_t parity, groups;          // taps parity, parity + 2, ... as groups of 8 in odd[]; groups 0: sum every tap
    float in_scale, scale_den;        // log compression (fused variant)
    float h[kMaxTaps];
    float odd[(kMaxTaps + 1) / 2 + 8];   // zero padded to whole groups
};

struct LogArgs {
    const void* in;
    void* out;
    uint64_t count;
    float in_scale, scale_den;
};

template <typename T> __device__ inline float load_as_float(const void* p, uint64_t i) {
    return static_cast<float>(static_cast<const T*>(p)[i]);
}

// clampCast (src/SupraLib/utilities/cudaUtility.h:111-147): fmaxf/fminf keep
// the non-NaN operand (NaN lands on the lower limit), then truncation.
template <typename T> __device__ inline T clamp_to(float x);
template <> __device__ inline float clamp_to<float>(float x) { return fminf(fmaxf(x, -FLT_MAX), FLT_MAX); }
template <> __device__ inline int16_t clamp_to<int16_t>(float x) {
    return static_cast<int16_t>(fminf(fmaxf(x, -32767.0f), 32767.0f));
}
template <> __device__ inline uint8_t clamp_to<uint8_t>(float x) {
    return static_cast<uint8_t>(fminf(fmaxf(x, 0.0f), 255.0f));
}

// thrustLogcompress::operator() (LogCompressor.cu:34-38).
__device__ inline float log_compress(float a, float in_scale, float scale_den) {
    return log10f(fabsf(a) * in_scale + 1.0f) * scale_den;
}

// Correctly rounded sqrt(x) of a finite x >= 2^-96 by one Newton step, as
// sqrt_rn in das_device.hpp; sqrtf where a lane of the wave has another x.
__device__ inline float wave_sqrt(float x) {
    if (__builtin_amdgcn_ballot_w64(!(x >= 0x1p-96f && x <= FLT_MAX)) != 0) return sqrtf(x);
    const float y = __builtin_amdgcn_rsqf(x);
    const float g = x * y;
    return fmaf(fmaf(-g, g, x), 0.5f * y, g);
}

template <typename OutT, bool LOG>
__device__ inline void store_envelope(const EnvArgs& a, OutT* out, uint64_t at, float v, float acc) {
    float env = wave_sqrt(v * v + acc * acc);
    // the fused path sees the envelope as the float image the two-node
    // chain passes on: clampCast<float> first (NaN -> -FLT_MAX, inf -> FLT_MAX)
    if (LOG) env = log_compress(clamp_to<float>(env), a.in_scale, a.scale_den);
    out[at] = clamp_to<OutT>(env);
}

// HALVED: the filter has groups of taps (else every tap is summed, and the kernel
// holds 16 registers instead of 63).
template <typename InT, typename OutT, bool LOG, int ROWS, bool HALVED>
__global__ __launch_bounds__(ROWS * 8) void envelope_kernel(const EnvArgs a) {
    constexpr uint32_t kWaves = ROWS / 8;
    extern __shared__ float win[];                 // [ROWS + 2 half + kEnvPadRows rows][64 lanes]
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)));
    const uint32_t s = blockIdx.x * 64u + lane;
    const uint32_t t0 = blockIdx.y * ROWS;
    const uint64_t frame = static_cast<uint64_t>(blockIdx.z) * a.n_s * a.n_rx;
    const uint32_t rows = ROWS + 2u * a.half, staged = rows + (HALVED ? kEnvPadRows : 0);
    const bool col = s < a.n_rx;
    const InT* in = static_cast<const InT*>(a.in) + frame;
    bool odd_value = false;                        // a staged value that is not finite
    for (uint32_t r0 = wave; r0 < staged; r0 += 8u * kWaves) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const uint32_t r = r0 + u * kWaves;
            const int64_t c = static_cast<int64_t>(t0) + r - a.half;
            v[u] = 0.0f;
            if (r < rows && col && c >= 0 && c < static_cast<int64_t>(a.n_s))
                v[u] = static_cast<float>(in[static_cast<uint64_t>(c) * a.n_rx + s]);
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const uint32_t r = r0 + u * kWaves;
            if (r < staged) win[r * 64u + lane] = v[u];
            if (sizeof(InT) == 4) odd_value |= !(fabsf(v[u]) <= FLT_MAX);
        }
    }
    bool every_tap = true;
    if constexpr (HALVED) every_tap = __syncthreads_or(odd_value);
    else __syncthreads();
    OutT* out = static_cast<OutT*>(a.out) + frame;
    if (every_tap) {
        if (!col) return;
        for (uint32_t i = wave; i < ROWS; i += kWaves) {
            const uint32_t t = t0 + i;
            if (t >= a.n_s) break;
            float acc = 0.0f;
#pragma unroll 8
            for (uint32_t j = 0; j < a.used_taps; j++) acc += win[(i + j) * 64u + lane] * a.h[j];
            store_envelope<OutT, LOG>(a, out, static_cast<uint64_t>(t) * a.n_rx + s, win[(i + a.half) * 64u + lane], acc);
        }
        return;
    }
    // output rows i0 + 2 m; tap parity + 2 q of row i0 + 2 m is window row
    // i0 + parity + 2 (m + q)
    const uint32_t i0 = (wave >> 1) * 16u + (wave & 1u);
    const float* x = win + (i0 + a.parity) * 64u + lane;
    float acc[kEnvOut], hp[8], hc[8];
#pragma unroll
    for (int m = 0; m < kEnvOut; m++) acc[m] = 0.0f;
#pragma unroll
    for (int q = 0; q < 8; q++) hc[q] = a.odd[q];
#pragma unroll
    for (int i = 0; i < 8; i++) {                  // rows m + q = 0 .. 7
        const float v = x[i * 128];
#pragma unroll
        for (int m = 0; m <= i; m++) acc[m] += v * hc[i - m];
    }
    for (uint32_t g = 1; g < a.groups; g++) {
        x += 8 * 128;
#pragma unroll
        for (int q = 0; q < 8; q++) {
            hp[q] = hc[q];
            hc[q] = a.odd[8 * g + q];
        }
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float v = x[i * 128];
#pragma unroll
            for (int m = 0; m < kEnvOut; m++) acc[m] += v * (i >= m ? hc[(i - m) & 7] : hp[(8 + i - m) & 7]);
        }
    }
    x += 8 * 128;
#pragma unroll
    for (int i = 0; i < 7; i++) {
        const float v = x[i * 128];
#pragma unroll
        for (int m = i + 1; m < kEnvOut; m++) acc[m] += v * hc[8 + i - m];
    }
    if (!col) return;
#pragma unroll
    for (int m = 0; m < kEnvOut; m++) {
        const uint32_t t = t0 + i0 + 2 * m;
        if (t < a.n_s)                             // uniform
            store_envelope<OutT, LOG>(a, out, static_cast<uint64_t>(t) * a.n_rx + s,
                                      win[(i0 + 2 * m + a.half) * 64u + lane], acc[m]);
    }
}

template <typename InT, typename OutT>
__global__ __launch_bounds__(256) void logcompress_kernel(const LogArgs a) {
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < a.count; i += stride)
        static_cast<OutT*>(a.out)[i] = clamp_to<OutT>(log_compress(load_as_float<InT>(a.in, i), a.in_scale, a.scale_den));
}

// FirFilterFactory::createFilter(N, FilterTypeHilbertTransformer,
// FilterWindowHamming): 2/(pi k) at odd offsets k from the centre, 0 at even
// ones, in double then float, times the float Hamming window.
void hilbert_taps(uint32_t n, float* h) {
    const int half = (static_cast<int>(n) - 1) / 2;
    const size_t max_n = n - 1;
    for (uint32_t i = 0; i < n; i++) {
        const int k = static_cast<int>(i) - half;
        h[i] = (k % 2 == 0) ? 0.0f : static_cast<float>(2.0 / (M_PI * k));
        h[i] *= static_cast<float>(0.54 - 0.46 * std::cos(2 * M_PI * i / max_n));
    }
}

// thrustLogcompress's constructor (LogCompressor.cu:28-31, :56-60): inMax is
// converted to the input element type first, outMax is 255 for both the
// float and the uint8 image.
void log_constants(int in_dtype, double dynamic_range_db, double gain, double in_max, float* in_scale,
                   float* scale_den) {
    const double dr = std::pow(10.0, dynamic_range_db / 20);
    double m = in_max;
    if (in_dtype == SUPRA_INT16) m = static_cast<int16_t>(in_max);
    else if (in_dtype == SUPRA_UINT8) m = static_cast<uint8_t>(in_max);
    else m = static_cast<float>(in_max);
    *in_scale = static_cast<float>(dr / m);
    *scale_den = static_cast<float>(gain * 255.0 / std::log10(dr + 1));
}

int check_types(const char* what, int in_dtype, int out_dtype, bool allow_u8_in, bool allow_i16_out, bool allow_u8_out) {
    const bool in_ok = in_dtype == SUPRA_FLOAT32 || in_dtype == SUPRA_INT16 || (allow_u8_in && in_dtype == SUPRA_UINT8);
    const bool out_ok = out_dtype == SUPRA_FLOAT32 || (allow_i16_out && out_dtype == SUPRA_INT16) ||
                        (allow_u8_out && out_dtype == SUPRA_UINT8);
    if (!in_ok || !out_ok) return fail(SUPRA_ERR_UNSUPPORTED, "%s: element types %d -> %d are not provided", what,
                                       in_dtype, out_dtype);
    return SUPRA_OK;
}

template <bool LOG, typename InT, typename OutT>
void launch_env_typed(const EnvArgs& a, uint32_t n_frames, hipStream_t s) {
    const uint32_t columns = (a.n_rx + 63) / 64;
    const bool halved = a.groups != 0;
    const size_t window = static_cast<size_t>(2 * a.half + (halved ? kEnvPadRows : 0));
    // tall tiles where at least 512 workgroups (two per CU) remain; a filter that
    // sums every tap gains nothing from them (32 frames of 2080 x 128 to
    // uint8, 1 tap: 21.6 us, 17.3 with short ones, no padding and no registers
    // for the groups)
    const dim3 short_tiles(columns, (a.n_s + 31) / 32, n_frames);
    if (!halved)
        hipLaunchKernelGGL((envelope_kernel<InT, OutT, LOG, 32, false>), short_tiles, dim3(256), (32 + window) * 256, s, a);
    else if (static_cast<uint64_t>(columns) * ((a.n_s + 63) / 64) * n_frames >= 512)
        hipLaunchKernelGGL((envelope_kernel<InT, OutT, LOG, 64, true>), dim3(columns, (a.n_s + 63) / 64, n_frames), dim3(512),
                           (64 + window) * 256, s, a);
    else
        hipLaunchKernelGGL((envelope_kernel<InT, OutT, LOG, 32, true>), short_tiles, dim3(256), (32 + window) * 256, s, a);
}

template <bool LOG>
int launch_envelope(const char* what, const void* image, int in_dtype, uint32_t n_rx, uint32_t n_s,
                    uint32_t n_frames, uint32_t filter_length, float in_scale, float scale_den, void* out,
                    int out_dtype, void* stream) {
    if (!image || !out) return fail(SUPRA_ERR_INVALID_ARG, "%s: null argument", what);
    if (n_frames > 65535u) return fail(SUPRA_ERR_TOO_LARGE, "%s: %u frames in one call (at most 65535)", what, n_frames);
    if (n_rx == 0 || n_s == 0 || n_frames == 0) return SUPRA_OK;
    if (filter_length < 1 || filter_length > kMaxTaps)
        return fail(SUPRA_ERR_INVALID_ARG, "%s: filter length %u outside [1, %d]", what, filter_length, kMaxTaps);
    int st = check_types(what, in_dtype, out_dtype, false, !LOG, LOG);
    if (st != SUPRA_OK) return st;
    if (static_cast<uint64_t>(n_s) * n_rx >= (1ull << 40)) return fail(SUPRA_ERR_TOO_LARGE, "%s: image too large", what);
    EnvArgs a;
    std::memset(&a, 0, sizeof(a));
    a.in = image;
    a.out = out;
    a.n_rx = n_rx;
    a.n_s = n_s;
    a.n_taps = filter_length;
    a.half = filter_length / 2;
    a.used_taps = std::min(filter_length, 2 * a.half + 1);
    a.in_scale = in_scale;
    a.scale_den = scale_den;
    hilbert_taps(filter_length, a.h);
    a.parity = ((filter_length - 1) / 2 + 1) % 2;
    bool halved = filter_length > 1;
    for (uint32_t j = 0; j < a.used_taps; j++) {
        if (j % 2 == a.parity) a.odd[j / 2] = a.h[j];
        else halved = halved && a.h[j] == 0.0f;
    }
    const uint32_t n_odd = a.used_taps > a.parity ? (a.used_taps - a.parity + 1) / 2 : 0;
    a.groups = halved ? (n_odd + 7) / 8 : 0;
    if ((n_s + 31) / 32 > 65535u) return fail(SUPRA_ERR_TOO_LARGE, "%s: too many samples per scanline", what);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (in_dtype == SUPRA_INT16) {
        if (out_dtype == SUPRA_FLOAT32) launch_env_typed<LOG, int16_t, float>(a, n_frames, s);
        else if (out_dtype == SUPRA_INT16) launch_env_typed<LOG, int16_t, int16_t>(a, n_frames, s);
        else launch_env_typed<LOG, int16_t, uint8_t>(a, n_frames, s);
    } else {
        if (out_dtype == SUPRA_FLOAT32) launch_env_typed<LOG, float, float>(a, n_frames, s);
        else if (out_dtype == SUPRA_INT16) launch_env_typed<LOG, float, int16_t>(a, n_frames, s);
        else launch_env_typed<LOG, float, uint8_t>(a, n_frames, s);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(SUPRA_ERR_HIP, "%s: launch: %s", what, hipGetErrorString(e));
    return SUPRA_OK;
}

template <typename InT, typename OutT>
void launch_log_typed(const LogArgs& a, hipStream_t s) {
    const uint64_t blocks = std::min<uint64_t>((a.count + 255) / 256, 256ull * 64ull);
    hipLaunchKernelGGL((logcompress_kernel<InT, OutT>), dim3(static_cast<uint32_t>(blocks)), dim3(256), 0, s, a);
}

}  // namespace
}  // namespace supra_amd

using namespace supra_amd;

extern "C" int supra_envelope_run(const void* image, int32_t in_dtype, uint32_t num_scanlines, uint32_t num_samples,
                                  uint32_t num_frames, uint32_t filter_length, void* out, int32_t out_dtype,
                                  void* stream) {
    clear_error();
    return launch_envelope<false>("envelope", image, in_dtype, num_scanlines, num_samples, num_frames, filter_length,
                                  0.0f, 0.0f, out, out_dtype, stream);
}

extern "C" int supra_logcompress_run(const void* in, int32_t in_dtype, uint64_t count, double dynamic_range_db,
                                     double gain, double in_max, void* out, int32_t out_dtype, void* stream) {
    clear_error();
    if (!in || !out) return fail(SUPRA_ERR_INVALID_ARG, "logcompress: null argument");
    int st = check_types("logcompress", in_dtype, out_dtype, true, false, true);
    if (st != SUPRA_OK) return st;
    if (count == 0) return SUPRA_OK;
    LogArgs a;
    a.in = in;
    a.out = out;
    a.count = count;
    log_constants(in_dtype, dynamic_range_db, gain, in_max, &a.in_scale, &a.scale_den);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool f32 = out_dtype == SUPRA_FLOAT32;
    if (in_dtype == SUPRA_INT16) f32 ? launch_log_typed<int16_t, float>(a, s) : launch_log_typed<int16_t, uint8_t>(a, s);
    else if (in_dtype == SUPRA_UINT8) f32 ? launch_log_typed<uint8_t, float>(a, s) : launch_log_typed<uint8_t, uint8_t>(a, s);
    else f32 ? launch_log_typed<float, float>(a, s) : launch_log_typed<float, uint8_t>(a, s);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(SUPRA_ERR_HIP, "logcompress: launch: %s", hipGetErrorString(e));
    return SUPRA_OK;
}

extern "C" int supra_envelope_logcompress_run(const void* image, int32_t in_dtype, uint32_t num_scanlines,
                                              uint32_t num_samples, uint32_t num_frames, uint32_t filter_length,
                                              double dynamic_range_db, double gain, double in_max, void* out,
                                              int32_t out_dtype, void* stream) {
    clear_error();
    float in_scale, scale_den;
    log_constants(SUPRA_FLOAT32, dynamic_range_db, gain, in_max, &in_scale, &scale_den);
    return launch_envelope<true>("envelope + logcompress", image, in_dtype, num_scanlines, num_samples, num_frames,
                                 filter_length, in_scale, scale_den, out, out_dtype, stream);
}
