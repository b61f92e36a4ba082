// The engine context shared by the entry points of the library, and the
// host helpers that build its dt-space tables.
#pragma once

#include <hip/hip_runtime.h>

#include <mutex>
#include <vector>

#include "bf_internal.hpp"
#include "supra_bf.h"

using supra_amd::ScanlineDT;

struct supra_bf_ctx {
    int device = 0;
    uint32_t n_rx = 0, rx_layout[2] = {0, 0}, n_depths = 0, n_el = 0, el_layout[2] = {0, 0};
    bool is3d = false;
    std::vector<supra_scanline_rx> scan_mm;
    std::vector<float> depths_mm, ex_mm, ey_mm;
    std::vector<int32_t> e2c;
    double geom_c = 0, depth_mm = 0;
    uint32_t max_channel_in_map = 0;

    ScanlineDT* d_scans = nullptr;
    float* d_depths = nullptr;
    float* d_ex = nullptr;
    float* d_ey = nullptr;
    int32_t* d_e2c = nullptr;

    std::vector<ScanlineDT> h_scans;
    std::vector<float> h_depths, h_ex, h_ey;
    double cached_dt = 0, cached_c = 0;
    // Launches have read d_scans/d_depths/d_ex/d_ey since their upload, on
    // these streams (the first kTableStreams distinct ones): an upload for
    // another (dt, c) waits for them.  tables_captured: a launch was captured
    // (and may be replayed at any time, on any stream).
    static constexpr size_t kTableStreams = 16;
    bool tables_used = false, more_table_streams = false, tables_captured = false;
    std::vector<hipStream_t> table_streams;
    // Transmits that the selected, resp. all weighted transmits of the
    // scanlines address (largest index + 1).
    uint64_t tx_selected = 0, tx_weighted = 0;
    // The last window table of the delay-and-sum entry points.
    int32_t lut_type = -1;
    float lut_parameter = 0.0f, lut[supra_amd::kWindowEntries];
    bool far_ok = false;   // dt-space depths are >= 0 and non-decreasing
    bool grid_ok = false;     // 3D: dt-space element (ix, iy) is at (X[ix], Z[iy])
    uint32_t max_rows = 0;    // 3D: largest last_y - first_y over scanlines and transmits
    bool far_ok_mm = false;   // the same for the millimetre depths (any c)
    bool nan_positions = false;   // some scanline's or element's position is NaN
    bool nan_lines = false;   // some transmit's delay or scanline's direction is NaN
    std::mutex mu;

    // Differentiable path: the millimetre geometry on the device, the
    // c-independent part of the scanline records, per-frame tables and
    // scratch, grown on demand.
    supra_scanline_rx* d_scan_mm = nullptr;
    ScanlineDT* d_scan_fixed = nullptr;
    float* d_depths_mm = nullptr;
    float* d_ex_mm = nullptr;
    void* d_frame_tables = nullptr;
    size_t frame_tables_cap = 0;
    void* d_beta = nullptr;
    size_t beta_cap = 0;
    void* d_dc_part = nullptr;
    size_t dc_part_cap = 0;
    // Writers of each (transmit, channel) RF line for the adjoint, cached per
    // (transmit interpolation, num_tx, num_channels).
    int lines_key_interp = -1;
    uint32_t lines_key_tx = 0, lines_key_ch = 0;
    bool lines_exclusive = false;
    uint32_t n_zero_lines = 0;
    uint32_t* d_zero_lines = nullptr;
    uint32_t max_aperture = 0;   // largest last_x - first_x over scanlines and transmits
    // This device's copy of the file-scope scratch array of the
    // allocation-free forward (shared by every context on the device; not owned).
    void* noalloc_scratch = nullptr;

    ~supra_bf_ctx() {
        (void)hipFree(d_scans);
        (void)hipFree(d_depths);
        (void)hipFree(d_ex);
        (void)hipFree(d_ey);
        (void)hipFree(d_e2c);
        (void)hipFree(d_scan_mm);
        (void)hipFree(d_scan_fixed);
        (void)hipFree(d_depths_mm);
        (void)hipFree(d_ex_mm);
        (void)hipFree(d_frame_tables);
        (void)hipFree(d_beta);
        (void)hipFree(d_dc_part);
        (void)hipFree(d_zero_lines);
    }
};


namespace supra_amd {

int hip_fail(hipError_t e, const char* what);
// RxBeamformerCuda::convertToDtSpace restated from the millimetre geometry
// into the context's host tables (h_scans, h_depths, h_ex, h_ey).
void build_dt_tables(supra_bf_ctx* ctx, double dt, double c);
int ensure_dt_tables(supra_bf_ctx* ctx, double dt, double c, hipStream_t stream);
int check_device(const supra_bf_ctx* ctx);
void tables_used_on(supra_bf_ctx* ctx, hipStream_t stream);
// build_window_lut() through the context's copy of the last table.
void context_window_lut(supra_bf_ctx* ctx, int32_t window_type, float window_parameter, float* lut);
int check_rawdelay_call(const supra_bf_ctx* ctx, const char* what, int32_t rf_dtype, uint32_t num_tx,
                        uint32_t num_channels, uint32_t num_samples, double fs, double f_number, double c,
                        int32_t window_type, bool allow3d);
DasArgs rawdelay_args(const supra_bf_ctx* ctx, const void* rf, uint32_t num_tx, uint32_t num_channels,
                      uint32_t num_samples, double dt, double f_number, double c, int32_t window_type,
                      float window_parameter);

}  // namespace supra_amd
