// Arguments and launchers of the scans whose output contraction runs on the
// matrix cores (mfma_scan.hip).
#pragma once

#include "mi_common.hpp"

namespace mi {

enum MfmaScanMode { kMScanModel = 0, kMScanChannel = 1, kMScanHead = 2, kMScanSsd = 3 };

struct MfmaScanArgs {
    const int8_t *x;         // [B*L][x_row]: the model's xs, else x
    const int8_t *dm;        // model: [B*L][x_row]
    const int8_t *z;         // gated modes: [B*L][z_row], at its first column
    const int8_t *b, *c;     // B and C rows of the first head, row stride bc_row
    const int8_t *dtc;       // SSD: the dt column of the first head, row stride bc_row
    const int32_t *decay;    // model: base [D][N]; channel: [D][N]; head: [H]; SSD: table [H][255]
    int8_t *yo;              // gated modes: [B*L][x_row]
    int32_t *y;              // channel and head modes: [B*L][x_row]
    int32_t *chunk_states;   // head mode, nullable: [B][nchunks_out][D][N]
    const int32_t *h_in;     // [B][D][N], nullable
    int32_t *h_out;
    int64_t x_row, z_row, bc_row;
    int B, L, D;             // D: channels of a row (over all heads)
    int P;                   // head and SSD modes: channels of a head
    int s_y;                 // gated modes
    int cs, nchunks_out;     // head mode
};

// The longest sequences that the mode's VALU kernel (scan_kernel, model_scan_kernel,
// ssd_scan_kernel) takes instead of the MFMA scan; D channels of a row, P of a head.
int valu_scan_steps(int mode, int N, int B, int D, int P);

// A chunk's rows are addressed by 32-bit byte offsets, so rows stay below this:
// 64 of them, as int32 outputs, below 2^31 bytes.
constexpr int64_t kMfmaMaxRow = (int64_t)1 << 22;

// N in {16, 32, 64} (channel and head modes also 128), decay shift 15, D and P
// multiples of 16, 16-byte aligned rows shorter than kMfmaMaxRow, at least one step.
hipError_t launch_mfma_scan(int mode, int N, const MfmaScanArgs &a, hipStream_t st);

}  // namespace mi
