// Dyadic selective scans (spec mi-spec-2, rule 1 and 4.7-4.11): entry points, the
// plain int64 kernels for every shape the fast kernels (mfma_scan.hip,
// model_scan.hip) do not take, and the elementwise forms.
//
// The recurrence h_t = sat32(floor(h_{t-1} * n / 2^k) + u_t) is not
// associative (the floor does not compose), so exact parallelism comes only
// from independent lanes: (batch, head, channel, state).  Time stays
// sequential inside every lane.
#include <algorithm>
#include <type_traits>

#include "mi_common.hpp"
#include "mfma_scan.hpp"

namespace mi {
namespace {

// steps that scan_kernel stages at a time; chunk lengths of chunk_states are multiples
// of it in the fast kernels (their staged chunks divide it)
constexpr int kTC = 64;

enum ScanMode { kModeChannel = 0, kModeHead = 1, kModeModel = 2 };

struct ScanArgs {
    const int8_t *x;       // channel/head modes: x; model mode: xs
    const int8_t *bsrc;    // B rows
    const int8_t *csrc;    // C rows
    const int32_t *decay;  // [P][N] (channel), [H] (head), base [P][N] (model)
    int32_t *y;            // int32 y (channel/head)
    int8_t *yo;            // int8 gated output (model)
    int32_t *chunk_states; // head mode, nullable
    const int32_t *h_in;
    int32_t *h_out;
    const int8_t *dm;      // model
    const int8_t *z;       // model
    int64_t x_row;         // element stride between consecutive (b,t) rows of x/y (= H*P)
    int64_t bc_row;        // stride between consecutive (b,t) rows of B/C
    int64_t z_row;         // model: row stride of z
    int B, L, H, P;
    int k;
    int s_y;
    int nchunks_out;       // head mode: number of chunk_states chunks (ceil(L/cs))
    int cs;                // head mode: chunk length of chunk_states
};

// ---------------------------------------------------------------- generic
// Plain int64 kernels for every shape the fast kernel does not take, and for
// chunk lengths that are not multiples of the staging chunk.  One thread per
// (b, head, channel), all states in a loop, inputs read straight from global.
template <int MODE>
__global__ __launch_bounds__(256) void scan_generic_kernel(ScanArgs a, int N) {
    const int64_t lane = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t lanes = (int64_t)a.B * a.H * a.P;
    if (lane >= lanes) return;
    const int p = (int)(lane % a.P);
    const int hd = (int)((lane / a.P) % a.H);
    const int b = (int)(lane / ((int64_t)a.P * a.H));
    int32_t h[128];
    const int64_t sidx = (((int64_t)b * a.H + hd) * a.P + p) * N;
    for (int n = 0; n < N; ++n) h[n] = a.h_in ? a.h_in[sidx + n] : 0;
    for (int t = 0; t < a.L; ++t) {
        const int64_t rr = (int64_t)b * a.L + t;
        int64_t xv;
        int dmv = 0;
        const int8_t *brow, *crow;
        if constexpr (MODE == kModeModel) {
            dmv = clamp32(a.dm[rr * a.x_row + p], -20, 20);
            xv = rshr64((int64_t)a.x[rr * a.x_row + p] * dt_q16(dmv), 10);
            brow = a.bsrc + rr * a.bc_row;
            crow = a.csrc + rr * a.bc_row;
        } else {
            xv = a.x[rr * a.x_row + (int64_t)hd * a.P + p];
            brow = a.bsrc + rr * a.bc_row + (MODE == kModeHead ? (int64_t)hd * N : 0);
            crow = a.csrc + rr * a.bc_row + (MODE == kModeHead ? (int64_t)hd * N : 0);
        }
        int64_t acc = 0;
        for (int n = 0; n < N; ++n) {
            int64_t nd;
            if constexpr (MODE == kModeChannel) nd = a.decay[(int64_t)p * N + n];
            else if constexpr (MODE == kModeHead) nd = a.decay[hd];
            else nd = clamp64((int64_t)a.decay[(int64_t)p * N + n] + dmv, 0, 32000);
            const int64_t dec = ((int64_t)h[n] * nd) >> a.k;
            h[n] = sat32_64(dec + (int64_t)brow[n] * xv);
            acc += (int64_t)crow[n] * h[n];
        }
        const int32_t y32 = sat32_64(acc);
        if constexpr (MODE == kModeModel) {
            const int zv = a.z[rr * a.z_row + p];
            const int64_t yg = ((int64_t)y32 * gate_q15(zv)) >> 15;
            a.yo[rr * a.x_row + p] = (int8_t)clamp64(rshr64(yg, a.s_y), -127, 127);
        } else {
            a.y[rr * a.x_row + (int64_t)hd * a.P + p] = y32;
        }
        if constexpr (MODE == kModeHead) {
            if (a.chunk_states && ((t + 1) % a.cs == 0 || t + 1 == a.L)) {
                const int cc = t / a.cs;
                int32_t *dst = a.chunk_states + ((((int64_t)b * a.nchunks_out + cc) * a.H + hd) * a.P + p) * N;
                for (int n = 0; n < N; ++n) dst[n] = h[n];
            }
        }
    }
    if (a.h_out)
        for (int n = 0; n < N; ++n) a.h_out[sidx + n] = h[n];
}

// -------------------------------------------------- VALU scan, short calls
// The channel and head layouts where a sequence has few steps (launch_scan has the
// lengths: a block of the MFMA scan starts slower, with its helper waves' staging, a
// barrier a chunk and mostly one block a CU) or rows too long for that kernel's
// offsets.  A block owns CH = 256/G channels of one (batch,
// head); G adjacent lanes share a channel and hold S = N/G states each, read as two
// 16-bit fields by the update (update16); their partial y sums are combined by DPP.
// Inputs of 64 steps go through LDS, x transposed to channel-major so one
// ds_read_b32 serves four steps, outputs leave through LDS in 16-byte stores.
constexpr int kThreads = 256;

// Sums of K independent values over the G adjacent lanes of a channel, stage by
// stage across all K (a DPP add then reads a register written K instructions
// earlier, so no wait states); every lane gets them.
template <int G, int K>
__device__ __forceinline__ void group_sums(int (&v)[K]) {
#pragma unroll
    for (int k = 0; k < K; ++k)
        if constexpr (G >= 2) v[k] += __builtin_amdgcn_update_dpp(0, v[k], 0xB1, 0xF, 0xF, false);   // quad_perm 1,0,3,2
#pragma unroll
    for (int k = 0; k < K; ++k)
        if constexpr (G >= 4) v[k] += __builtin_amdgcn_update_dpp(0, v[k], 0x4E, 0xF, 0xF, false);   // quad_perm 2,3,0,1
#pragma unroll
    for (int k = 0; k < K; ++k)
        if constexpr (G >= 8) v[k] += __builtin_amdgcn_update_dpp(0, v[k], 0x141, 0xF, 0xF, false);  // row_half_mirror
#pragma unroll
    for (int k = 0; k < K; ++k)
        if constexpr (G >= 16) v[k] += __builtin_amdgcn_update_dpp(0, v[k], 0x140, 0xF, 0xF, false); // row_mirror
}

__device__ __forceinline__ int sbyte(uint32_t w, int i) { return (int)(int8_t)(w >> (8 * i)); }

// Loads 16 consecutive bytes (16-byte aligned) or zeros when out of range.
__device__ __forceinline__ uint4 load16(const int8_t *p, bool ok) {
    if (ok) return *reinterpret_cast<const uint4 *>(p);
    return make_uint4(0, 0, 0, 0);
}

template <int N, int G, int MODE>
__global__ __launch_bounds__(kThreads) void scan_kernel(ScanArgs a) {
    static_assert(MODE != kModeModel, "the fused model scan has its own kernel (model_scan.hip)");
    constexpr int S = N / G;
    constexpr int CH = kThreads / G;
    constexpr int XP = kTC + 4;                 // padded row of the transposed x tile
    constexpr int X16 = CH / 16;                // 16-byte pieces per time row of x
    constexpr int XPIECES = kTC * X16;          // per chunk
    constexpr int XPER = (XPIECES + kThreads - 1) / kThreads;
    constexpr int BC16 = N / 16;
    constexpr int BCPIECES = kTC * BC16;
    constexpr int BCPER = (BCPIECES + kThreads - 1) / kThreads;

    __shared__ __align__(16) int8_t s_x[CH][XP];
    // WIDEB: B widened to int32, so the input term B * x and the saturating
    // add are one clamped v_mad_i32_i24 (which takes no SDWA byte select).
    // Lanes of one or two states keep B as bytes: their latency-bound chain
    // measured slower with the wider staging (config 1: 22.0 -> 25.1 us)
    constexpr bool WIDEB = S >= 4;
    constexpr bool STAGE_Y = CH <= 64;  // int32 y staged in LDS (16 KB at most)
    // blocks of <= 32 channels (G >= 8) reduce the y partials of four steps
    // together and park the exact (yhi, ylo) pairs here; the chunk epilogue
    // recombines and saturates once per (step, channel)
    constexpr bool DEFER = CH <= 32;
    // C32: C staged as int32 C * 2^16 as well (update16_cs: y's high partial in one
    // v_dot2c, no byte extraction per state), in the channel layout (64 rounds of N =
    // 16, 48 steps 73 -> 66 us) where two blocks a CU still fit
    constexpr int kLdsC32 = CH * (kTC + 4) + 2 * kTC * N * 4 + (STAGE_Y ? kTC * CH * 4 : 16) + (DEFER ? kTC * CH * 8 : 8);
    constexpr bool C32 = WIDEB && MODE == kModeChannel && kLdsC32 <= 81920;
    __shared__ __align__(16) std::conditional_t<WIDEB, int32_t, int8_t> s_b[kTC][N];
    __shared__ __align__(16) std::conditional_t<C32, int32_t, int8_t> s_c[kTC][N];
    __shared__ __align__(16) int32_t s_o32[STAGE_Y ? kTC : 1][STAGE_Y ? CH : 4];
    __shared__ __align__(16) int2 s_y[DEFER ? kTC : 1][DEFER ? CH : 1];

    const int tid = threadIdx.x;
    const int ch = tid / G;
    const int g = tid % G;
    const int p0 = blockIdx.x * CH;
    const int hd = blockIdx.y;
    const int b = blockIdx.z;
    const int p = p0 + ch;
    const bool active = p < a.P;

    // ---- per-thread constants and state
    int32_t n2[S];  // 2n: the update16 form takes the doubled decay
    int32_t h[S];
    {
        const int64_t sidx = ((((int64_t)b * a.H + hd) * a.P + (active ? p : 0)) * N) + g * S;
        for (int s = 0; s < S; ++s) {
            h[s] = (a.h_in && active) ? a.h_in[sidx + s] : 0;
            if constexpr (MODE == kModeChannel)
                n2[s] = 2 * (active ? a.decay[(int64_t)p * N + g * S + s] : 0);
            else
                n2[s] = 2 * a.decay[hd];
        }
    }

    // ---- staging registers
    uint4 rx[XPER];
    uint4 rb[BCPER], rc[BCPER];
    const int64_t row0 = (int64_t)b * a.L;  // first (b, t=0) row index

    auto prefetch = [&](int t0) {
        for (int j = 0; j < XPER; ++j) {
            const int i = tid + j * kThreads;
            const int tt = i / X16, c16 = i % X16;
            const bool ok = i < XPIECES && t0 + tt < a.L && p0 + c16 * 16 < a.P;
            rx[j] = load16(a.x + (row0 + t0 + tt) * a.x_row + (int64_t)hd * a.P + p0 + c16 * 16, ok);
        }
        for (int j = 0; j < BCPER; ++j) {
            const int i = tid + j * kThreads;
            const int tt = i / BC16, c16 = i % BC16;
            const bool ok = i < BCPIECES && t0 + tt < a.L;
            const int64_t off = (row0 + t0 + tt) * a.bc_row + (MODE == kModeHead ? (int64_t)hd * N : 0) + c16 * 16;
            rb[j] = load16(a.bsrc + off, ok);
            rc[j] = load16(a.csrc + off, ok);
        }
    };
    auto stash = [&]() {
        for (int j = 0; j < XPER; ++j) {
            const int i = tid + j * kThreads;
            if (i >= XPIECES) break;
            const int tt = i / X16, c16 = i % X16;
            const uint32_t w[4] = {rx[j].x, rx[j].y, rx[j].z, rx[j].w};
            for (int e = 0; e < 16; ++e) s_x[c16 * 16 + e][tt] = (int8_t)(w[e >> 2] >> (8 * (e & 3)));
        }
        for (int j = 0; j < BCPER; ++j) {
            const int i = tid + j * kThreads;
            if (i >= BCPIECES) break;
            const int tt = i / BC16, c16 = i % BC16;
            if constexpr (WIDEB) {
                const uint32_t w[4] = {rb[j].x, rb[j].y, rb[j].z, rb[j].w};
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<int4 *>(&s_b[tt][c16 * 16 + 4 * q]) =
                        make_int4(sbyte(w[q], 0), sbyte(w[q], 1), sbyte(w[q], 2), sbyte(w[q], 3));
            } else {
                *reinterpret_cast<uint4 *>(&s_b[tt][c16 * 16]) = rb[j];
            }
            if constexpr (C32) {
                const uint32_t w[4] = {rc[j].x, rc[j].y, rc[j].z, rc[j].w};
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<int4 *>(&s_c[tt][c16 * 16 + 4 * q]) = make_int4(
                        sbyte(w[q], 0) * 65536, sbyte(w[q], 1) * 65536, sbyte(w[q], 2) * 65536, sbyte(w[q], 3) * 65536);
            } else {
                *reinterpret_cast<uint4 *>(&s_c[tt][c16 * 16]) = rc[j];
            }
        }
    };

    // one step of this lane's S states: the exact int32 partials of y
    auto step = [&](int t, int xv, int &yhi, int &ylo) {
        yhi = 0;
        ylo = 0;
        if constexpr (C32) {
            // every coefficient read first, then the S updates
            int bv[S], cv[S];
#pragma unroll
            for (int q = 0; q < S / 4; ++q) {
                const int4 b4 = *reinterpret_cast<const int4 *>(&s_b[t][g * S + 4 * q]);
                const int4 c4 = *reinterpret_cast<const int4 *>(&s_c[t][g * S + 4 * q]);
                bv[4 * q] = b4.x; bv[4 * q + 1] = b4.y; bv[4 * q + 2] = b4.z; bv[4 * q + 3] = b4.w;
                cv[4 * q] = c4.x; cv[4 * q + 1] = c4.y; cv[4 * q + 2] = c4.z; cv[4 * q + 3] = c4.w;
            }
#pragma unroll
            for (int s = 0; s < S; ++s) update16_cs(h[s], n2[s], bv[s], xv, cv[s], yhi, ylo);
        } else if constexpr (WIDEB) {
            // every coefficient read first, then the S updates
            int bv[S];
            uint32_t cw[S / 4];
#pragma unroll
            for (int q = 0; q < S / 4; ++q) {
                const int4 b4 = *reinterpret_cast<const int4 *>(&s_b[t][g * S + 4 * q]);
                bv[4 * q] = b4.x; bv[4 * q + 1] = b4.y; bv[4 * q + 2] = b4.z; bv[4 * q + 3] = b4.w;
                cw[q] = *reinterpret_cast<const uint32_t *>(&s_c[t][g * S + 4 * q]);
            }
#pragma unroll
            for (int s = 0; s < S; ++s) update16_b(h[s], n2[s], bv[s], xv, sbyte(cw[s >> 2], s & 3), yhi, ylo);
        } else {
            uint32_t bw = 0, cw = 0;
            for (int s = 0; s < S; ++s) {
                bw |= (uint32_t)(uint8_t)s_b[t][g * S + s] << (8 * s);
                cw |= (uint32_t)(uint8_t)s_c[t][g * S + s] << (8 * s);
            }
#pragma unroll
            for (int s = 0; s < S; ++s) update16(h[s], n2[s], __mul24(sbyte(bw, s), xv), sbyte(cw, s), yhi, ylo);
        }
    };

    const int nchunks = (a.L + kTC - 1) / kTC;
    prefetch(0);
    for (int cidx = 0; cidx < nchunks; ++cidx) {
        const int t0 = cidx * kTC;
        const int tn = min(kTC, a.L - t0);
        __syncthreads();
        stash();
        __syncthreads();
        if (cidx + 1 < nchunks) prefetch(t0 + kTC);

        for (int t4 = 0; t4 < tn; t4 += 4) {
            const uint32_t xw = *reinterpret_cast<const uint32_t *>(&s_x[ch][t4]);
            const int tend = min(4, tn - t4);
            if constexpr (DEFER) {
                if (tend == 4) {
                    int y[8];
#pragma unroll
                    for (int tt = 0; tt < 4; ++tt) step(t4 + tt, sbyte(xw, tt), y[2 * tt], y[2 * tt + 1]);
                    group_sums<G>(y);
#pragma unroll
                    for (int tt = 0; tt < 4; ++tt) s_y[t4 + tt][ch] = make_int2(y[2 * tt], y[2 * tt + 1]);
                } else {
                    for (int tt = 0; tt < tend; ++tt) {
                        int y[2];
                        step(t4 + tt, sbyte(xw, tt), y[0], y[1]);
                        group_sums<G>(y);
                        s_y[t4 + tt][ch] = make_int2(y[0], y[1]);
                    }
                }
                continue;
            }
            for (int tt = 0; tt < tend; ++tt) {
                const int t = t4 + tt;
                int y[2];
                step(t, sbyte(xw, tt), y[0], y[1]);
                group_sums<G>(y);
                const int32_t y32 = sat32_64(((int64_t)y[0] << 16) + y[1]);
                if (g == 0) {
                    if constexpr (STAGE_Y) s_o32[t][ch] = y32;
                    else if (active) a.y[(row0 + t0 + t) * a.x_row + (int64_t)hd * a.P + p] = y32;
                }
            }
        }
        __syncthreads();
        if constexpr (DEFER) {
            // chunk epilogue: y = sat32(yhi * 2^16 + ylo)
            for (int i = tid; i < kTC * CH; i += kThreads) {
                const int tt = i / CH, cc = i % CH;
                if (tt < tn) {
                    const int2 yv = s_y[tt][cc];
                    s_o32[tt][cc] = sat32_64(((int64_t)yv.x << 16) + yv.y);
                }
            }
            __syncthreads();
        }
        // ---- write the staged outputs of this chunk
        if constexpr (STAGE_Y) {
            constexpr int Y4 = CH / 4;
            for (int i = tid; i < kTC * Y4; i += kThreads) {
                const int tt = i / Y4, c4 = i % Y4;
                if (tt < tn && p0 + c4 * 4 < a.P)
                    *reinterpret_cast<uint4 *>(a.y + (row0 + t0 + tt) * a.x_row + (int64_t)hd * a.P + p0 + c4 * 4) =
                        *reinterpret_cast<const uint4 *>(&s_o32[tt][c4 * 4]);
            }
        }
        if constexpr (MODE == kModeHead) {
            // chunk_states at every multiple of cs (cs is a multiple of kTC) and at the end
            const int tdone = t0 + tn;
            if (a.chunk_states && active && (tdone % a.cs == 0 || tdone == a.L)) {
                const int cc = (tdone - 1) / a.cs;
                int32_t *dst = a.chunk_states +
                               ((((int64_t)b * a.nchunks_out + cc) * a.H + hd) * a.P + p) * N + g * S;
                for (int s = 0; s < S; ++s) dst[s] = h[s];
            }
        }
    }
    if (a.h_out && active) {
        const int64_t sidx = ((((int64_t)b * a.H + hd) * a.P + p) * N) + g * S;
        for (int s = 0; s < S; ++s) a.h_out[sidx + s] = h[s];
    }
}


// Lanes per channel: enough waves to cover the 1024 SIMDs when possible.
int pick_g(int N, int64_t channels) {
    int g = 1;
    while (g < 16 && N % (2 * g) == 0 && (N / g > 32 || channels * g / 64 < 1024)) g *= 2;
    return g;
}

template <int N, int MODE>
hipError_t launch_valu_n(const ScanArgs &a, hipStream_t st) {
    auto grid = [&](int ch) { return dim3((unsigned)((a.P + ch - 1) / ch), (unsigned)a.H, (unsigned)a.B); };
    const int g = pick_g(N, (int64_t)a.B * a.H * a.P);
#define MI_CASE_G(GG)                                                                                     \
    if constexpr (N / GG <= 32)                                                                           \
        if (g == GG) hipLaunchKernelGGL((scan_kernel<N, GG, MODE>), grid(kThreads / GG), dim3(kThreads), 0, st, a);
    MI_CASE_G(1)
    MI_CASE_G(2)
    MI_CASE_G(4)
    MI_CASE_G(8)
    MI_CASE_G(16)
#undef MI_CASE_G
    return hipGetLastError();
}

template <int MODE>
hipError_t launch_valu_scan(const ScanArgs &a, int N, hipStream_t st) {
    switch (N) {
        case 16: return launch_valu_n<16, MODE>(a, st);
        case 32: return launch_valu_n<32, MODE>(a, st);
        case 64: return launch_valu_n<64, MODE>(a, st);
        default: return launch_valu_n<128, MODE>(a, st);
    }
}

// ------------------------------------------------------------- dispatch
template <int MODE>
hipError_t launch_generic(const ScanArgs &a, int N, hipStream_t st) {
    const int64_t lanes = (int64_t)a.B * a.H * a.P;
    hipLaunchKernelGGL((scan_generic_kernel<MODE>), dim3((unsigned)((lanes + 255) / 256)), dim3(256), 0, st, a, N);
    return hipGetLastError();
}

// mode channel or head; fast: what mfma_scan_kernel and scan_kernel take but for
// the row length
template <int MODE>
hipError_t launch_scan(const ScanArgs &a, int N, bool fast, hipStream_t st) {
    if (!fast) return launch_generic<MODE>(a, N, st);
    const int64_t row = std::max(a.x_row, a.bc_row);
    const int mode = MODE == kModeChannel ? kMScanChannel : kMScanHead;
    const bool wide = row >= kMfmaMaxRow;
    if (a.H <= 65535 && (wide || a.L <= valu_scan_steps(mode, N, a.B, a.H * a.P, a.P))) return launch_valu_scan<MODE>(a, N, st);   // (heads along y)
    if (wide) return launch_generic<MODE>(a, N, st);
    MfmaScanArgs m{};
    m.x = a.x; m.b = a.bsrc; m.c = a.csrc; m.decay = a.decay; m.y = a.y; m.chunk_states = a.chunk_states; m.h_in = a.h_in; m.h_out = a.h_out;
    m.x_row = a.x_row; m.bc_row = a.bc_row; m.B = a.B; m.L = a.L; m.D = a.H * a.P; m.P = a.P; m.cs = a.cs; m.nchunks_out = a.nchunks_out;
    return launch_mfma_scan(mode, N, m, st);
}

bool fast_shape(int N, int P, int k, int mode) {
    if (N != 16 && N != 32 && N != 64 && !(N == 128 && mode != kModeModel)) return false;
    return P % 16 == 0 && k == 15;
}

// ------------------------------------------------ float-compat reference
// Exact semantics of the reference launch_dyadic_scan
// (dyadic_mamba_kernel.cu:35-63): one lane per (b, d), int64 state.
__global__ __launch_bounds__(256) void scan_f32_kernel(const float *x, const int32_t *nums, const int32_t *shifts,
                                                       float *h, int B, int S, int D, int sb) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)B * D) return;
    const int d = (int)(idx % D);
    const int b = (int)(idx / D);
    const float scale_f = (float)((long long)1 << sb);
    long long hc = 0;
    for (int t = 0; t < S; ++t) {
        const int64_t off = ((int64_t)b * S + t) * D + d;
        const float xs = x[off] * scale_f;
        const long long xf = (long long)xs;
        hc = hc * (long long)nums[off];
        hc = hc >> shifts[off];
        hc += xf;
        h[off] = (float)hc / scale_f;
    }
}

// Elementwise integer recurrence over u, n [B][L][C] (DyadicScanFunction, and with
// CHUNKED the per-chunk outputs of ssd_chunked_scan_forward, ssd_chunked_scan.py:
// 382-422: the state at each chunk's last step and the chunk's cumulative decay
// in Q30, 2^30 decayed by the chunk's steps and rounded down after each).
//
// Bound: HBM (12 bytes a step and channel) where enough bytes are in flight,
// else the chain of steps.  With one lane per channel a load brings 4 bytes a
// lane of one step, and a wave can have 63 memory operations outstanding: about
// 20 steps, so a memory latency every 20 steps bounds small channel counts.  Here
// a wave owns 64 / R channels and its R rows of lanes load R consecutive steps at
// once (kElemAhead groups of R steps in registers).  Every row then runs all R
// steps: the rows' operands are exchanged by v_permlane16/32_swap, and row r
// keeps step r's state for one store per group.  The update is the 64-bit
// product, its shift and a clamped add when every decay of the group lies in
// [0, 2^k] (a vote), else the saturating 64-bit form.  B1 x L2048 x 24576 channels
// 963 -> 146 us (4.1 TB/s); chunked B4 x L1000 x 1536 145 -> 56 us.
constexpr int kElemAhead = 16;

// Every row's value of v for all rows: o[i] = v of row i (R rows of 64 / R lanes).
template <int R>
__device__ __forceinline__ void row_values(int v, int (&o)[R]) {
    if constexpr (R == 1) {
        o[0] = v;
    } else if constexpr (R == 2) {
        const auto ab = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
        o[0] = (int)ab[0];
        o[1] = (int)ab[1];
    } else {
        const auto ab = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);   // (a a c c), (b b d d)
        const auto ac = __builtin_amdgcn_permlane32_swap(ab[0], ab[0], false, false);
        const auto bd = __builtin_amdgcn_permlane32_swap(ab[1], ab[1], false, false);
        o[0] = (int)ac[0];
        o[1] = (int)bd[0];
        o[2] = (int)ac[1];
        o[3] = (int)bd[1];
    }
}

template <bool CHUNKED, int R, int W>
__global__ __launch_bounds__(64 * W) void elem_scan_kernel(const int32_t *u, const int32_t *n, int k, int cs, int32_t *h,
                                                           int32_t *final_h, int32_t *dte, const int32_t *h_in,
                                                           int32_t *h_out, int L, int C, int cblocks, int nc) {
    constexpr int CW = 64 / R;                    // channels of a wave
    const int lane = threadIdx.x & 63, r = lane / CW;
    const int64_t b = blockIdx.x / cblocks;
    const int c0 = ((int)(blockIdx.x % cblocks) * W + wave_id()) * CW;
    if (c0 >= C) return;
    const int c = min(c0 + lane % CW, C - 1);     // lanes past the end repeat the last channel, values and stores alike
    int32_t s = h_in ? h_in[b * C + c] : 0;
    int32_t p = 1 << 30;
    int left = cs, chunk = 0;                     // steps left in the chunk
    const uint32_t lim = 1u << k;

    const int64_t base = b * L * C;
    const uint32_t off = (uint32_t)r * (uint32_t)C + (uint32_t)c;
    const int groups = L / R;                     // whole ones
    auto row = [&](const int32_t *q, int g) { return q + base + (int64_t)g * R * C + off; };
    auto step = [&](int uv, int nv, bool fast) {
        if (fast) {
            s = __builtin_elementwise_add_sat((int32_t)(((int64_t)s * nv) >> k), uv);
            if constexpr (CHUNKED) p = (int32_t)(((int64_t)p * nv) >> k);
        } else {
            s = sat32_64((((int64_t)s * nv) >> k) + (int64_t)uv);
            if constexpr (CHUNKED) p = sat32_64(((int64_t)p * nv) >> k);
        }
    };
    // after `steps` steps, the last of them the chunk's or the sequence's: wave-uniform
    auto chunk_end = [&](int steps, bool last) {
        left -= steps;
        if (left == 0 || last) {
            const int64_t co = (b * nc + chunk) * C + c;
            if (r == 0) {
                if (final_h) final_h[co] = s;
                if (dte) dte[co] = p;
            }
            p = 1 << 30;
            left = cs;
            ++chunk;
        }
    };
    int32_t uu[kElemAhead], nn[kElemAhead];
    if (groups > 0) {
#pragma unroll
        for (int j = 0; j < kElemAhead; ++j) {
            uu[j] = *row(u, min(j, groups - 1));
            nn[j] = *row(n, min(j, groups - 1));
        }
    }
    auto group = [&](int32_t uv, int32_t nv, int g) {
        int ur[R], nr[R];
        row_values<R>(uv, ur);
        row_values<R>(nv, nr);
        int keep = 0;
        if (!__any((uint32_t)nv > lim)) {
#pragma unroll
            for (int e = 0; e < R; ++e) {
                step(ur[e], nr[e], true);
                keep = r == e ? s : keep;
            }
        } else {
#pragma unroll
            for (int e = 0; e < R; ++e) {
                step(ur[e], nr[e], false);
                keep = r == e ? s : keep;
            }
        }
        *const_cast<int32_t *>(row(h, g)) = keep;
        if constexpr (CHUNKED) chunk_end(R, g * R + R == L);   // (R divides the chunk length)
    };
    // whole rounds of kElemAhead groups (no exits inside: the register arrays
    // would be copied at each), then the last groups, already loaded
    int g0 = 0;
    for (; g0 + kElemAhead <= groups; g0 += kElemAhead) {
#pragma unroll
        for (int j = 0; j < kElemAhead; ++j) {
            const int32_t uv = uu[j], nv = nn[j];
            const int nx = min(g0 + j + kElemAhead, groups - 1);   // past the end: the last group again, unused
            uu[j] = *row(u, nx);
            nn[j] = *row(n, nx);
            group(uv, nv, g0 + j);
        }
    }
#pragma unroll
    for (int j = 0; j < kElemAhead - 1; ++j)
        if (g0 + j < groups) group(uu[j], nn[j], g0 + j);
    for (int t = R * groups; t < L; ++t) {   // fewer than R steps, every row the same
        const int64_t o = base + (int64_t)t * C + c;
        const int nv = n[o];
        step(u[o], nv, false);
        if (r == 0) h[o] = s;
        if constexpr (CHUNKED) chunk_end(1, t + 1 == L);
    }
    if (h_out && r == 0) h_out[b * C + c] = s;
}

// One lane per (sequence, channel), flat over both, the operands of A steps loaded
// before the dependent chain runs over them (from clamped addresses; steps past the
// end are skipped by a branch that is uniform): for sequences of few steps or
// few channels, where elem_scan_kernel's rows and per-sequence blocks leave lanes
// and loads idle (launch_elem_scan).
template <bool CHUNKED, int A>
__global__ __launch_bounds__(256) void elem_lane_kernel(const int32_t *u, const int32_t *n, int k, int cs, int32_t *h,
                                                        int32_t *final_h, int32_t *dte, const int32_t *h_in,
                                                        int32_t *h_out, int B, int L, int C, int nc) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)B * C) return;
    const int64_t b = idx / C;
    const int c = (int)(idx - b * C);
    const int64_t base = b * L * C + c;
    int32_t s = h_in ? h_in[idx] : 0;
    int32_t p = 1 << 30;
    int left = cs, chunk = 0;                     // steps left in the chunk
    for (int t0 = 0; t0 < L; t0 += A) {
        int32_t uu[A], nn[A];
#pragma unroll
        for (int j = 0; j < A; ++j) {
            const int64_t off = base + (int64_t)min(t0 + j, L - 1) * C;
            uu[j] = u[off];
            nn[j] = n[off];
        }
#pragma unroll
        for (int j = 0; j < A; ++j) {
            const int t = t0 + j;
            if (t < L) {
                s = sat32_64((((int64_t)s * nn[j]) >> k) + (int64_t)uu[j]);
                h[base + (int64_t)t * C] = s;
                if constexpr (CHUNKED) {
                    p = sat32_64(((int64_t)p * nn[j]) >> k);
                    if (--left == 0 || t + 1 == L) {
                        const int64_t co = (b * nc + chunk) * C + c;
                        if (final_h) final_h[co] = s;
                        if (dte) dte[co] = p;
                        p = 1 << 30;
                        left = cs;
                        ++chunk;
                    }
                }
            }
        }
    }
    if (h_out) h_out[idx] = s;
}

template <bool CHUNKED, int R, int W>
void launch_elem_rows(const int32_t *u, const int32_t *n, int k, int cs, int32_t *h, int32_t *final_h, int32_t *dte,
                      const int32_t *h_in, int32_t *h_out, int B, int L, int C, int nc, hipStream_t st) {
    constexpr int CB = 64 / R * W;   // channels of a block
    const int64_t cb = ((int64_t)C + CB - 1) / CB;
    hipLaunchKernelGGL((elem_scan_kernel<CHUNKED, R, W>), dim3((unsigned)(cb * B)), dim3(64 * W), 0, st, u, n, k, cs, h,
                       final_h, dte, h_in, h_out, L, C, (int)cb, nc);
}
template <bool CHUNKED>
void launch_elem_scan(const int32_t *u, const int32_t *n, int k, int cs, int32_t *h, int32_t *final_h, int32_t *dte,
                      const int32_t *h_in, int32_t *h_out, int B, int L, int C, int nc, hipStream_t st) {
    // Rows of steps by the channels there are: four where the waves are few (each
    // then has the most steps in flight), two and one, whose accesses are whole
    // 128- and 256-byte lines, where there are enough waves without.  us for
    // four / two / one (elementwise): 6144 channels x 1000 steps 45 / 62 / 81, 16384
    // x 2048 104 / 142 / 192, 24576 x 2048 183 / 146 / 200, 65536 x 2048 432 / 319 /
    // 293.  A chunk ends with a group: fewer rows where four do not divide it.
    const int64_t lanes = (int64_t)B * C;
    const int even = !CHUNKED || cs % 4 == 0 ? 4 : cs % 2 == 0 ? 2 : 1;
    const int rows = std::min(lanes >= 49152 ? 1 : lanes >= 20480 ? 2 : 4, even);
    // One lane per channel instead for few steps, where the rows' 16 groups ahead are
    // mostly the last one again (rows / lanes, us: 32768 x 64 channels, 1 step 21.7 /
    // 7.1, 16 steps 49.0 / 46.4; 512 x 32, 8 steps 3.1 / 2.7, 16 steps 3.4 / 3.4, 32
    // steps 4.3 / 4.7), and for sequences that fill half a wave or less where their
    // waves, several on a SIMD, take longer.  ns a step measured at 1000 steps and more
    // (rows 4 / 2 / 1, lanes): 1024 sequences of one channel 46 / 56 / 73, 125; 4096 100 /
    // 135 / 167, 130; 8192 170 / 225 / 285, 135; chunked, 6000 in odd chunks - / - / 305,
    // 150; a wave's 24 / 32 / 40 each (chunked a quarter more) and the loads of 64 steps
    // before the first, a lane's chain 140 and the stream of 0.5 for 1024 lanes.  And for
    // 2^24 sequences and more: a launch has less blocks of 256 lanes than that.
    // Four steps and fewer: one load ahead (eight repeat the last).  Blocks of 64 lanes
    // where there are few, and in the chunked form (32768 x 3, 64 steps 27 us, 33 with
    // 256 lanes; elementwise 8192 x 100, 16 steps 26 with 64, 21 with 256).
    const int64_t cw = 64 / rows, waves = B * ((C + cw - 1) / cw), simds = 4 * (int64_t)device_cus();
    const double wave_ns = (rows == 4 ? 24 : rows == 2 ? 32 : 40) * (CHUNKED ? 1.25 : 1.0);
    const double rows_ns = (double)((waves + simds - 1) / simds) * wave_ns * (L + 64.0);
    const double lanes_ns = (140 + 0.5 * (double)lanes / 1024) * L;
    if (L < (rows == 4 ? 16 : 32) || (2 * (int64_t)C <= cw && rows_ns > lanes_ns) || B >= 1 << 24) {
        const bool one = L < 4 || (!CHUNKED && L == 4);
        const unsigned threads = one || (!CHUNKED && lanes >= 65536) ? 256 : 64;
        const dim3 grid((unsigned)((lanes + threads - 1) / threads));
        if (one)
            hipLaunchKernelGGL((elem_lane_kernel<CHUNKED, 1>), grid, dim3(threads), 0, st, u, n, k, cs, h, final_h, dte,
                               h_in, h_out, B, L, C, nc);
        else
            hipLaunchKernelGGL((elem_lane_kernel<CHUNKED, 8>), grid, dim3(threads), 0, st, u, n, k, cs, h, final_h, dte,
                               h_in, h_out, B, L, C, nc);
        return;
    }
    auto go = [&](auto f) { f(u, n, k, cs, h, final_h, dte, h_in, h_out, B, L, C, nc, st); };
    if (rows == 4)
        go(lanes > 8192 ? launch_elem_rows<CHUNKED, 4, 4> : launch_elem_rows<CHUNKED, 4, 2>);
    else if (rows == 2)
        go(launch_elem_rows<CHUNKED, 2, 4>);
    else
        go(launch_elem_rows<CHUNKED, 1, 4>);
}

}  // namespace

hipError_t launch_model_scan(const int8_t *xs, const int8_t *dm, const int8_t *z, const int8_t *bsrc,
                             const int8_t *csrc, const int32_t *base, int8_t *yo, const int32_t *h_in, int32_t *h_out,
                             int64_t x_row, int64_t z_row, int64_t bc_row, int B, int L, int D, int N, int s_y,
                             hipStream_t st);
hipError_t launch_ssd_scan(const int8_t *xs, const int8_t *xp, const int8_t *z, const int32_t *tab, int8_t *yo,
                           const int32_t *h_in, int32_t *h_out, int64_t x_row, int64_t xp_row, int64_t z_row, int B,
                           int L, int H, int P, int N, int s_y, hipStream_t st);
}  // namespace mi

using namespace mi;

extern "C" mi_status mi_dyadic_scan(const int8_t *x, const int8_t *b, const int8_t *c, const int32_t *decay_num,
                                    int decay_shift, int32_t *y, const int32_t *h_in, int32_t *h_out, int batch,
                                    int len, int d, int nstate, void *stream) {
    clear_error();
    MI_REQUIRE(batch >= 0 && len >= 0 && d >= 0, MI_ERR_BAD_DIM, "mi_dyadic_scan: negative size");
    MI_REQUIRE(nstate >= 1 && nstate <= 128, MI_ERR_BAD_DIM, "mi_dyadic_scan: nstate=%d outside [1,128]", nstate);
    MI_REQUIRE(decay_shift >= 1 && decay_shift <= 16, MI_ERR_BAD_ARG, "mi_dyadic_scan: decay_shift=%d outside [1,16]",
               decay_shift);
    if ((int64_t)batch * d == 0) return MI_OK;
    MI_REQUIRE(decay_num && y, MI_ERR_NULL_POINTER, "mi_dyadic_scan: decay_num and y are required");
    if (len > 0) MI_REQUIRE(x && b && c, MI_ERR_NULL_POINTER, "mi_dyadic_scan: x, b and c are required");
    ScanArgs a{};
    a.x = x; a.bsrc = b; a.csrc = c; a.decay = decay_num; a.y = y; a.h_in = h_in; a.h_out = h_out;
    a.x_row = d; a.bc_row = nstate; a.B = batch; a.L = len; a.H = 1; a.P = d; a.k = decay_shift;
    const bool fast = len > 0 && fast_shape(nstate, d, decay_shift, kModeChannel) && aligned(x, 16) && aligned(b, 16) &&
                      aligned(c, 16) && aligned(y, 16);
    if (len == 0 && !h_out) return MI_OK;
    hipError_t e = launch_scan<kModeChannel>(a, nstate, fast, as_stream(stream));
    if (e != hipSuccess) return fail(MI_ERR_HIP, "mi_dyadic_scan: launch failed: %s", hipGetErrorString(e));
    return MI_OK;
}

extern "C" mi_status mi_ssd_chunked_scan(const int8_t *x, const int8_t *b, const int8_t *c, const int32_t *decay_num,
                                         int decay_shift, int32_t *y, int32_t *chunk_states, const int32_t *h_in,
                                         int32_t *h_out, int batch, int len, int heads, int head_dim, int nstate,
                                         int chunk, void *stream) {
    clear_error();
    MI_REQUIRE(batch >= 0 && len >= 0 && heads >= 0 && head_dim >= 0, MI_ERR_BAD_DIM,
               "mi_ssd_chunked_scan: negative size");
    MI_REQUIRE(nstate >= 1 && nstate <= 128, MI_ERR_BAD_DIM, "mi_ssd_chunked_scan: nstate=%d outside [1,128]", nstate);
    MI_REQUIRE(chunk >= 1, MI_ERR_BAD_ARG, "mi_ssd_chunked_scan: chunk=%d must be >= 1", chunk);
    MI_REQUIRE(decay_shift >= 1 && decay_shift <= 16, MI_ERR_BAD_ARG,
               "mi_ssd_chunked_scan: decay_shift=%d outside [1,16]", decay_shift);
    if ((int64_t)batch * heads * head_dim == 0 || (len == 0 && !h_out)) return MI_OK;
    MI_REQUIRE(decay_num && (len == 0 || (x && b && c && y)), MI_ERR_NULL_POINTER,
               "mi_ssd_chunked_scan: x, b, c, decay_num, y required");
    ScanArgs a{};
    a.x = x; a.bsrc = b; a.csrc = c; a.decay = decay_num; a.y = y; a.chunk_states = chunk_states;
    a.h_in = h_in; a.h_out = h_out;
    a.x_row = (int64_t)heads * head_dim; a.bc_row = (int64_t)heads * nstate;
    a.B = batch; a.L = len; a.H = heads; a.P = head_dim; a.k = decay_shift;
    a.cs = chunk; a.nchunks_out = (len + chunk - 1) / chunk;
    const bool fast = len > 0 && fast_shape(nstate, head_dim, decay_shift, kModeHead) && (chunk % kTC == 0) && aligned(x, 16) &&
                      aligned(b, 16) && aligned(c, 16) && aligned(y, 16);
    hipError_t e = launch_scan<kModeHead>(a, nstate, fast, as_stream(stream));
    if (e != hipSuccess) return fail(MI_ERR_HIP, "mi_ssd_chunked_scan: launch failed: %s", hipGetErrorString(e));
    return MI_OK;
}

extern "C" mi_status mi_block_scan(const int8_t *xs, const int8_t *dm, const int8_t *xp, int xp_stride, int b_off,
                                   const int8_t *z, int z_stride, int z_off, const int32_t *base, int decay_shift,
                                   int s_y, int8_t *yo, const int32_t *h_in, int32_t *h_out, int batch, int len,
                                   int d_inner, int nstate, void *stream) {
    clear_error();
    MI_REQUIRE(batch >= 0 && len >= 0 && d_inner >= 0, MI_ERR_BAD_DIM, "mi_block_scan: negative size");
    MI_REQUIRE(nstate >= 1 && nstate <= 64, MI_ERR_BAD_DIM, "mi_block_scan: nstate=%d outside [1,64]", nstate);
    MI_REQUIRE(decay_shift == 15, MI_ERR_BAD_ARG, "mi_block_scan: decay_shift=%d, the model path uses 15", decay_shift);
    MI_REQUIRE(s_y >= 0 && s_y <= 30, MI_ERR_BAD_ARG, "mi_block_scan: s_y=%d outside [0,30]", s_y);
    MI_REQUIRE(b_off >= 0 && b_off + 2 * nstate <= xp_stride, MI_ERR_BAD_DIM,
               "mi_block_scan: B/C columns [%d,%d) exceed xp_stride=%d", b_off, b_off + 2 * nstate, xp_stride);
    MI_REQUIRE(z_off >= 0 && z_off + d_inner <= z_stride, MI_ERR_BAD_DIM,
               "mi_block_scan: z columns exceed z_stride=%d", z_stride);
    if ((int64_t)batch * d_inner == 0 || (len == 0 && !h_out)) return MI_OK;
    MI_REQUIRE(base && (len == 0 || (xs && dm && xp && z && yo)), MI_ERR_NULL_POINTER,
               "mi_block_scan: a required pointer is NULL");
    ScanArgs a{};
    a.x = xs; a.dm = dm; a.z = z + z_off; a.bsrc = xp + b_off; a.csrc = xp + b_off + nstate; a.decay = base;
    a.yo = yo; a.h_in = h_in; a.h_out = h_out;
    a.x_row = d_inner; a.bc_row = xp_stride; a.z_row = z_stride;
    a.B = batch; a.L = len; a.H = 1; a.P = d_inner; a.k = decay_shift; a.s_y = s_y;
    const bool fast = len > 0 && fast_shape(nstate, d_inner, decay_shift, kModeModel) && aligned(xs, 16) && aligned(dm, 16) &&
                      aligned(a.z, 16) && aligned(a.bsrc, 16) && aligned(a.csrc, 16) && aligned(yo, 16) &&
                      xp_stride % 16 == 0 && z_stride % 16 == 0;
    hipError_t e;
    if (fast)
        e = launch_model_scan(xs, dm, a.z, a.bsrc, a.csrc, base, yo, h_in, h_out, d_inner, z_stride, xp_stride, batch,
                              len, d_inner, nstate, s_y, as_stream(stream));
    else
        e = launch_generic<kModeModel>(a, nstate, as_stream(stream));
    if (e != hipSuccess) return fail(MI_ERR_HIP, "mi_block_scan: launch failed: %s", hipGetErrorString(e));
    return MI_OK;
}

extern "C" mi_status mi_ssd_block_scan(const int8_t *xs, const int8_t *xp, int xp_stride, const int8_t *z,
                                       int z_stride, int z_off, const int32_t *decay_tab, int n_heads, int s_y,
                                       int8_t *yo, const int32_t *h_in, int32_t *h_out, int batch, int len,
                                       int d_inner, int nstate, void *stream) {
    const char *fn = "mi_ssd_block_scan";
    clear_error();
    MI_REQUIRE(batch >= 0 && len >= 0 && d_inner >= 0 && n_heads >= 1, MI_ERR_BAD_DIM, "%s: bad size", fn);
    MI_REQUIRE(nstate == 16 || nstate == 32 || nstate == 64, MI_ERR_BAD_DIM, "%s: nstate=%d (16, 32 or 64)", fn,
               nstate);
    MI_REQUIRE(d_inner % n_heads == 0 && (d_inner / n_heads) % 16 == 0, MI_ERR_BAD_DIM,
               "%s: d_inner=%d must split into %d heads of a multiple of 16 channels", fn, d_inner, n_heads);
    MI_REQUIRE(s_y >= 0 && s_y <= 30, MI_ERR_BAD_ARG, "%s: s_y=%d outside [0,30]", fn, s_y);
    MI_REQUIRE(xp_stride >= 2 * n_heads * nstate + n_heads && xp_stride % 16 == 0, MI_ERR_BAD_DIM,
               "%s: xp_stride=%d must hold B, C and dt of every head and be a multiple of 16", fn, xp_stride);
    MI_REQUIRE(z_off >= 0 && z_off + d_inner <= z_stride && z_stride % 16 == 0 && z_off % 16 == 0, MI_ERR_BAD_DIM,
               "%s: z columns [%d,%d) and stride %d (multiples of 16)", fn, z_off, z_off + d_inner, z_stride);
    if ((int64_t)batch * d_inner == 0 || (len == 0 && !h_out)) return MI_OK;
    MI_REQUIRE(decay_tab && (len == 0 || (xs && xp && z && yo)), MI_ERR_NULL_POINTER, "%s: a required pointer is NULL",
               fn);
    MI_REQUIRE(len == 0 || (aligned(xs, 16) && aligned(xp, 16) && aligned(z, 16) && aligned(yo, 16)),
               MI_ERR_BAD_ALIGNMENT, "%s: xs, xp, z and yo must be 16-byte aligned", fn);
    MI_REQUIRE(aligned(h_in, 4) && aligned(h_out, 4) && aligned(decay_tab, 4), MI_ERR_BAD_ALIGNMENT,
               "%s: h_in, h_out and decay_tab must be 4-byte aligned", fn);
    const hipError_t e = launch_ssd_scan(xs, xp, z + z_off, decay_tab, yo, h_in, h_out, d_inner, xp_stride, z_stride,
                                         batch, len, n_heads, d_inner / n_heads, nstate, s_y, as_stream(stream));
    if (e != hipSuccess) return fail(MI_ERR_HIP, "%s: launch failed: %s", fn, hipGetErrorString(e));
    return MI_OK;
}

extern "C" mi_status mi_dyadic_scan_f32(const float *x, const int32_t *nums, const int32_t *shifts, float *h,
                                        int batch, int seq, int dim, int scale_bits, void *stream) {
    clear_error();
    MI_REQUIRE(batch >= 0 && seq >= 0 && dim >= 0, MI_ERR_BAD_DIM, "mi_dyadic_scan_f32: negative size");
    MI_REQUIRE(scale_bits >= 0 && scale_bits <= 62, MI_ERR_BAD_ARG, "mi_dyadic_scan_f32: scale_bits=%d outside [0,62]",
               scale_bits);
    if ((int64_t)batch * seq * dim == 0) return MI_OK;
    MI_REQUIRE(x && nums && shifts && h, MI_ERR_NULL_POINTER, "mi_dyadic_scan_f32: a required pointer is NULL");
    const int64_t lanes = (int64_t)batch * dim;
    hipLaunchKernelGGL(scan_f32_kernel, dim3((unsigned)((lanes + 255) / 256)), dim3(256), 0, as_stream(stream), x,
                       nums, shifts, h, batch, seq, dim, scale_bits);
    return check_launch("mi_dyadic_scan_f32");
}

extern "C" mi_status mi_dyadic_scan_elementwise(const int32_t *u, const int32_t *nums, int decay_shift, int32_t *h,
                                                const int32_t *h_in, int32_t *h_out, int batch, int len, int channels,
                                                void *stream) {
    clear_error();
    MI_REQUIRE(batch >= 0 && len >= 0 && channels >= 0, MI_ERR_BAD_DIM, "mi_dyadic_scan_elementwise: negative size");
    MI_REQUIRE(decay_shift >= 1 && decay_shift <= 30, MI_ERR_BAD_ARG,
               "mi_dyadic_scan_elementwise: decay_shift=%d outside [1,30]", decay_shift);
    // len == 0 with h_out: the kernel runs no step and writes h_out = h_in (zeros when NULL)
    if ((int64_t)batch * channels == 0 || (len == 0 && !h_out)) return MI_OK;
    MI_REQUIRE(len == 0 || (u && nums && h), MI_ERR_NULL_POINTER,
               "mi_dyadic_scan_elementwise: u, nums and h are required");
    launch_elem_scan<false>(u, nums, decay_shift, 0, h, nullptr, nullptr, h_in, h_out, batch, len, channels, 0,
                            as_stream(stream));
    return check_launch("mi_dyadic_scan_elementwise");
}

extern "C" mi_status mi_dyadic_chunked_scan(const int32_t *u, const int32_t *nums, int decay_shift, int chunk,
                                            int32_t *h, int32_t *final_h, int32_t *decay_to_end, const int32_t *h_in,
                                            int32_t *h_out, int batch, int len, int channels, void *stream) {
    clear_error();
    MI_REQUIRE(batch >= 0 && len >= 0 && channels >= 0, MI_ERR_BAD_DIM, "mi_dyadic_chunked_scan: negative size");
    MI_REQUIRE(decay_shift >= 1 && decay_shift <= 30, MI_ERR_BAD_ARG,
               "mi_dyadic_chunked_scan: decay_shift=%d outside [1,30]", decay_shift);
    MI_REQUIRE(chunk >= 1, MI_ERR_BAD_ARG, "mi_dyadic_chunked_scan: chunk=%d must be >= 1", chunk);
    // len == 0 with h_out: the kernel runs no step and writes h_out = h_in (zeros when NULL)
    if ((int64_t)batch * channels == 0 || (len == 0 && !h_out)) return MI_OK;
    MI_REQUIRE(len == 0 || (u && nums && h), MI_ERR_NULL_POINTER, "mi_dyadic_chunked_scan: u, nums and h are required");
    const int nc = (int)((len + (int64_t)chunk - 1) / chunk);
    launch_elem_scan<true>(u, nums, decay_shift, chunk, h, final_h, decay_to_end, h_in, h_out, batch, len, channels, nc,
                           as_stream(stream));
    return check_launch("mi_dyadic_chunked_scan");
}
