// Dyadic scans with the output contraction y = C . h on the matrix cores
// (spec mi-spec-2, rules 1, 4.7-4.11 and 7.4-7.8), for decay shift 15.
//
// State update: sat32(floor(h * n / 2^15) + b * x) is three instructions, the
// 64-bit product (v_mad_i64_i32), its shift (v_alignbit_b32) and a clamped
// v_mad_i32_i16 on int16 pairs of B and x, plus the decay's sum in the model.
// Measured on gfx950, cycles per wave instruction: v_mad_i64_i32, v_alignbit,
// v_mad_i32_i16, the 24-bit and SDWA forms all 4.2-4.7, dependent or not; so the
// 64-bit product beats two half products and their sum (13.1 against 17.4
// cycles an update).
//
// Output: computing y on the VALU costs as much again, three instructions per
// state and a reduction over the lanes that share a channel.  Here one
// v_mfma_i32_16x16x64_i8 per four steps and four states does both.  A state is
// four bytes, and the MFMA's B operand takes 16 bytes per lane: the states of
// four steps go in as they are, k = (lane group g, step t', byte p).
// Lane l = (g = l / 16, channel l % 16) holds state 4 * quad + g of its channel,
// so the MFMA's sum over k runs over the quad's four states, and the A operand
// picks one (step, byte) per output row: row 4 t' + p is C[t'][state] at byte p
// of step t' and zero elsewhere.  Then D register p of lane group t' is the exact
// sum over the quad of C * (byte p of h) for the lane's own channel, with no
// cross-lane reduction.  Bytes 0-2 of h are unsigned and the MFMA's are signed:
// h ^ 0x00808080 turns them into b - 128, and the epilogue adds 128 * sum(C)
// back per byte.  y = hi * 2^16 + lo with hi = D2 + 256 D3, lo = D0 + 256 D1
// (|D| <= N * 2^14, so all of it stays inside int32 up to N = 128).
//
// A block has two kinds of waves.  Scan waves only run steps: a wave holds 4 S
// states (S a lane) of M x 16 channels and leaves its (hi, lo) per (step,
// channel) in LDS.  Four helper waves stage the next chunk of TC steps (global
// loads issued two chunks ahead) and finish the previous one (sum the scan
// waves' partials, saturate, gate, requant, store); they run at a raised wave
// priority, since a chunk's barrier waits for them.
//
// Bound: VALU issue where every CU has a block (B8 x L2048 x 1536 channels, N16, one
// block of 48 channels a CU: 9.6 instructions per update of 64 states, 13.6 with y on
// the VALU, at 67% of the issue cycles); the CUs themselves where the blocks are
// fewer (the head layout below: 192 blocks of 32 channels on 256 CUs, at 74% of the
// issue cycles of those that work); with few channels one block's chain of steps
// (33 ns a step).  us per launch alone, y on the VALU against here:
//   model block   B8 x L2048 x 1536, N16      210 -> 149 (in the model, behind other
//                                             kernels, 146 to 164)
//                 B2 x L1000 x 1536           105 -> 37      B3 x L701 x 2048   75 -> 42
//                 B64 x L512 x 4096           806 -> 778
//   SSD block     B2 x L1023, 24 x 64, N64    160 -> 71      B8 x L2048        590 -> 392
//   head layout   B4 x L8192, 24 x 64, N128  2119 -> 1579
//   channels      B1 x L256 x 512, N16         22 -> 8       B8 x L2048 x 1536 285 -> 111
#include <stddef.h>

#include <initializer_list>
#include <type_traits>
#include <utility>

#include "mfma_scan.hpp"
#include "mi_mfma.hpp"

namespace mi {
namespace {

constexpr int kHelpers = 256;   // threads of the four helper waves
// word 3 of a raw buffer resource (32-bit data format, no swizzle)
constexpr int kBufferRsrcWord3 = 0x00020000;
typedef unsigned v4u __attribute__((ext_vector_type(4)));

__device__ __forceinline__ int sbyte(uint32_t w, int i) { return (int)(int8_t)(w >> (8 * i)); }
__device__ __forceinline__ int at(const int4 &v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

// Sum over the R adjacent lanes of an aligned group (R = 2, 4 or 8).
template <int R>
__device__ __forceinline__ int row_sum(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, true);                       // quad_perm 1,0,3,2
    if constexpr (R >= 4) v += __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, true);   // quad_perm 2,3,0,1
    if constexpr (R >= 8) v += __builtin_amdgcn_update_dpp(0, v, 0x141, 0xF, 0xF, true);  // row_half_mirror
    return v;
}

template <int MODE, int N, int S, int M, int MW, int TC>
struct MfmaScan {
    static constexpr bool MODEL = MODE == kMScanModel, CHAN = MODE == kMScanChannel, HEAD = MODE == kMScanHead,
                          SSD = MODE == kMScanSsd;
    static constexpr bool GATED = MODEL || SSD;          // int8 output through the gate; else int32 y
    static constexpr int NQ = N / (4 * S);               // scan waves of a channel
    static constexpr int NS = NQ * MW;                   // scan waves: NQ state groups x MW channel groups
    static constexpr int NT = 64 * NS + kHelpers;
    static constexpr int CH = 16 * M * MW;               // channels of a block
    static constexpr int TP = TC + 8;                    // row pitch of the staged x and B (int16)
    static constexpr int XP = TC * CH / 8;               // x pieces of two steps x four channels
    static constexpr int XW = (XP + 63) / 64;            // helper waves that stage them
    static constexpr int FR = TC * CH / 256;             // epilogue rounds of 64 (step, four channels) items
    static constexpr int FPER = (FR + 3) / 4;            // rounds per helper wave, at most
    static constexpr int PB = TC * N < 512 ? 4 : TC * N / 128;   // bytes of a B or C piece (128 threads each)
    static constexpr int PW = PB / 4;
    static constexpr int RP = N / PB;                    // pieces per row of B or C
    // row pitch of the staged C: the four steps that a wave reads at once fall in
    // different banks
    static constexpr int CP = N > 16 ? N + 16 : N;
    static_assert(N % (4 * S) == 0 && TC % 8 == 0 && (RP == 2 || RP == 4 || RP == 8), "split");
    static_assert(XW <= 4 && TC * CH % 256 == 0, "helper rounds");
    static_assert((PB == 4 || PB == 8 || PB == 16) && TC * RP <= 128, "B and C pieces");

    // The row of state n: the pieces of a step (states PB apart) are written to
    // neighbouring rows, so to different banks (the pitch is a multiple of 16 bytes)
    __device__ static constexpr int brow(int n) { return n % PB * (N / PB) + n / PB; }

    struct Smem {
        int16_t x[2][CH][TP];          // input of a step (the model: xs * dt)
        int16_t b[2][N][TP];           // rows in the order of brow
        uint32_t c[2][TC][CP];         // C in all four bytes of a word
        int8_t dm[MODEL ? 2 : 1][MODEL ? CH : 1][TP];
        alignas(16) int32_t n[SSD ? 2 : 1][SSD ? TC : 4];     // decay of a step
        alignas(16) int32_t y[2][NQ][2][TC][CH];   // hi and lo partials of a channel's scan waves
        int32_t csum[3][TC];           // 128 * sum of C over the states
        uint32_t dt[MODEL ? 256 : 1];  // by the raw byte of dm: dt << 16 | (clamped dm & 255)
        int32_t tab[SSD ? 255 : 1];
        int32_t gate[GATED ? 256 : 1]; // by the raw byte of z
    };
    // read as 16-byte vectors
    static_assert(offsetof(Smem, x) % 16 == 0 && offsetof(Smem, b) % 16 == 0 && offsetof(Smem, c) % 16 == 0 &&
                  offsetof(Smem, n) % 16 == 0 && offsetof(Smem, y) % 16 == 0, "alignment");
    static_assert(TP * 2 % 16 == 0 && CP * 4 % 16 == 0 && CH * 4 % 16 == 0, "row alignment");
};

template <int MODE, int N, int S, int M, int MW, int TC>
__global__ __launch_bounds__(64 * (N / (4 * S)) * MW + kHelpers) void mfma_scan_kernel(MfmaScanArgs a) {
    using K = MfmaScan<MODE, N, S, M, MW, TC>;
    constexpr bool MODEL = K::MODEL, CHAN = K::CHAN, HEAD = K::HEAD, SSD = K::SSD, GATED = K::GATED;
    constexpr int CH = K::CH;
    __shared__ __align__(16) typename K::Smem sm;
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
    const int p0 = blockIdx.x * CH;                        // first channel, flat over the heads
    const int b = blockIdx.y;
    const int head = HEAD || SSD ? p0 / a.P : 0;           // (CH divides P: a block lies in one head)
    const int64_t row0 = (int64_t)b * a.L;
    const int nchunks = (a.L + TC - 1) / TC;

    if constexpr (MODEL)
        for (int i = tid; i < 256; i += K::NT) {
            const int d = clamp32((int)(int8_t)i, -20, 20);
            sm.dt[i] = ((uint32_t)dt_q16(d) << 16) | (uint32_t)(d & 255);
        }
    if constexpr (SSD)
        for (int i = tid; i < 255; i += K::NT) sm.tab[i] = a.decay[(int64_t)head * 255 + i];
    if constexpr (GATED)
        for (int i = tid; i < 256; i += K::NT) sm.gate[i] = gate_q15((int)(int8_t)i);
    __syncthreads();

    if (wave < K::NS) {
        // ---------------------------------------------------- scan waves
        const int c16 = lane & 15, g = lane >> 4;
        const int wq = wave % K::NQ, cb = wave / K::NQ * 16 * M;   // state group, first channel of the block
        const int n0 = wq * 4 * S + g;                   // state s of this lane: n0 + 4 s
        int32_t h[M][S], nd[M][S];                        // states, decays
        bool safe = true;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int p = min(p0 + cb + 16 * m + c16, a.D - 1);   // channels past the end repeat the last one, unstored
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const int n = n0 + 4 * s;
                h[m][s] = a.h_in ? a.h_in[((int64_t)b * a.D + p) * N + n] : 0;
                if constexpr (MODEL || CHAN) {
                    nd[m][s] = a.decay[(int64_t)p * N + n];
                    safe = safe && nd[m][s] >= 20 && nd[m][s] <= 32000 - 20;
                }
            }
        }
        int32_t nh = 0;
        if constexpr (HEAD) nh = a.decay[head];
        // a wave-uniform choice: base + dm cannot leave [0, 32000], no decay clamp
        const bool wave_safe = __all(safe);
        // A operand of this lane's row 4 tq + p: C at byte p of dword tq
        const int tq = c16 >> 2;
        v4u am;
#pragma unroll
        for (int j = 0; j < 4; ++j) am[j] = j == tq ? 0xffu << (8 * (c16 & 3)) : 0u;

        struct Group {           // the operands of eight steps
            v4i x[M], b[S];      // int16 pairs
            int4 n[2];
            uint2 dm[M];
            uint32_t c[S][2];
        };
        auto run = [&](int chunk, auto clamp_tag) {
            constexpr bool CLAMP = decltype(clamp_tag)::value;
            const int bf = chunk & 1;
            const int tn = min(TC, a.L - chunk * TC);
            auto load = [&](int t8, Group &r) {
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    r.x[m] = *reinterpret_cast<const v4i *>(&sm.x[bf][cb + 16 * m + c16][t8]);
                    if constexpr (MODEL) r.dm[m] = *reinterpret_cast<const uint2 *>(&sm.dm[bf][cb + 16 * m + c16][t8]);
                }
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    r.b[s] = *reinterpret_cast<const v4i *>(&sm.b[bf][K::brow(n0 + 4 * s)][t8]);
                    r.c[s][0] = sm.c[bf][t8 + tq][n0 + 4 * s];
                    r.c[s][1] = sm.c[bf][t8 + 4 + tq][n0 + 4 * s];
                }
                if constexpr (SSD) {
                    r.n[0] = *reinterpret_cast<const int4 *>(&sm.n[bf][t8]);
                    r.n[1] = *reinterpret_cast<const int4 *>(&sm.n[bf][t8 + 4]);
                }
            };
            v4i acc[M];
            auto put = [&](int t4) {
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    sm.y[bf][wq][0][t4 + g][cb + 16 * m + c16] = acc[m][2] + (acc[m][3] << 8);
                    sm.y[bf][wq][1][t4 + g][cb + 16 * m + c16] = acc[m][0] + (acc[m][1] << 8);
                }
            };
            // the four steps of half H of a group (of a ragged chunk: nv of them)
            auto steps = [&](const Group &r, auto half_tag, int t4, int nv, bool flush) {
                constexpr int H = decltype(half_tag)::value;
                v4i hx[M][S];
                auto step = [&](auto tt_tag) {
                    constexpr int TT = decltype(tt_tag)::value;
                    if (TT < nv) {   // wave-uniform
#pragma unroll
                        for (int m = 0; m < M; ++m)
#pragma unroll
                            for (int s = 0; s < S; ++s) {
                                int n = SSD ? at(r.n[H], TT) : HEAD ? nh : nd[m][s];
                                if constexpr (MODEL) {
                                    n += sbyte(H ? r.dm[m].y : r.dm[m].x, TT);
                                    if constexpr (CLAMP) n = clamp32(n, 0, 32000);
                                }
                                // floor(h * n / 2^15): the 64-bit product and its shift are two
                                // instructions (v_mad_i64_i32 issues at the rate of a 24-bit multiply)
                                h[m][s] = mad16_sat<TT & 1>(r.b[s][2 * H + TT / 2], r.x[m][2 * H + TT / 2],
                                                            (int32_t)(((int64_t)h[m][s] * n) >> 15));
                            }
                    }
#pragma unroll
                    for (int m = 0; m < M; ++m)
#pragma unroll
                        for (int s = 0; s < S; ++s) hx[m][s][TT] = h[m][s] ^ 0x00808080;
                };
                step(std::integral_constant<int, 0>{});
                step(std::integral_constant<int, 1>{});
                step(std::integral_constant<int, 2>{});
                step(std::integral_constant<int, 3>{});
                if (flush) put(t4 - 4);   // the previous half's sums: its MFMAs have long finished
#pragma unroll
                for (int m = 0; m < M; ++m) acc[m] = v4i{0, 0, 0, 0};
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    const v4u cv = v4u{r.c[s][H], r.c[s][H], r.c[s][H], r.c[s][H]} & am;
#pragma unroll
                    for (int m = 0; m < M; ++m) acc[m] = mfma_i8(__builtin_bit_cast(v4i, cv), hx[m][s], acc[m]);
                }
            };
            using H0 = std::integral_constant<int, 0>;
            using H1 = std::integral_constant<int, 1>;
            // the next group's operands are read while this group runs (the
            // scheduling barriers keep the reads ahead of it: moved down to their
            // uses, each exposed an LDS latency)
            Group r0, r1;
            load(0, r0);
            if (tn == TC) {
#pragma unroll
                for (int t8 = 0; t8 < TC; t8 += 16) {
                    if (t8 + 8 < TC) load(t8 + 8, r1);
                    __builtin_amdgcn_sched_barrier(0);
                    steps(r0, H0{}, t8, 4, t8 > 0);
                    steps(r0, H1{}, t8 + 4, 4, true);
                    if (t8 + 8 < TC) {
                        if (t8 + 16 < TC) load(t8 + 16, r0);
                        __builtin_amdgcn_sched_barrier(0);
                        steps(r1, H0{}, t8 + 8, 4, true);
                        steps(r1, H1{}, t8 + 12, 4, true);
                    }
                }
                put(TC - 4);
            } else {
#pragma unroll 1
                for (int t8 = 0; t8 < tn; t8 += 8) {
                    if (t8 > 0) load(t8, r0);
                    steps(r0, H0{}, t8, tn - t8, t8 > 0);
                    if (t8 + 4 < tn) steps(r0, H1{}, t8 + 4, tn - t8 - 4, true);
                }
                put((tn - 1) & ~3);
            }
            if constexpr (HEAD) {
                // chunk_states at every multiple of cs (a multiple of TC) and at the end
                const int tdone = chunk * TC + tn;
                if (a.chunk_states && (tdone % a.cs == 0 || tdone == a.L)) {
                    const int64_t cc = (int64_t)b * a.nchunks_out + (tdone - 1) / a.cs;
#pragma unroll
                    for (int m = 0; m < M; ++m) {
                        int32_t *dst = a.chunk_states + (cc * a.D + p0 + cb + 16 * m + c16) * N + n0;
#pragma unroll
                        for (int s = 0; s < S; ++s) dst[4 * s] = h[m][s];
                    }
                }
            }
        };
        __syncthreads();   // chunk 0 is staged
        for (int i = 0; i <= nchunks; ++i) {
            if (i < nchunks) {
                if (!MODEL || wave_safe) run(i, std::false_type{});
                else run(i, std::true_type{});
            }
            __syncthreads();
        }
        if (a.h_out) {
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const int p = p0 + cb + 16 * m + c16;
                if (p < a.D)
#pragma unroll
                    for (int s = 0; s < S; ++s) a.h_out[((int64_t)b * a.D + p) * N + n0 + 4 * s] = h[m][s];
            }
        }
        return;
    }

    // ------------------------------------------------------- helper waves
    __builtin_amdgcn_s_setprio(3);
    const int ht = tid - 64 * K::NS, hw = wave - K::NS;
    const bool isc = hw >= 2;                             // waves 0-1 stage B, 2-3 C
    const int bt = (ht & 127) / K::RP % TC, bq = (ht & 127) % K::RP;
    // x piece of this thread (waves 0 .. XW - 1): steps xt, xt + 1, channels xc .. xc + 3
    const int xi = min(ht, K::XP - 1), xt = 2 * (xi / (CH / 4)), xc = 4 * (xi % (CH / 4));
    const bool xw = hw < K::XW;
    // epilogue rounds (hw - XW) mod 4, + 4, ...: the waves without x pieces take the odd ones
    const int fr0 = (hw + 4 - K::XW % 4) & 3;
    auto item = [&](int j, int &t, int &c) {
        const int i = min(fr0 + 4 * j, K::FR - 1) * 64 + lane;
        t = i / (CH / 4);
        c = 4 * (i % (CH / 4));
    };
    // Global rows of a chunk through buffer resources built per chunk (scalar
    // work): a load is one instruction, and rows past the sequence's end lie
    // outside the resource (loads give zeros, stores are dropped).  What such
    // rows and channels past D hold only reaches steps and outputs that are
    // never used.
    const int x_row = (int)a.x_row, z_row = (int)a.z_row, bc_row = (int)a.bc_row;
    auto rows_of = [&](int chunk) { return min(TC, a.L - chunk * TC); };
    auto rsrc = [&](const int8_t *p, int64_t row, int chunk, int width) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t *>(p + (row0 + chunk * TC) * row), 0,
                                                 (rows_of(chunk) - 1) * (int)row + width, kBufferRsrcWord3);
    };
    const int8_t *bcp = (isc ? a.c : a.b) + (HEAD || SSD ? (int64_t)head * N : 0);
    const int xoff = xt * x_row + p0 + xc, boff = bt * bc_row + bq * K::PB;
    int zoff[K::FPER], ooff[K::FPER];
#pragma unroll
    for (int j = 0; j < K::FPER; ++j) {
        int t, c;
        item(j, t, c);
        zoff[j] = t * z_row + p0 + c;
        // a store of a channel past D goes outside the output resource as well
        const bool own = p0 + c < a.D && (K::FR % 4 == 0 || fr0 + 4 * j < K::FR);
        ooff[j] = own ? (t * x_row + p0 + c) * (GATED ? 1 : 4) : -1;
    }
    uint32_t rx[2][2], rd[2][2], rz[2][K::FPER];
    v4u rb[2];
    int rn[2] = {0, 0};
    auto load = [&](int chunk, auto set_tag) {
        constexpr int ST = decltype(set_tag)::value;
        const int ck = min(chunk, nchunks - 1);
        const auto xr = rsrc(a.x, a.x_row, ck, a.D), br = rsrc(bcp, a.bc_row, ck, N);
#pragma unroll
        for (int k = 0; k < 2; ++k) rx[ST][k] = __builtin_amdgcn_raw_buffer_load_b32(xr, xoff + k * x_row, 0, 0);
        if constexpr (MODEL) {
            const auto dr = rsrc(a.dm, a.x_row, ck, a.D);
#pragma unroll
            for (int k = 0; k < 2; ++k) rd[ST][k] = __builtin_amdgcn_raw_buffer_load_b32(dr, xoff + k * x_row, 0, 0);
        }
        if constexpr (K::PW == 1) {
            rb[ST][0] = __builtin_amdgcn_raw_buffer_load_b32(br, boff, 0, 0);
        } else if constexpr (K::PW == 2) {
            const auto v = __builtin_amdgcn_raw_buffer_load_b64(br, boff, 0, 0);
            rb[ST][0] = v[0];
            rb[ST][1] = v[1];
        } else {
            rb[ST] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(br, boff, 0, 0));
        }
        if constexpr (SSD)
            rn[ST] = (int8_t)__builtin_amdgcn_raw_buffer_load_b8(rsrc(a.dtc + head, a.bc_row, ck, 1), min(ht, TC - 1) * bc_row, 0, 0);
    };
    auto load_z = [&](int chunk, auto set_tag) {
        constexpr int ST = decltype(set_tag)::value;
        if constexpr (GATED) {
            const auto zr = rsrc(a.z, a.z_row, min(chunk, nchunks - 1), a.D);
#pragma unroll
            for (int j = 0; j < K::FPER; ++j) rz[ST][j] = __builtin_amdgcn_raw_buffer_load_b32(zr, zoff[j], 0, 0);
        }
    };
    auto stage = [&](int chunk, auto set_tag) {
        constexpr int ST = decltype(set_tag)::value;
        const int bf = chunk & 1;
        {
            int v[K::PB], sum = 0;
#pragma unroll
            for (int e = 0; e < K::PB; ++e) v[e] = sbyte(rb[ST][e >> 2], e & 3);
            if constexpr (SSD) {
                // the row scaled to a unit vector in Q7 (spec rule 7.4)
                int ss = 0;
#pragma unroll
                for (int e = 0; e < K::PB; ++e) ss += v[e] * v[e];
                const int32_t inv = unit_inv(row_sum<K::RP>(ss));
#pragma unroll
                for (int e = 0; e < K::PB; ++e) v[e] = clamp32(rshr32(v[e] * inv, 15), -127, 127);
            }
            if (!isc) {
#pragma unroll
                for (int e = 0; e < K::PB; ++e) sm.b[bf][K::brow(bq * K::PB + e)][bt] = (int16_t)v[e];
            } else {
#pragma unroll
                for (int q = 0; q < K::PW; ++q) {
                    v4u w;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        w[e] = __builtin_amdgcn_perm(0, (uint32_t)v[4 * q + e], 0);   // byte 0 in all four
                        sum += v[4 * q + e];
                    }
                    *reinterpret_cast<v4u *>(&sm.c[bf][bt][bq * K::PB + 4 * q]) = w;
                }
                sum = row_sum<K::RP>(sum);
                if (bq == 0) sm.csum[chunk % 3][bt] = 128 * sum;
            }
        }
        if constexpr (SSD)
            if (ht < TC) sm.n[bf][ht] = sm.tab[clamp32(rn[ST], -127, 127) + 127];
        if (xw) {   // (threads past the last piece repeat it)
            uint32_t d[4][2];
            if constexpr (MODEL) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int k = 0; k < 2; ++k) d[e][k] = sm.dt[(rd[ST][k] >> (8 * e)) & 255];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                int v[2];
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    v[k] = sbyte(rx[ST][k], e);
                    // |x| <= 128, dt <= 6554: a 24-bit product
                    if constexpr (MODEL) v[k] = (__mul24(v[k], (int)(d[e][k] >> 16)) + 512) >> 10;
                }
                *reinterpret_cast<uint32_t *>(&sm.x[bf][xc + e][xt]) =
                    __builtin_amdgcn_perm((uint32_t)v[1], (uint32_t)v[0], 0x05040100u);
                if constexpr (MODEL)
                    *reinterpret_cast<uint16_t *>(&sm.dm[bf][xc + e][xt]) =
                        (uint16_t)__builtin_amdgcn_perm(d[e][1], d[e][0], 0x00000400u);
            }
        }
    };
    const int rsh = 15 + a.s_y;
    const int64_t radd = GATED && a.s_y > 0 ? (int64_t)1 << (a.s_y + 14) : 0;
    auto finish = [&](int chunk, auto set_tag) {
        constexpr int ST = decltype(set_tag)::value;
        const int bf = chunk & 1;
        constexpr int OB = GATED ? 1 : 4;   // bytes of an output
        const auto o_rs = __builtin_amdgcn_make_buffer_rsrc(
            (GATED ? a.yo : reinterpret_cast<int8_t *>(a.y)) + (row0 + chunk * TC) * a.x_row * OB, 0,
            rows_of(chunk) * x_row * OB, kBufferRsrcWord3);
#pragma unroll
        for (int j = 0; j < K::FPER; ++j) {
            if (K::FR % 4 != 0 && fr0 + 4 * j >= K::FR) break;   // wave-uniform
            int t, c;
            item(j, t, c);
            const int cs = sm.csum[chunk % 3][t];
            int hi[4], lo[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                hi[e] = cs;            // byte 2 of the high half
                lo[e] = cs + (cs << 8);
            }
#pragma unroll
            for (int w = 0; w < K::NQ; ++w) {
                const v4i u = *reinterpret_cast<const v4i *>(&sm.y[bf][w][0][t][c]);
                const v4i v = *reinterpret_cast<const v4i *>(&sm.y[bf][w][1][t][c]);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    hi[e] += u[e];
                    lo[e] += v[e];
                }
            }
            int o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                // y = hi * 2^16 + (lo mod 2^16) once lo's high half has moved
                // over, and y fits int32 exactly when hi then fits 16 bits
                const int hs = hi[e] + (lo[e] >> 16);
                const int hc = clamp32(hs, -32768, 32767);
                int32_t y = (int32_t)__builtin_amdgcn_perm((uint32_t)hc, (uint32_t)lo[e], 0x05040100u);
                // a y whose high half was clipped is within 2^16 of the int32
                // limit: the SSD clamp, or the gate (at least 1821 / 2^15) and a
                // requant by up to 19 bits, saturate either value alike
                if (!SSD && !(MODEL && a.s_y <= 19) && hs != hc) y = hs > 0 ? INT32_MAX : INT32_MIN;
                if constexpr (GATED) {
                    if constexpr (SSD) y = clamp32(y, -(100 << 18), 100 << 18);
                    // rshr(floor(y * gate / 2^15), s_y) in one shift: nested floors
                    // of a quotient are the floor of the whole one
                    const int32_t gt = sm.gate[(rz[ST][j] >> (8 * e)) & 255];   // in [0, 2^15]
                    o[e] = clamp32((int32_t)(((int64_t)y * gt + radd) >> rsh), -127, 127);
                } else {
                    o[e] = y;
                }
            }
            if constexpr (GATED)
                __builtin_amdgcn_raw_buffer_store_b32(
                    __builtin_amdgcn_perm(__builtin_amdgcn_perm((uint32_t)o[3], (uint32_t)o[2], 0x00000400u),
                                          __builtin_amdgcn_perm((uint32_t)o[1], (uint32_t)o[0], 0x00000400u), 0x05040100u),
                    o_rs, ooff[j], 0, 0);
            else
                __builtin_amdgcn_raw_buffer_store_b128(v4u{(uint32_t)o[0], (uint32_t)o[1], (uint32_t)o[2], (uint32_t)o[3]},
                                                       o_rs, ooff[j], 0, 0);
        }
    };

    // set c & 1 holds chunk c's pieces: loaded two iterations before they are
    // staged (z: two before its epilogue)
    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    load(0, S0{});
    load(1, S1{});   // (rows clamped: in bounds also when there is one chunk)
    load_z(0, S0{});
    stage(0, S0{});
    load(2, S0{});
    __syncthreads();
    // Every wave issues the same loads in every iteration (from clamped rows
    // where it has no use for them): the compiler can then count exactly how
    // many younger loads may stay in flight at each wait.  With the x loads
    // under a branch it waited for all of them, a memory latency per chunk
    // (B8 x L2048 x 1536 channels: 154 against 143 us).
    auto iter = [&](int i, auto cur, auto oth) {
        if (i + 1 < nchunks) stage(i + 1, oth);
        if (i > 0) finish(i - 1, oth);
        load_z(i + 1, oth);
        load(i + 3, oth);
        __syncthreads();
    };
    for (int i = 0; i <= nchunks; i += 2) {
        iter(i, S0{}, S1{});
        if (i + 1 <= nchunks) iter(i + 1, S1{}, S0{});
    }
}

template <int MODE, int N, int S, int M, int MW, int TC>
hipError_t launch(const MfmaScanArgs &a, hipStream_t st) {
    using K = MfmaScan<MODE, N, S, M, MW, TC>;
    static_assert(sizeof(typename K::Smem) <= 163840, "LDS of a CU");
    hipLaunchKernelGGL((mfma_scan_kernel<MODE, N, S, M, MW, TC>), dim3((unsigned)((a.D + K::CH - 1) / K::CH), (unsigned)a.B),
                       dim3(K::NT), 0, st, a);
    return hipGetLastError();
}

}  // namespace

// Channels of a block, by the blocks of 16, 32 and 48 channels that the call makes (us
// per 1000 steps measured with one block on every CU):
//   N = 16   16-channel blocks of 64-step chunks 33; 32 channels 50 (42 without
//            the gate); 48 channels 67 (73).  The least rounds x time wins: one
//            block per CU of 16 channels up to 4096 channels, 32 up to 8192, 48
//            up to 12288 and beyond (B64 x L512 x 4096 channels: 778 us, 855 with
//            32-channel blocks).
//   N = 32   two states a lane; the model's 48-channel blocks beyond one round of
//            16 (B8 x L200 x 1536 channels 32.8 against 34.9 us, B32 115 / 114)
//   N = 64   four states a lane (two: B8 x L1000 x 1536 channels 200 against 174 us)
//   N = 128  four states a lane; beyond one round of 16-channel blocks 32 channels
//            (two sets share a lane's C operand; B4 x L8192 x 24 heads of 64: 1600
//            against 2045 us), in heads that they divide
static int block_channels(int mode, int N, int B, int D, int P) {
    const int64_t cus = device_cus();
    auto rounds = [&](int ch) { return ((int64_t)B * ((D + ch - 1) / ch) + cus - 1) / cus; };
    const int64_t r16 = rounds(16), r32 = rounds(32), r48 = rounds(48);
    if (N == 16 && (mode == kMScanModel || mode == kMScanChannel)) {
        const int64_t t32 = mode == kMScanModel ? 50 : 42, t48 = mode == kMScanModel ? 67 : 73;
        if (33 * r16 <= t32 * r32 && 33 * r16 <= t48 * r48) return 16;
        return t32 * r32 <= t48 * r48 ? 32 : 48;
    }
    if (N == 32 && mode == kMScanModel) return r16 <= 1 ? 16 : 48;
    if (N == 128) return r16 <= 1 || (mode == kMScanHead && P % 32) ? 16 : 32;
    return 16;
}

// A block of the MFMA scan starts slower than one of the VALU kernels (tables, five
// waves' first loads, the helpers' barriers) and its rounds are whole, so short
// sequences are faster there, and with several blocks a CU some of any length.  The
// steps up to which they were, by rounds: the blocks' channels in sixteens over CUs, to
// the next whole block.  Taken from 71,000 random sizes of 2 to 500 steps, both
// kernels each: 0.4% are slower by more than 4% than on the VALU kernels alone (one
// table over channels, not whole blocks, left 2.9%, up to 1.9 times).  MFMA / VALU, us:
//   model N16   6 x 42 x 2048 (batch x steps x channels) 16.8 / 10.2, 31 x 41 x 784 31.7 /
//               14.0, 8 x 512 x 1536 43 / 63, 53 x 269 x 3264 362 / 308 (14 rounds of 48)
//         N32   12 x 38 x 1024 20.7 / 12.4, 59 x 494 x 400 211 / 161; N64 beyond two rounds
//   heads N64   55 x 17 x 54 of 128 206 / 113, 53 x 374 x 5 of 32 65 / 115
//         N32   57 x 21 x 52 of 128 157 / 108; N128 22 x 18 x 21 of 48 35.2 / 29.0
//   channels    N16 64 x 16 x 4096 54 / 39, 1 x 32 x 4096 4.7 / 5.1
int valu_scan_steps(int mode, int N, int B, int D, int P) {
    const int ch = block_channels(mode, N, B, D, P);
    const double r = (double)B * ((D + ch - 1) / ch) * (ch / 16) / device_cus();
    constexpr double kRest = 1e30;
    constexpr int kAll = INT32_MAX;
    auto steps = [&](std::initializer_list<std::pair<double, int>> table) {   // (rounds up to, steps)
        for (const auto &e : table)
            if (r <= e.first) return e.second;
        return 0;
    };
    if (mode == kMScanChannel) {
        if (N == 16 && ch == 16) return steps({{1, 16}, {kRest, 64}});
        if (N == 16 && ch == 32) return steps({{6, 16}, {8, 24}, {12, 12}, {16, 28}, {21, 4}, {kRest, 24}});
        if (N == 16) return 12;
        if (N == 32) return steps({{2, 14}, {3, 4}, {4, 22}, {6, 2}, {8, 12}, {10, 0}, {16, 8}});
        if (N == 64) return steps({{1, 14}, {2, 6}, {3, 0}, {4, 6}, {6, 0}, {8, 6}});
        return ch == 16 ? 0 : steps({{2, 4}, {4, 14}});
    }
    if (mode == kMScanHead) {
        if (N == 16) return steps({{3, 14}, {4, 28}, {5.5, 16}, {8, 28}, {11, 18}, {16, 24}, {21, 14}, {39, 18}, {kRest, 32}});
        if (N == 32) return steps({{2, 14}, {4, 24}, {12, 14}, {16, 20}, {27, 10}, {kRest, 24}});
        if (N == 64) return steps({{1, 28}, {4, 18}, {6, 12}, {8, 20}, {13, 10}, {23, 14}, {45, 18}, {kRest, 40}});
        if (ch == 16) return steps({{1, 18}, {2, 64}, {5.5, 20}, {9, 14}, {kRest, 36}});
        return steps({{2, 14}, {4, 28}, {6, 10}, {10, 18}, {21, 28}, {kRest, 40}});
    }
    if (mode == kMScanModel) {
        if (N == 16 && ch == 16) return steps({{1, 2}, {kRest, 128}});
        if (N == 16 && ch == 32) return steps({{2, 14}, {6, 40}, {14, 64}, {kRest, kAll}});
        if (N == 16) return steps({{4.5, 24}, {6, 40}, {18, 64}, {57, kAll}, {kRest, 128}});
        if (N == 32 && ch == 16) return 4;
        if (N == 32) return steps({{2, kAll}, {3, 24}, {4, kAll}, {4.5, 160}, {6, 80}, {8, kAll}, {9, 64}, {kRest, kAll}});
        return steps({{1, 28}, {2, 160}, {kRest, kAll}});
    }
    if (N == 16) return steps({{1, 0}, {2, 6}, {3, 12}, {10, 40}, {kRest, 64}});
    if (N == 32) return steps({{1, 2}, {2, 10}, {3, 28}, {5, 48}, {kRest, 64}});
    return steps({{1, 18}, {7, 64}, {kRest, 128}});
}

// The model's 32- and 48-channel blocks of N = 16 run up to 256 steps, beyond one round,
// as 32-channel blocks of 16-step chunks, two resident a CU: a block's start costs as
// much as its steps (B16 x L64 x 1536 16.9 -> 15.4 us, B32 x L256 x 4096 205 -> 193,
// B64 x L128 x 4096 234 -> 204).
// Returns hipErrorInvalidValue for a state count it does not take (mfma_scan.hpp has
// the other conditions; short sequences go to other kernels before this).
hipError_t launch_mfma_scan(int mode, int N, const MfmaScanArgs &a, hipStream_t st) {
    const int ch = block_channels(mode, N, a.B, a.D, a.P);
    const bool one16 = (int64_t)a.B * ((a.D + 15) / 16) <= device_cus();
    if (mode == kMScanModel) {
        if (N == 16) {
            if (ch == 16) return launch<kMScanModel, 16, 1, 1, 1, 64>(a, st);
            if (a.L <= 256 && (int64_t)a.B * ((a.D + 47) / 48) > device_cus()) return launch<kMScanModel, 16, 1, 1, 2, 16>(a, st);
            return ch == 32 ? launch<kMScanModel, 16, 1, 1, 2, 32>(a, st) : launch<kMScanModel, 16, 1, 1, 3, 32>(a, st);
        }
        if (N == 32) return ch == 16 ? launch<kMScanModel, 32, 2, 1, 1, 32>(a, st) : launch<kMScanModel, 32, 2, 1, 3, 32>(a, st);
        if (N == 64) return launch<kMScanModel, 64, 2, 1, 1, 32>(a, st);
    } else if (mode == kMScanChannel) {
        if (N == 16)
            return ch == 16   ? launch<kMScanChannel, 16, 1, 1, 1, 64>(a, st)
                   : ch == 32 ? launch<kMScanChannel, 16, 1, 1, 2, 32>(a, st)
                              : launch<kMScanChannel, 16, 1, 1, 3, 32>(a, st);
        if (N == 32) return launch<kMScanChannel, 32, 2, 1, 1, 32>(a, st);
        if (N == 64) return launch<kMScanChannel, 64, 4, 1, 1, 32>(a, st);
        if (N == 128) return ch == 16 ? launch<kMScanChannel, 128, 4, 1, 1, 16>(a, st) : launch<kMScanChannel, 128, 4, 2, 1, 16>(a, st);
    } else if (mode == kMScanHead) {
        // (a block lies in one head: more than 16 channels only where they divide it)
        if (N == 16) return one16 ? launch<kMScanHead, 16, 1, 1, 1, 64>(a, st) : launch<kMScanHead, 16, 1, 1, 1, 32>(a, st);
        if (N == 32) return launch<kMScanHead, 32, 2, 1, 1, 32>(a, st);
        if (N == 64) return launch<kMScanHead, 64, 4, 1, 1, 32>(a, st);
        if (N == 128) return ch == 16 ? launch<kMScanHead, 128, 4, 1, 1, 16>(a, st) : launch<kMScanHead, 128, 4, 2, 1, 16>(a, st);
    } else if (mode == kMScanSsd) {
        if (N == 16) return launch<kMScanSsd, 16, 1, 1, 1, 32>(a, st);
        if (N == 32) return launch<kMScanSsd, 32, 2, 1, 1, 32>(a, st);
        if (N == 64) return launch<kMScanSsd, 64, 4, 1, 1, 32>(a, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace mi
