// Calls the library's entry points, built for the host (hip/hip_runtime.h beside this
// file), over random sizes with buffers of exactly the documented extents.
//   addresses FAMILY COUNT SEED
#include <hip/hip_runtime.h>

#include <random>
#include <vector>

#include "mamba_int.h"

dim3 blockIdx, threadIdx, blockDim, gridDim;
int8_t *host_dynamic_lds;
int host_vote, host_cus, host_dry, host_error;
const char *host_kernel = "";

void host_die(const char *what, long long a, long long b) {
    printf("%s: %lld of %lld in %s, block %u,%u thread %u\n", what, a, b, host_kernel, blockIdx.x, blockIdx.y, threadIdx.x);
    fflush(stdout);
    abort();
}

namespace {

std::mt19937 rng;
int uni(int a, int b) { return a + (int)(rng() % (unsigned)(b - a + 1)); }
int logu(int lo, int hi) {
    const int v = (int)lround(exp(log(lo) + (log(hi) - log(lo)) * (rng() / 4294967296.0)));
    return v < lo ? lo : v > hi ? hi : v;
}
int up(int v, int u) { return (v + u - 1) / u * u; }

struct Pool {   // the buffers of one call
    std::vector<void *> v;
    ~Pool() { for (void *p : v) free(p); }
    template <class T> T *get(size_t n) {
        T *p = (T *)malloc(n ? n * sizeof(T) : 1);
        v.push_back(p);
        for (size_t i = 0; i < n * sizeof(T); i += 1 + rng() % 7) ((uint8_t *)p)[i] = (uint8_t)(rng() >> 3);
        return p;
    }
};
int calls, refused;
void call(mi_status st) {
    ++calls;
    refused += st != MI_OK;
}

// path: 0 by rows, 1 the GEMM, 2 the GEMV; a's last row ends with its used part
void linear(Pool &p, const int8_t *a, int lda, int kind, int m, int n, int k, void *out, int ldo, int path = 0) {
    auto f = path == 1 ? mi_bitlinear_gemm : path == 2 ? mi_bitlinear_gemv : mi_bitlinear;
    const bool stats = kind == MI_OUT_RESIDUAL && uni(0, 1);
    call(f(a, lda, p.get<uint8_t>((size_t)n * k / 4), out, ldo, kind, m, n, k, kind == MI_OUT_INT8 || kind == MI_OUT_DECAY_MOD ? 6 : 0,
           4719, uni(0, 3) ? 16 : 40, 0, kind == MI_OUT_FLOAT ? p.get<float>(m) : nullptr, 1.0f, stats ? p.get<int64_t>((size_t)2 * m) : nullptr, nullptr));
}

void bitlinear(bool large) {
    Pool p;
    const int m = large ? uni(1500, 2600) : logu(1, 3000), n = large ? 256 * uni(24, 30) : logu(1, 3000);
    const int k = large ? 128 * uni(1, 2) : 16 * logu(1, 130), kind = uni(0, 4);
    const int lda = k + 16 * (uni(0, 2) == 0), ldo = up(n, uni(0, 1) ? 4 : 16), out1 = kind == MI_OUT_INT8 || kind == MI_OUT_DECAY_MOD;
    linear(p, p.get<int8_t>((size_t)(m - 1) * lda + k), lda, kind, m, n, k, p.get<int8_t>((size_t)m * ldo * (out1 ? 1 : 4)), ldo,
           m <= 64 ? uni(0, 2) : uni(0, 1));
}

void bitlinear_f32() {
    Pool p;
    const int m = logu(1, 1500), n = 4 * logu(1, 768), k = logu(1, 5000), kp = up(k, uni(0, 1) ? 16 : 64), off = uni(0, 3);
    call(mi_bitlinear_f32(p.get<float>((size_t)m * k + off) + off, k, p.get<uint8_t>((size_t)n * kp / 4), kp, 1.0f,
                          uni(0, 1) ? p.get<float>(n) : nullptr, p.get<int8_t>((size_t)m * kp), p.get<float>(m),
                          p.get<float>((size_t)m * n), n, m, n, nullptr));
}

// the prefill kernels of a dyadic block
void block(int B, int L, int d, int R, int N) {
    Pool p;
    const int D = 2 * d, T = B * L, X = R + 2 * N;
    const bool state = uni(0, 1);
    int32_t *r = p.get<int32_t>((size_t)T * d), *h = p.get<int32_t>((size_t)B * D * N), *cb = p.get<int32_t>(D);
    int8_t *a = p.get<int8_t>((size_t)T * d), *xz = p.get<int8_t>((size_t)T * 2 * D), *xs = p.get<int8_t>((size_t)T * D);
    int8_t *xp = p.get<int8_t>((size_t)T * X), *dm = p.get<int8_t>((size_t)T * D), *yo = p.get<int8_t>((size_t)T * D);
    int8_t *cw = p.get<int8_t>((size_t)D * 4), *c0 = p.get<int8_t>((size_t)B * 3 * D), *c1 = p.get<int8_t>((size_t)B * 3 * D);
    call(mi_bitshift_norm(r, p.get<int16_t>(d), a, T, d, uni(0, 1) ? p.get<int64_t>((size_t)T * 2) : nullptr, nullptr));
    if (D % 128 == 0 && d % 64 == 0) {
        call(mi_in_proj_conv(a, d, p.get<uint8_t>((size_t)2 * D * d / 4), 6, cw, cb, state ? c0 : nullptr, c1, xs, xz, 2 * D, B, L, d, D, nullptr));
    } else {
        linear(p, a, d, MI_OUT_INT8, T, 2 * D, d, xz, 2 * D);
        call(mi_conv_squareplus(xz, 2 * D, cw, cb, state ? c0 : nullptr, c1, xs, B, L, D, nullptr));
    }
    linear(p, xs, D, MI_OUT_INT8, T, X, D, xp, X);
    linear(p, xp, X, MI_OUT_DECAY_MOD, T, D, R, dm, D);
    call(mi_block_scan(xs, dm, xp, X, R, xz, 2 * D, D, p.get<int32_t>((size_t)D * N), 15, 14, yo, state ? h : nullptr, h, B, L, D, N, nullptr));
    linear(p, yo, D, MI_OUT_RESIDUAL, T, d, D, r, d);
}

void ssd_scan(int B, int L, int H, int P, int N) {
    Pool p;
    const int D = H * P, X = up(2 * H * N + H, 16) + 16 * uni(0, 1), Z = 2 * D + 16 * uni(0, 1);
    const size_t T = (size_t)B * L;
    int32_t *h = p.get<int32_t>((size_t)B * D * N);
    call(mi_ssd_block_scan(p.get<int8_t>(T * D), p.get<int8_t>((T - 1) * X + 2 * H * N + H), X, p.get<int8_t>((T - 1) * Z + 2 * D), Z, D,
                           p.get<int32_t>((size_t)H * 255), H, 12, p.get<int8_t>(T * D), uni(0, 1) ? h : nullptr, uni(0, 2) ? h : nullptr, B,
                           L, D, N, nullptr));
}

void scans(int B, int L) {
    {
        Pool p;
        const int D = 16 * logu(1, 128) + (uni(0, 4) == 0), N = uni(0, 5) ? 16 << uni(0, 3) : uni(1, 128);
        const size_t T = (size_t)B * L;
        int32_t *h = p.get<int32_t>((size_t)B * D * N);
        call(mi_dyadic_scan(p.get<int8_t>(T * D), p.get<int8_t>(T * N), p.get<int8_t>(T * N), p.get<int32_t>((size_t)D * N), 15,
                            p.get<int32_t>(T * D), uni(0, 1) ? h : nullptr, h, B, L, D, N, nullptr));
    }
    {
        Pool p;
        const int H = logu(1, 24), P = 16 * uni(1, 4), N = 16 << uni(0, 3), cs = 64 * uni(1, 3);
        const size_t T = (size_t)B * L;
        int32_t *h = p.get<int32_t>((size_t)B * H * P * N);
        call(mi_ssd_chunked_scan(p.get<int8_t>(T * H * P), p.get<int8_t>(T * H * N), p.get<int8_t>(T * H * N), p.get<int32_t>(H), 15,
                                 p.get<int32_t>(T * H * P), p.get<int32_t>((size_t)B * ((L + cs - 1) / cs) * H * P * N),
                                 uni(0, 1) ? h : nullptr, h, B, L, H, P, N, cs, nullptr));
    }
}

void elementwise(int B, int L, int C) {
    Pool p;
    const size_t n = (size_t)B * L * C, s = (size_t)B * C;
    const int cs = logu(1, 300);
    const size_t q = (size_t)B * ((L + cs - 1) / cs) * C;
    call(mi_dyadic_scan_elementwise(p.get<int32_t>(n), p.get<int32_t>(n), 15, p.get<int32_t>(n), p.get<int32_t>(s), p.get<int32_t>(s), B, L, C, nullptr));
    call(mi_dyadic_chunked_scan(p.get<int32_t>(n), p.get<int32_t>(n), 15, cs, p.get<int32_t>(n), p.get<int32_t>(q), p.get<int32_t>(q),
                                p.get<int32_t>(s), p.get<int32_t>(s), B, L, C, nullptr));
}

// the fused and batched stages of one decode step (calls past a stage's limits are refused)
void decode(int m, int d, int N, int R) {
    Pool p;
    const int D = 2 * d, nx = R + 2 * N, V = uni(1, 300), np = uni(0, 2), parts = np == 2 ? (d + 15) / 16 : 1, nk = (V + 63) / 64;
    int32_t *r = p.get<int32_t>((size_t)m * d), *h = p.get<int32_t>((size_t)m * D * N), *cb = p.get<int32_t>(D), *base = p.get<int32_t>((size_t)D * N);
    int64_t *st = np ? p.get<int64_t>((size_t)m * parts * 2) : nullptr, *keys = p.get<int64_t>((size_t)m * nk), *ids = p.get<int64_t>(m);
    int16_t *ga = p.get<int16_t>(d);
    int8_t *cw = p.get<int8_t>((size_t)D * 4), *cs = p.get<int8_t>((size_t)m * 3 * D), *xs = p.get<int8_t>((size_t)m * D);
    int8_t *xz = p.get<int8_t>((size_t)m * 2 * D), *xp = p.get<int8_t>((size_t)m * nx), *yo = p.get<int8_t>((size_t)m * D), *emb = p.get<int8_t>((size_t)V * d);
    uint8_t *wi = p.get<uint8_t>((size_t)2 * D * d / 4), *wx = p.get<uint8_t>((size_t)nx * D / 4), *wd = p.get<uint8_t>((size_t)D * R / 4);
    uint8_t *wo = p.get<uint8_t>((size_t)d * D / 4), *wh = p.get<uint8_t>((size_t)V * d / 4);
    int32_t *xpart = p.get<int32_t>((size_t)m * (D / 16) * nx), *xq = p.get<int32_t>((size_t)m * 4 * nx);
    call(mi_embed(p.get<int64_t>(m), emb, r, m, d, V, p.get<int64_t>((size_t)2 * m), 1, nullptr));
    call(mi_norm_in_proj_conv(r, st, parts, ga, wi, 6, cw, cb, cs, xs, xz, m, d, D, nullptr));
    call(mi_norm_v2_in_proj_conv(r, st, parts, ga, wi, 6, cw, cb, cs, xs, xz, m, d, D, nullptr));
    call(mi_norm_in_proj_conv_xpart(r, st, parts, ga, wi, 6, cw, cb, cs, xs, xz, wx, nx, xpart, m, d, D, nullptr));
    call(mi_xpart_dt_scan_step(xpart, D / 16, 6, R, wd, 5, xs, xz, 2 * D, D, base, 15, 14, h, yo, m, D, N, nullptr));
    call(mi_xproj_dt_scan_step(xs, wx, 6, R, wd, 5, xz, 2 * D, D, base, 15, 14, h, yo, m, D, N, nullptr));
    call(mi_dt_scan_step(xp, nx, R, wd, 5, xs, xz, 2 * D, D, base, 15, 14, h, yo, m, D, N, nullptr));
    call(mi_conv_step_xproj(xz, 2 * D, cw, cb, cs, xs, wx, 6, nx, xp, nx, m, D, nullptr));
    call(mi_conv_step_xpart(xz, 2 * D, cw, cb, cs, xs, wx, nx, xq, m, D, nullptr));
    call(mi_xpart_dt_scan_step(xq, 4, 6, R, wd, 5, xs, xz, 2 * D, D, base, 15, 14, h, yo, m, D, N, nullptr));
    int64_t *ps = p.get<int64_t>((size_t)m * ((d + 15) / 16) * 2);
    call(mi_bitlinear_residual_parts(yo, D, wo, r, d, m, d, D, 4719, 16, 0, ps, nullptr));
    call(mi_bitshift_norm_parts(r, ga, p.get<int8_t>((size_t)m * d), m, d, ps, (d + 15) / 16, uni(0, 1), nullptr));
    call(mi_norm_bitlinear(r, st, parts, ga, wh, p.get<int32_t>((size_t)m * up(V, 4)), up(V, 4), MI_OUT_INT32, m, V, d, 0, nullptr));
    call(mi_norm_bitlinear_argmax(r, st, parts, ga, wh, p.get<int32_t>((size_t)m * up(V, 4)), up(V, 4), keys, m, V, d, nullptr));
    call(mi_argmax_keys(keys, nk, ids, m, nullptr));
    call(mi_embed_argmax(keys, nk, ids, emb, r, m, d, V, p.get<int64_t>((size_t)2 * m), 1, nullptr));
    call(mi_argmax_i32(p.get<int32_t>((size_t)m * V), V, ids, m, V, nullptr));
}

// calls at the launch limits, which no kernel runs for: every one has a kernel that takes it
void limits() {
    host_dry = 1;
    host_cus = 256;
    auto *p = (int32_t *)(1ull << 40);
    auto *b = (int8_t *)p;
    for (int B : {1 << 24, 16867619, 20000000})
        for (int C : {33, 36}) {
            call(mi_dyadic_scan_elementwise(p, p, 15, p, p, p, B, 33, C, nullptr));
            call(mi_dyadic_chunked_scan(p, p, 15, 12, p, p, p, p, p, B, 33, C, nullptr));
        }
    for (int m : {585956566, 586902066})
        for (int k : {16, 32, 48, 64})
            for (int kind : {MI_OUT_INT8, MI_OUT_DECAY_MOD})
                call(mi_bitlinear_gemm(b, k, (uint8_t *)b, b, 352, kind, m, 352, k, 6, 0, 0, 0, nullptr, 1.0f, nullptr, nullptr));
    if (refused) printf("last kernel %s\n", host_kernel), exit(4);
}

}  // namespace

int main(int argc, char **argv) {
    const char *what = argv[1];
    auto is = [&](const char *s) { return !strcmp(what, s); };
    rng.seed(atoi(argv[3]));
    if (is("limits")) limits();
    for (int i = 0; i < atoi(argv[2]); ++i) {
        host_vote = i & 1;
        // the dispatch of small and of large devices, so that every split is reached at small sizes
        host_cus = uni(0, 1) ? 256 : logu(1, 64);
        if (is("bitlinear")) bitlinear(i % 24 == 0);
        else if (is("bitlinear_f32")) bitlinear_f32();
        else if (is("block")) block(logu(1, 6), logu(1, 250), (uni(0, 5) ? 64 : 16) * logu(1, 10), 16 * uni(1, 5), 16 << uni(0, 2));
        else if (is("block_2103")) block(3, 701, 1024, 64, 16);
        else if (is("ssd_scan")) ssd_scan(logu(1, 8), logu(1, 200), logu(1, 24), 16 * uni(1, 5), 16 << uni(0, 2));
        else if (is("scans")) scans(logu(1, 16), logu(1, 250));
        else if (is("elementwise")) elementwise(logu(1, 64), logu(1, 150), logu(1, 1500));
        else if (is("limits")) continue;
        else if (is("decode")) decode(logu(1, 70), 64 * logu(1, 10), 16 << uni(0, 2), 16 * uni(1, 5));
        else return 2;
    }
    printf("%d calls, %d refused\n", calls, refused);
    return calls > refused ? 0 : 3;
}
