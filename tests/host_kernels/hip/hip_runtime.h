// Stand-in for the HIP runtime that runs the library's kernels on the host, one thread
// after another: LDS arrays are static, barriers and waits do nothing, cross-lane
// operations give a lane its own value and matrix products are not computed.  Results
// mean nothing; the addresses, which follow from the arguments alone, are the kernels'
// own, and AddressSanitizer sees each access to global memory and to LDS arrays.
#pragma once
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <type_traits>
#include <utility>
#define __global__
#define __device__
#define __host__
#define __forceinline__ inline
#define __shared__ static
#define __constant__
#define __launch_bounds__(...)
#define amdgpu_waves_per_eu(x) unused
#define __align__(n) __attribute__((aligned(n)))
struct dim3 { unsigned x, y, z; constexpr dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {} };
extern dim3 blockIdx, threadIdx, blockDim, gridDim;
extern int8_t *host_dynamic_lds;
struct int2 { int x, y; } __attribute__((aligned(8)));
struct uint2 { unsigned x, y; } __attribute__((aligned(8)));
struct int4 { int x, y, z, w; } __attribute__((aligned(16)));
struct uint4 { unsigned x, y, z, w; } __attribute__((aligned(16)));
inline int2 make_int2(int a, int b) { return {a, b}; }
inline uint2 make_uint2(unsigned a, unsigned b) { return {a, b}; }
inline int4 make_int4(int a, int b, int c, int d) { return {a, b, c, d}; }
inline uint4 make_uint4(unsigned a, unsigned b, unsigned c, unsigned d) { return {a, b, c, d}; }
template <class A, class B> constexpr std::common_type_t<A, B> min(A a, B b) { return (std::common_type_t<A, B>)a < (std::common_type_t<A, B>)b ? a : b; }
template <class A, class B> constexpr std::common_type_t<A, B> max(A a, B b) { return (std::common_type_t<A, B>)a < (std::common_type_t<A, B>)b ? b : a; }
inline void __syncthreads() {}
template <class T> T __shfl_xor(T v, int, int = 64) { return v; }
template <class T> T __shfl(T v, int, int = 64) { return v; }
template <class T> T __shfl_down(T v, int, int = 64) { return v; }
extern int host_vote;   // what every vote gives: 0 or 1
inline int __all(int) { return host_vote; }
inline int __any(int) { return host_vote; }
inline float __fdiv_rn(float a, float b) { return a / b; }
inline float __fmul_rn(float a, float b) { return a * b; }
inline float __fadd_rn(float a, float b) { return a + b; }
inline int __mul24(int a, int b) { return (int)((int64_t)(a << 8 >> 8) * (b << 8 >> 8)); }
inline unsigned __umul24(unsigned a, unsigned b) { return (a & 0xffffff) * (b & 0xffffff); }
inline unsigned __umulhi(unsigned a, unsigned b) { return (unsigned)((uint64_t)a * b >> 32); }
template <class T> T atomicAdd(T *p, T v) { T o = *p; *p += v; return o; }
template <class T> T atomicMax(T *p, T v) { T o = *p; if (v > o) *p = v; return o; }
inline unsigned __builtin_amdgcn_alignbit(unsigned h, unsigned l, unsigned s) { return (unsigned)((((uint64_t)h << 32) | l) >> (s & 31)); }
inline unsigned __builtin_amdgcn_cvt_pk_u8_f32(float f, unsigned r, unsigned o) { int v = f < 0 ? 0 : f > 255 ? 255 : (int)rintf(f); return (o & ~(255u << 8 * r)) | (unsigned)v << 8 * r; }
typedef int host_v4i __attribute__((ext_vector_type(4)));
typedef int host_v16i __attribute__((ext_vector_type(16)));
typedef unsigned host_v2u __attribute__((ext_vector_type(2)));
typedef unsigned host_v4u __attribute__((ext_vector_type(4)));
typedef short host_v2s __attribute__((ext_vector_type(2)));
inline host_v4i __builtin_amdgcn_mfma_i32_16x16x64_i8(host_v4i a, host_v4i b, host_v4i c, int, int, int) { return c + (a ^ b); }
inline host_v16i __builtin_amdgcn_mfma_i32_32x32x32_i8(host_v4i a, host_v4i b, host_v16i c, int, int, int) { c[0] += a[0] ^ b[0]; return c; }
inline int __builtin_amdgcn_mov_dpp(int v, int, int, int, bool) { return v; }
inline int __builtin_amdgcn_update_dpp(int, int v, int, int, int, bool) { return v; }
inline unsigned __builtin_amdgcn_perm(unsigned a, unsigned b, unsigned s) {
    uint64_t q = ((uint64_t)a << 32) | b; unsigned r = 0;
    for (int i = 0; i < 4; ++i) { unsigned k = (s >> 8 * i) & 255, v = k < 8 ? (q >> 8 * k) & 255 : 0; r |= v << 8 * i; }
    return r;
}
inline host_v2u __builtin_amdgcn_permlane16_swap(unsigned a, unsigned b, bool, bool) { return host_v2u{a, b}; }
inline host_v2u __builtin_amdgcn_permlane32_swap(unsigned a, unsigned b, bool, bool) { return host_v2u{a, b}; }
inline int __builtin_amdgcn_readfirstlane(int v) { return v; }
inline void __builtin_amdgcn_s_barrier() {}
inline void __builtin_amdgcn_wave_barrier() {}
inline void __builtin_amdgcn_s_setprio(int) {}
inline void __builtin_amdgcn_s_waitcnt(int) {}
inline void __builtin_amdgcn_sched_barrier(int) {}
inline void __builtin_amdgcn_sched_group_barrier(int, int, int) {}
inline int __builtin_amdgcn_sdot2(host_v2s a, host_v2s b, int c, bool) { return (int)((unsigned)c + a[0] * b[0] + a[1] * b[1]); }
inline int __builtin_amdgcn_sdot4(int a, int b, int c, bool) { for (int i = 0; i < 4; ++i) c += (int)(int8_t)(a >> 8 * i) * (int)(int8_t)(b >> 8 * i); return c; }
inline float __builtin_amdgcn_sqrtf(float v) { return sqrtf(v); }
inline float __builtin_amdgcn_rcpf(float v) { return 1.0f / v; }
// buffers: an access is in range as a whole, out of range as a whole, or the run ends
struct __amdgpu_buffer_rsrc_t { char *base; uint32_t num; };
[[noreturn]] void host_die(const char *what, long long a, long long b);
template <class T> __amdgpu_buffer_rsrc_t __builtin_amdgcn_make_buffer_rsrc(T *p, short, int num, int) {
    if (num < 0) host_die("negative num_records", num, 0);
    return {(char *)p, (uint32_t)num};
}
inline char *host_buf(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t so, uint32_t n) {
    const uint64_t a = (uint64_t)off + so;
    if (off >= r.num || a >= r.num) return nullptr;
    if (a + n > r.num) host_die("access straddles the end of its buffer", (long long)a, r.num);
    return r.base + a;
}
template <class T> T host_load(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t so) { T v{}; if (char *p = host_buf(r, off, so, sizeof(T))) v = *(T *)p; return v; }
inline uint8_t __builtin_amdgcn_raw_buffer_load_b8(__amdgpu_buffer_rsrc_t r, uint32_t o, uint32_t s, int) { return host_load<uint8_t>(r, o, s); }
inline uint32_t __builtin_amdgcn_raw_buffer_load_b32(__amdgpu_buffer_rsrc_t r, uint32_t o, uint32_t s, int) { return host_load<uint32_t>(r, o, s); }
inline host_v2u __builtin_amdgcn_raw_buffer_load_b64(__amdgpu_buffer_rsrc_t r, uint32_t o, uint32_t s, int) { return host_load<host_v2u>(r, o, s); }
inline host_v4u __builtin_amdgcn_raw_buffer_load_b128(__amdgpu_buffer_rsrc_t r, uint32_t o, uint32_t s, int) { return host_load<host_v4u>(r, o, s); }
inline void __builtin_amdgcn_raw_buffer_store_b32(uint32_t v, __amdgpu_buffer_rsrc_t r, uint32_t o, uint32_t s, int) { if (char *p = host_buf(r, o, s, 4)) *(uint32_t *)p = v; }
inline void __builtin_amdgcn_raw_buffer_store_b128(host_v4u v, __amdgpu_buffer_rsrc_t r, uint32_t o, uint32_t s, int) { if (char *p = host_buf(r, o, s, 16)) *(host_v4u *)p = v; }
typedef __attribute__((address_space(3))) void host_lds;
typedef __attribute__((address_space(1))) void host_glob;
inline void __builtin_amdgcn_raw_ptr_buffer_load_lds(__amdgpu_buffer_rsrc_t r, host_lds *l, int n, uint32_t off, uint32_t so, int imm, int) {
    char *d = (char *)(void *)l + imm + n * (threadIdx.x & 63);
    char *p = host_buf(r, off + imm, so, n);
    if (!p) host_die("LDS load outside its buffer", off, r.num);
    memcpy(d, p, n);
}
inline void __builtin_amdgcn_global_load_lds(host_glob *g, host_lds *l, int n, int imm, int) {
    memcpy((char *)(void *)l + imm + n * (threadIdx.x & 63), (char *)(void *)g + imm, n);
}
// host side
typedef void *hipStream_t;
typedef int hipError_t;
enum { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorNotReady = 2, hipDeviceAttributeMultiprocessorCount = 0 };
extern int host_cus;
inline const char *hipGetErrorString(int) { return "error"; }
extern int host_dry, host_error;   // dry: launches are checked against the runtime's limits, not run
inline int hipGetLastError() { const int e = host_error; host_error = 0; return e; }
inline int hipGetDevice(int *d) { *d = 0; return 0; }
inline int hipDeviceGetAttribute(int *v, int, int) { *v = host_cus; return 0; }
enum { hipMemcpyDeviceToDevice, hipMemcpyHostToDevice };
inline int hipMemcpyAsync(void *d, const void *s, size_t n, int, void *) { memcpy(d, s, n); return 0; }
template <class F> int hipFuncSetAttribute(F, int, int) { return 0; }
enum { hipFuncAttributeMaxDynamicSharedMemorySize };
extern const char *host_kernel;
template <class... P, class... A> void host_launch(const char *name, void (*f)(P...), dim3 g, dim3 b, size_t dyn, A... a) {
    host_kernel = name;
    gridDim = g; blockDim = b;
    if (host_dry) {
        if (!g.x || (uint64_t)g.x * b.x >> 32 || !g.y || g.y > 65535 || !g.z || g.z > 65535) host_error = hipErrorInvalidValue;
        return;
    }
    host_dynamic_lds = dyn ? (int8_t *)aligned_alloc(16, (dyn + 15) / 16 * 16) : nullptr;
    for (unsigned z = 0; z < g.z; ++z) for (unsigned y = 0; y < g.y; ++y) for (unsigned x = 0; x < g.x; ++x) {
        blockIdx = dim3(x, y, z);
        for (unsigned t = 0; t < b.x; ++t) { threadIdx = dim3(t, 0, 0); f(static_cast<P>(a)...); }
    }
    free(host_dynamic_lds);
}
#define hipLaunchKernelGGL(k, g, b, s, st, ...) ((void)(st), host_launch(#k, k, g, b, s, __VA_ARGS__))
