// Shared helpers for the gfx950 kernels: error reporting, dtype conversion,
// 16-byte vector access.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#include "../../include/mindspeed_amd.h"

namespace ms {

// 16-byte vector as a native clang vector (usable with the nontemporal builtins).
typedef unsigned int v16 __attribute__((ext_vector_type(4)));

// Streaming (non-temporal) access for data that is touched once.
#define MS_NT_LOAD(p) __builtin_nontemporal_load(p)
#define MS_NT_STORE(v, p) __builtin_nontemporal_store((v), (p))

// ---- host-side error plumbing ------------------------------------------------
void set_error(const char *fmt, ...);

#define MS_REQUIRE(cond, code, ...)      \
    do {                                 \
        if (!(cond)) {                   \
            ms::set_error(__VA_ARGS__);  \
            return (code);               \
        }                                \
    } while (0)

#define MS_CHECK_LAUNCH(what)                                                     \
    do {                                                                          \
        hipError_t e_ = hipGetLastError();                                        \
        if (e_ != hipSuccess) {                                                   \
            ms::set_error("%s: launch failed: %s", (what), hipGetErrorString(e_)); \
            return MS_ERR_HIP;                                                    \
        }                                                                         \
    } while (0)

// hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes), issued once per kernel and device
// (and again only if a larger size is asked for); later calls are a table lookup.  Returns a hipError_t.
hipError_t set_max_dynamic_lds(const void *fn, int bytes);

inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }
inline int dtype_size(int dtype) { return dtype == MS_FP32 ? 4 : 2; }

// ---- device-side dtype helpers -----------------------------------------------
struct BF16 {
    using storage = uint16_t;
    static __device__ __forceinline__ float to_float(uint16_t v) {
        return __uint_as_float(static_cast<uint32_t>(v) << 16);
    }
    static __device__ __forceinline__ uint16_t from_float(float f) {
        __bf16 b = static_cast<__bf16>(f);  // round-to-nearest-even, NaN preserved
        return __builtin_bit_cast(uint16_t, b);
    }
};

struct FP16 {
    using storage = uint16_t;
    static __device__ __forceinline__ float to_float(uint16_t v) {
        return static_cast<float>(__builtin_bit_cast(_Float16, v));
    }
    static __device__ __forceinline__ uint16_t from_float(float f) {
        _Float16 h = static_cast<_Float16>(f);
        return __builtin_bit_cast(uint16_t, h);
    }
};

struct FP32 {
    using storage = float;
    static __device__ __forceinline__ float to_float(float v) { return v; }
    static __device__ __forceinline__ float from_float(float f) { return f; }
};

// A 16-byte vector of DT elements, convertible to / from floats.
template <typename DT>
struct Vec16 {
    static constexpr int N = 16 / sizeof(typename DT::storage);
    v16 raw;
    __device__ __forceinline__ void unpack(float *f) const {
        const typename DT::storage *p = reinterpret_cast<const typename DT::storage *>(&raw);
#pragma unroll
        for (int i = 0; i < N; ++i) f[i] = DT::to_float(p[i]);
    }
    __device__ __forceinline__ void pack(const float *f) {
        typename DT::storage *p = reinterpret_cast<typename DT::storage *>(&raw);
#pragma unroll
        for (int i = 0; i < N; ++i) p[i] = DT::from_float(f[i]);
    }
};

// Load a per-row scalar (probability) of runtime dtype as float.
__device__ __forceinline__ float load_scalar_as_float(const void *p, int64_t i, int dtype) {
    if (dtype == MS_FP32) return reinterpret_cast<const float *>(p)[i];
    uint16_t v = reinterpret_cast<const uint16_t *>(p)[i];
    return dtype == MS_BF16 ? BF16::to_float(v) : FP16::to_float(v);
}
__device__ __forceinline__ void store_float_as(void *p, int64_t i, int dtype, float f) {
    if (dtype == MS_FP32) {
        reinterpret_cast<float *>(p)[i] = f;
    } else {
        reinterpret_cast<uint16_t *>(p)[i] = dtype == MS_BF16 ? BF16::from_float(f) : FP16::from_float(f);
    }
}

// 1 / (1 + exp(-x)) of a 16-bit value, for results that are rounded to 16 bits.  The reciprocal instruction (1 ulp) and one Newton
// step, five instructions where the division takes ten.  The instruction has no subnormal results, but x times one is a normal
// bfloat16 (x = -87.5, -88, -88.5): it sees a quarter of 1 + exp(-x), at most 2^126, and the last product is the only one that
// rounds to a subnormal.  Past exp's overflow the step's factor is NaN, which fmaxf takes out: 0, as the division gives.
__device__ __forceinline__ float sigmoid16(float x) {
    const float d = fmaf(__expf(-x), 0.25f, 0.25f);
    const float r = __builtin_amdgcn_rcpf(d);
    return fmaf(fmaxf(fmaf(-d, r, 1.f), -1.f), r, r) * 0.25f;
}

// ---- prefix sums over the lanes of a wavefront ----------------------------------
// v moved over the lanes (data-parallel primitives: 8 clocks each, a shuffle through LDS takes a hundred); lanes without a
// source get 0.
template <int CTRL, int ROWS>
__device__ __forceinline__ int lane_move(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, false);
}
// ... of a value made of 32-bit words
template <int CTRL, int ROWS, typename T>
__device__ __forceinline__ T lanes_move(const T &v) {
    static_assert(sizeof(T) % 4 == 0, "scan items are made of 32-bit words");
    T r;
#pragma unroll
    for (int w = 0; w < static_cast<int>(sizeof(T) / 4); ++w)
        reinterpret_cast<int *>(&r)[w] = lane_move<CTRL, ROWS>(reinterpret_cast<const int *>(&v)[w]);
    return r;
}
// Inclusive prefix of v over the 64 lanes of a wavefront (all of them active); all-zero words must be neutral for op.
template <typename T, typename Op>
__device__ __forceinline__ T wave_scan(T v, Op op) {
    v = op(v, lanes_move<0x111, 0xf>(v));       // row_shr:1
    v = op(v, lanes_move<0x112, 0xf>(v));       // row_shr:2
    v = op(v, lanes_move<0x114, 0xf>(v));       // row_shr:4
    v = op(v, lanes_move<0x118, 0xf>(v));       // row_shr:8
    v = op(v, lanes_move<0x142, 0xa>(v));       // row_bcast:15 to rows 1 and 3
    return op(v, lanes_move<0x143, 0xc>(v));    // row_bcast:31 to rows 2 and 3
}
// The value of the lane below (0 in lane 0).
template <typename T>
__device__ __forceinline__ T lane_below(const T &v) { return lanes_move<0x138, 0xf>(v); }      // wave_shr:1

}  // namespace ms
