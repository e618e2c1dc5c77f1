// Device helpers of the kernels that filter the history from an LDS window (taa_window.hip,
// taa_upscale.hip): images through buffer resources, scalar values, wave minima, the packed store.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "taa_device.hpp"
#include "taa_fast_math.hpp"

namespace taastar {
namespace {

__device__ __forceinline__ int scalar(int v) { return __builtin_amdgcn_readfirstlane(v); }
// a kernel argument, read here: read where it is used, each would be a scalar load to wait for in the middle of a phase
__device__ __forceinline__ int scalar_now(int v) {
    asm volatile("" : "+s"(v));
    return v;
}
__device__ __forceinline__ float scalar_now(float v) {
    asm volatile("" : "+s"(v));
    return v;
}
__device__ __forceinline__ bool flag(int v) { return scalar_now(v) != 0; }

// Images through buffer resources: a wave's row is the scalar offset and the column the vector
// offset of one instruction (flat addresses took a 64-bit vector addition a load), and what lies
// behind the image's last texel reads as zero.
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
struct Image {
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ Image(const void* p, int pitch, int w, int h, int bytes)
        : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)(((uint32_t)(h - 1) * (uint32_t)pitch + (uint32_t)w) * (uint32_t)bytes),
                                              0x00020000)) {}
    __device__ __forceinline__ uint32_t ld1(uint32_t v, uint32_t s) const { return __builtin_amdgcn_raw_buffer_load_b32(r, (int)v, (int)s, 0); }
    __device__ __forceinline__ uint2 ld2(uint32_t v, uint32_t s) const {
        const u32x2 q = __builtin_amdgcn_raw_buffer_load_b64(r, (int)v, (int)s, 0);
        return make_uint2(q.x, q.y);
    }
    __device__ __forceinline__ u32x4 ld4(uint32_t v, uint32_t s) const { return __builtin_amdgcn_raw_buffer_load_b128(r, (int)v, (int)s, 0); }
    __device__ __forceinline__ void st2(uint2 q, uint32_t v, uint32_t s) const {
        __builtin_amdgcn_raw_buffer_store_b64(u32x2{q.x, q.y}, r, (int)v, (int)s, 0);
    }
};
__device__ __forceinline__ void ld_vel(const Image& im, uint32_t v, uint32_t s, uint32_t& o) { o = im.ld1(v, s); }
__device__ __forceinline__ void ld_vel(const Image& im, uint32_t v, uint32_t s, uint2& o) { o = im.ld2(v, s); }

__device__ __forceinline__ float lo16(uint32_t v) { return h2f(v & 0xffffu); }
__device__ __forceinline__ float hi16(uint32_t v) { return h2f(v >> 16); }

// two fp32 values as fp16, nearest even, saturating to +-65504, NaN kept: an overflow rounds to
// infinity, which the NaN-propagating minimum / maximum bring back to the largest finite value
__device__ __forceinline__ uint32_t pack_sat(float a, float b) {
    const f32x2_t v = {a, b};
    const h2 hi = {(_Float16)65504.0f, (_Float16)65504.0f};
    h2 r = __builtin_convertvector(v, f16x2_t);
    r = __builtin_elementwise_maximum(__builtin_elementwise_minimum(r, hi), -hi);
    return __builtin_bit_cast(uint32_t, r);
}

// An option of the parameter block: fixed by the kernel's form, or read per launch (kAny).
constexpr int kAny = -1;
__device__ __forceinline__ bool opt(int fixed, bool value) { return fixed == kAny ? value : fixed != 0; }

// min(max(v, LO), hi)
template <int LO>
__device__ __forceinline__ int med3(int v, int hi) {
    int r;
    asm("v_med3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "n"(LO), "s"(hi));
    return r;
}
// minima over the wave of four values (DPP, the four side by side: each step's result is not the next instruction's input)
template <int CTRL, int ROWS>
__device__ __forceinline__ int4 min_step(int4 v) {
    constexpr int kId = 0x7fffffff;
    const int a = __builtin_amdgcn_update_dpp(kId, v.x, CTRL, ROWS, 0xf, false), b = __builtin_amdgcn_update_dpp(kId, v.y, CTRL, ROWS, 0xf, false),
              c = __builtin_amdgcn_update_dpp(kId, v.z, CTRL, ROWS, 0xf, false), d = __builtin_amdgcn_update_dpp(kId, v.w, CTRL, ROWS, 0xf, false);
    return make_int4(min(v.x, a), min(v.y, b), min(v.z, c), min(v.w, d));
}
__device__ __forceinline__ int4 wave_min(int4 v) {
    v = min_step<0x111, 0xf>(v);  // row_shr:1, 2, 4, 8
    v = min_step<0x112, 0xf>(v);
    v = min_step<0x114, 0xf>(v);
    v = min_step<0x118, 0xf>(v);
    v = min_step<0x142, 0xa>(v);  // row_bcast:15, 31
    v = min_step<0x143, 0xc>(v);
    return make_int4(__builtin_amdgcn_readlane(v.x, 63), __builtin_amdgcn_readlane(v.y, 63), __builtin_amdgcn_readlane(v.z, 63),
                     __builtin_amdgcn_readlane(v.w, 63));
}

__device__ __forceinline__ uint32_t select(bool c, uint32_t a, uint32_t b) { return c ? a : b; }
__device__ __forceinline__ uint2 select(bool c, uint2 a, uint2 b) { return make_uint2(c ? a.x : b.x, c ? a.y : b.y); }

}  // namespace
}  // namespace taastar
