// The passes over a finished image: the edge-AA fallback for the texels the segmentation mask puts in
// category 1 (the prepare + FXAA passes of source/taa.hpp:1061-1107) with the library's own filter --
// every texel gets alpha = luma (the prepare pass); a category-1 texel with enough local luma contrast is
// blended with the 4-neighbour across its edge (include/taastar/taa_abi.h states the filter) -- and
// sharpen_cas.comp on its own. FP32 arithmetic without contraction (this file is compiled with
// -ffp-contract=off), in the oracle's order.
//
// What bounds them: HBM at the rate of a copy. A texel a lane with its neighbours gathered from memory left the loads
// exposed one behind the other (centre and mask, then the eight neighbours, then the blended one) and cost a vector load
// each. Now a wave takes 16 bytes a lane of four rows and the row on either side, all loads first: the neighbours in a row
// come from the lanes beside (two texels at the wave's ends from a load of their own, which keeps the stores aligned to whole
// lines; waves that overlap by a lane instead ran 3% slower on FP32 storage), those above and below from registers, and a texel's
// luma is computed once, not by nine.
// us for both passes, before and now: 2560x1440 RGBA16F 41.1 and 31.1, 3840x2160 86.7 and 60.1, 1280x720 12.7 and 10.9;
// RGBA32F 2560x1440 54.7 and 47.8, 3840x2160 117 and 118 (565 MB: the card copies 4.78 TB/s).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "taa_device.hpp"
#include "taa_internal.hpp"
#include "taa_wave.hpp"

namespace taastar {
namespace {

// the value of the lane before / after (a wave shift); the first / last lane's is `other`
__device__ __forceinline__ uint32_t lane_before(uint32_t v, uint32_t other) { return (uint32_t)__builtin_amdgcn_update_dpp((int)other, (int)v, 0x138, 0xf, 0xf, false); }
__device__ __forceinline__ uint32_t lane_after(uint32_t v, uint32_t other) { return (uint32_t)__builtin_amdgcn_update_dpp((int)other, (int)v, 0x130, 0xf, 0xf, false); }
__device__ __forceinline__ float lane_before(float v, float o) { return __uint_as_float(lane_before(__float_as_uint(v), __float_as_uint(o))); }
__device__ __forceinline__ float lane_after(float v, float o) { return __uint_as_float(lane_after(__float_as_uint(v), __float_as_uint(o))); }
__device__ __forceinline__ f3 lane_before(f3 v, f3 o) { return {lane_before(v.x, o.x), lane_before(v.y, o.y), lane_before(v.z, o.z)}; }
__device__ __forceinline__ f3 lane_after(f3 v, f3 o) { return {lane_after(v.x, o.x), lane_after(v.y, o.y), lane_after(v.z, o.z)}; }
__device__ __forceinline__ uint2 lane_before(uint2 v, uint2 o) { return make_uint2(lane_before(v.x, o.x), lane_before(v.y, o.y)); }
__device__ __forceinline__ uint2 lane_after(uint2 v, uint2 o) { return make_uint2(lane_after(v.x, o.x), lane_after(v.y, o.y)); }

// A wave filters R rows of 64 lanes' texels, 16 bytes a lane (two RGBA16F texels or one RGBA32F); its first and last lane
// hold the texel beside the wave's as well. Four waves of a workgroup lie below each other.
template <bool S16, int R_>
struct Rows {
    static constexpr int T = S16 ? 2 : 1, R = R_, OUT = 64 * T;
    typedef typename std::conditional<S16, uint2, f3>::type Tex;
    int x, y0, beside;  // the lane's first texel, the wave's first row, the column beside it (-1: another lane's)
    bool store, inside;
    __device__ __forceinline__ Rows(int tile, int tiles_x, int W) {
        const int ty = scalar(tile / tiles_x), lane = (int)threadIdx.x & 63;
        const int first = (tile - ty * tiles_x) * OUT;
        x = first + T * lane;
        y0 = (ty * 4 + scalar((int)threadIdx.x >> 6)) * R;
        store = x < W;
        inside = first + OUT <= W;  // no texel of the wave to clamp
        beside = lane == 0 ? max(x - 1, 0) : lane == 63 ? min(x + T, W - 1) : -1;
    }
    // row y, clamped to the image's edge
    __device__ __forceinline__ void load(const Image& src, int pitch, int y, int W, int H, Tex (&e)[T]) const {
        const uint32_t r = (uint32_t)clampi(y, 0, H - 1) * (uint32_t)pitch;
        if constexpr (S16) {
            u32x4 v;
            if (inside) {
                v = src.ld4((r + (uint32_t)x) * 8u, 0u);
            } else {
                const uint2 a = src.ld2((r + (uint32_t)clampi(x, 0, W - 1)) * 8u, 0u), b = src.ld2((r + (uint32_t)clampi(x + 1, 0, W - 1)) * 8u, 0u);
                v = u32x4{a.x, a.y, b.x, b.y};
            }
            e[0] = make_uint2(v.x, v.y);
            e[1] = make_uint2(v.z, v.w);
        } else {
            const u32x4 v = src.ld4((r + (uint32_t)clampi(x, 0, W - 1)) * 16u, 0u);
            e[0] = {__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z)};
        }
    }
    // the first and last lane's texel beside the wave's, row y
    __device__ __forceinline__ Tex load_beside(const Image& src, int pitch, int y, int H) const {
        const uint32_t o = (uint32_t)clampi(y, 0, H - 1) * (uint32_t)pitch + (uint32_t)beside;  // (an offset past the image reads nothing)
        if constexpr (S16) {
            return src.ld2(beside < 0 ? ~15u : o * 8u, 0u);
        } else {
            const u32x4 v = src.ld4(beside < 0 ? ~15u : o * 16u, 0u);
            return {__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z)};
        }
    }
    // the lane's texels of row y
    __device__ __forceinline__ void save(void* dst, int pitch, int y, int W, const float4 (&o)[T]) const {
        if (!store) return;
        const uint32_t i = (uint32_t)y * (uint32_t)pitch + (uint32_t)x;
        if constexpr (S16) {
            const u32x4_a8 v = {pack_sat(o[0].x, o[0].y), pack_sat(o[0].z, o[0].w), pack_sat(o[1].x, o[1].y), pack_sat(o[1].z, o[1].w)};
            if (x + 1 < W) gstore<u32x4_a8>(dst, i * 8u, v);
            else gstore<uint2>(dst, i * 8u, make_uint2(v.x, v.y));
        } else {
            gstore<float4>(dst, i * 16u, o[0]);
        }
    }
};
__device__ __forceinline__ f3 rgb_of(uint2 t) { return {lo16(t.x), hi16(t.x), lo16(t.y)}; }
__device__ __forceinline__ f3 rgb_of(f3 t) { return t; }

// ------------------------------------------------------------------------------------------
// edge AA

struct EdgeAaArgs {
    const void* src;
    const uint32_t* mask;
    void* dst;
    int W, H, pitch, seg_pitch;
    float subpix, thr, thr_min;
    int tiles_x, tiles_y;
};

__device__ __forceinline__ float aa_luma(f3 c) { return c.x * 0.299f + c.y * 0.587f + c.z * 0.114f; }

template <bool S16, int R>
__global__ __launch_bounds__(256) void k_edge_aa(const EdgeAaArgs a) {
    typedef Rows<S16, R> G;
    constexpr int T = G::T;
    const int W = a.W, H = a.H;
    const G g(xcd_tile((int)blockIdx.x, a.tiles_x * a.tiles_y), a.tiles_x, W);
    if (g.y0 >= H) return;
    const Image src(a.src, a.pitch, W, H, S16 ? 8 : 16);
    typename G::Tex e[R + 2][T], eb[R + 2];
    uint32_t m[R][T];
#pragma unroll
    for (int r = 0; r < R + 2; ++r) {
        g.load(src, a.pitch, g.y0 - 1 + r, W, H, e[r]);
        eb[r] = g.load_beside(src, a.pitch, g.y0 - 1 + r, H);
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int j = 0; j < T; ++j)
            m[r][j] = gload<uint32_t>(a.mask, ((uint32_t)min(g.y0 + r, H - 1) * (uint32_t)a.seg_pitch + (uint32_t)clampi(g.x + j, 0, W - 1)) * 4u);
    float l[R + 2][T], lw[R + 2], le[R + 2];  // lumas of the lane's texels, and of those beside them
#pragma unroll
    for (int r = 0; r < R + 2; ++r) {
#pragma unroll
        for (int j = 0; j < T; ++j) l[r][j] = aa_luma(rgb_of(e[r][j]));
        const float lb = aa_luma(rgb_of(eb[r]));
        lw[r] = lane_before(l[r][T - 1], lb);
        le[r] = lane_after(l[r][0], lb);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int y = g.y0 + r;
        if (y >= H) break;
        bool edge[T], any = false;
#pragma unroll
        for (int j = 0; j < T; ++j) any |= edge[j] = (m[r][j] & 3u) == 1u;
        float4 out[T];
#pragma unroll
        for (int j = 0; j < T; ++j) {
            const f3 c = rgb_of(e[r + 1][j]);
            out[j] = make_float4(c.x, c.y, c.z, l[r + 1][j]);
        }
        if (__builtin_amdgcn_ballot_w64(any)) {
            const auto ew = lane_before(e[r + 1][T - 1], eb[r + 1]), ee = lane_after(e[r + 1][0], eb[r + 1]);
#pragma unroll
            for (int j = 0; j < T; ++j) {
                auto west = [&](int q) { return j > 0 ? l[q][j > 0 ? j - 1 : 0] : lw[q]; };
                auto east = [&](int q) { return j < T - 1 ? l[q][j < T - 1 ? j + 1 : 0] : le[q]; };
                const float lC = l[r + 1][j], lN = l[r][j], lS = l[r + 2][j], lW = west(r + 1), lE = east(r + 1);
                const float lNW = west(r), lNE = east(r), lSW = west(r + 2), lSE = east(r + 2);
                const float lmin = fminf(lC, fminf(fminf(lN, lS), fminf(lW, lE)));
                const float lmax = fmaxf(lC, fmaxf(fmaxf(lN, lS), fmaxf(lW, lE)));
                const float range = lmax - lmin;
                if (edge[j] && !(range < fmaxf(a.thr_min, lmax * a.thr))) {
                    const float gx = (lNE + 2.0f * lE + lSE) - (lNW + 2.0f * lW + lSW);
                    const float gy = (lSW + 2.0f * lS + lSE) - (lNW + 2.0f * lN + lNE);
                    const bool vertical = fabsf(gy) >= fabsf(gx);
                    const bool first = vertical ? fabsf(lN - lC) >= fabsf(lS - lC) : fabsf(lW - lC) >= fabsf(lE - lC);
                    const f3 n = rgb_of(e[r][j]), s = rgb_of(e[r + 2][j]);
                    const f3 w = rgb_of(j > 0 ? e[r + 1][j > 0 ? j - 1 : 0] : ew), o = rgb_of(j < T - 1 ? e[r + 1][j < T - 1 ? j + 1 : 0] : ee);
                    const float avg = (((lN + lS) + (lW + lE)) * 2.0f + ((lNW + lNE) + (lSW + lSE))) / 12.0f;
                    const float blend = a.subpix * 0.5f * gclamp(fabsf(avg - lC) / range, 0.0f, 1.0f);
                    auto mix = [&](float c, float cn, float cs, float cw, float ce) {
                        const float x = vertical ? (first ? cn : cs) : (first ? cw : ce);
                        return c * (1.0f - blend) + x * blend;
                    };
                    out[j] = make_float4(mix(out[j].x, n.x, s.x, w.x, o.x), mix(out[j].y, n.y, s.y, w.y, o.y), mix(out[j].z, n.z, s.z, w.z, o.z), lC);
                }
            }
        }
        g.save(a.dst, a.pitch, y, W, out);
    }
}

// ------------------------------------------------------------------------------------------
// CAS

struct CasArgs {
    const void* src;
    void* dst;
    int W, H, pitch;
    uint32_t peak_bits;
    int tiles_x, tiles_y;
};

template <bool S16, int R>
__global__ __launch_bounds__(256) void k_cas(const CasArgs a) {
    typedef Rows<S16, R> G;
    constexpr int T = G::T;
    const int W = a.W, H = a.H;
    const G g(xcd_tile((int)blockIdx.x, a.tiles_x * a.tiles_y), a.tiles_x, W);
    if (g.y0 >= H) return;
    const Image src(a.src, a.pitch, W, H, S16 ? 8 : 16);
    const float peak = __uint_as_float(a.peak_bits);
    typename G::Tex e[R + 2][T], eb[R];
#pragma unroll
    for (int r = 0; r < R + 2; ++r) g.load(src, a.pitch, g.y0 - 1 + r, W, H, e[r]);
#pragma unroll
    for (int r = 0; r < R; ++r) eb[r] = g.load_beside(src, a.pitch, g.y0 + r, H);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int y = g.y0 + r;
        if (y >= H) break;
        const auto ew = lane_before(e[r + 1][T - 1], eb[r]), ee = lane_after(e[r + 1][0], eb[r]);
        float4 out[T];
#pragma unroll
        for (int j = 0; j < T; ++j) {
            const f3 o = cas_filter(rgb_of(e[r][j]), rgb_of(j > 0 ? e[r + 1][j > 0 ? j - 1 : 0] : ew), rgb_of(e[r + 1][j]),
                                    rgb_of(j < T - 1 ? e[r + 1][j < T - 1 ? j + 1 : 0] : ee), rgb_of(e[r + 2][j]), peak);
            out[j] = make_float4(o.x, o.y, o.z, 1.0f);
        }
        g.save(a.dst, a.pitch, y, W, out);
    }
}

// f(R) with the tiling of a launch: four rows a wave, one where that leaves the device part empty (both passes, four rows and
// one, us: RGBA16F 960x540 (272 tiles) 11.2 and 10.3, 1280x720 (450) 12.5 and 10.9; 1600x900 (741) 16.2)
template <class A, class F>
void for_rows(A& a, int columns, F&& f) {
    a.tiles_x = tiles_for(a.W, columns);
    a.tiles_y = tiles_for(a.H, 16);
    if (a.tiles_x * a.tiles_y >= 512) return f(std::integral_constant<int, 4>());
    a.tiles_y = tiles_for(a.H, 4);
    f(std::integral_constant<int, 1>());
}

}  // namespace

int launch_edge_aa(const void* src, const uint32_t* mask, void* dst, int W, int H, int pitch, int seg_pitch, int fmt,
                   float subpix, float thr, float thr_min, void* stream) {
    const bool s16 = fmt == TAA_FMT_RGBA16F;
    EdgeAaArgs a{src, mask, dst, W, H, pitch, seg_pitch, subpix, thr, thr_min, 0, 0};
    hipStream_t st = static_cast<hipStream_t>(stream);
    for_rows(a, s16 ? 128 : 64, [&](auto r) {
        const dim3 g(a.tiles_x * a.tiles_y);
        if (s16) hipLaunchKernelGGL((k_edge_aa<true, decltype(r)::value>), g, dim3(256), 0, st, a);
        else hipLaunchKernelGGL((k_edge_aa<false, decltype(r)::value>), g, dim3(256), 0, st, a);
    });
    return (int)hipGetLastError();
}

int launch_cas(const void* src, void* dst, int W, int H, int pitch, int fmt, uint32_t peak_bits, void* stream) {
    const bool s16 = fmt == TAA_FMT_RGBA16F;
    CasArgs a{src, dst, W, H, pitch, peak_bits, 0, 0};
    hipStream_t st = static_cast<hipStream_t>(stream);
    for_rows(a, s16 ? 128 : 64, [&](auto r) {
        const dim3 g(a.tiles_x * a.tiles_y);
        if (s16) hipLaunchKernelGGL((k_cas<true, decltype(r)::value>), g, dim3(256), 0, st, a);
        else hipLaunchKernelGGL((k_cas<false, decltype(r)::value>), g, dim3(256), 0, st, a);
    });
    return (int)hipGetLastError();
}

}  // namespace taastar
