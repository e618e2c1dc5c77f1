// gfx950 exact FP32 resolve with the production feature set (variance box, clip, YCoCg, Catmull-Rom history,
// closest-depth RG velocity of the colour's precision, depth culling, Lottes, outside rejection; no debug or
// inspect image), operation for operation that of the general kernel (taa_kernels.hip).
//
// What bounds it: VALU issue (about 70% of the time at 1920x1080) and exposed latency. Against the general kernel's
// tiles: the 4x4 footprint filtered from an LDS window as in taa_window.hip (a thread gathered sixteen 16-byte texels, 256
// clocks of the CU's vector-memory path a wave); velocity staged; the closest-depth search by rows, which a thread's two
// rows of one column share; the linear-depth rejection and the clip without their divisions where these cannot matter
// (linear_depth_reject; |v| <= e), and one test of special values for six quotients by 9 and one for three square roots; 80 and
// 85 VGPRs instead of 94 and 107, so five or six workgroups a CU. The sums keep taa.comp's order (centre first), so the rows'
// sums cannot be shared as in the FP16 kernel.
// With the segmentation mask, whose kernel linearised eight depths and converted two angles' normals at 1.65 staged texels a
// texel, depth is linearised once a staged texel (with the other mask inputs at 1.46 a texel), the luma is the staged
// Y and the resolved texels lie over the staged ones, so five workgroups share a CU.
// us a frame, before and now: with the mask 1920x1080 FP32 storage with CAS 115 and 72.6, FP16 storage and arithmetic 82 and
// 53; without it FP32 storage with CAS 1920x1080 58.6 and 49.0, 3840x2160 208 and 203, without CAS 1920x1080
// 52.7 and 42.0, 3840x2160 200 and 168; FP16 storage with CAS 1920x1080 54.2 and 42.8, 3840x2160 186 and 169.
// The plain form (no closest-depth velocity, depth culling, Lottes weighting or outside rejection) ran the general kernel with its
// switches: FP32 storage 640x360 without CAS 10.5 and 7.8, 1920x1080 with CAS 77 and 44, FP16 storage 68 and 38.
// Measured and not kept: four rows a thread (1920x1080 with CAS 51.6, 3840x2160 211: four waves a SIMD), 512 threads of two
// rows (55.7, 235) or of one (54.6; footprints gathered without the window 65.8).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "taa_device.hpp"
#include "taa_fast_math.hpp"
#include "taa_internal.hpp"
#include "taa_production.hpp"
#include "taa_wave.hpp"

namespace taastar {
namespace {

// SEG: the frame also writes the segmentation mask; PLAIN: the texel's own velocity, no depth culling, Lottes weighting or
// outside rejection
template <bool CAS, bool S16, bool SEG_ = false, bool FA = false, bool PLAIN_ = false, int NT = 256, int RPT = 2>
struct ExactGeo : ProdGeo<NT, RPT, CAS, S16, FA> {
    typedef ProdGeo<NT, RPT, CAS, S16, FA> Base;
    static constexpr bool SEG = SEG_, PLAIN = PLAIN_;
    typedef typename Base::VelT VelT;
    static constexpr int RW = Base::RW, RH = Base::RH;
    // staged inputs: the region and one texel around it, two texels of a row a thread, SR rows a pass
    static constexpr int SW = RW + 2, SH = RH + 2, NS = SW * SH, SC = SW / 2, SR = NT / SC, SP = (SH + SR - 1) / SR;
    static constexpr int kStaged = PLAIN ? 0 : NS * (4 + (int)sizeof(VelT) + (SEG ? 20 : 0)),
                         kWin = Base::WIN ? Base::WP * Base::WH * (int)sizeof(typename Base::Win) : 16,
                         kRes = RW * RH * Base::TB, kMost = kStaged > kWin ? kStaged : kWin;
    struct Smem {
        alignas(16) unsigned char win[kMost > kRes ? kMost : kRes];  // velocity, depth and the mask's inputs, then the window, then the resolved texels
        alignas(16) float2 c01[NS];                                  // Y, Co
        alignas(8) float c2[NS];                                     // Cg
        float ux[SW], uy[SH];
        alignas(16) int4 box[NT / 64];
    };
};

template <class G>
__device__ __forceinline__ void resolve_exact(const FrameDesc& fd, const taa_uniforms_t& U, int tile, typename G::Smem& sm, const SegDesc* sg = nullptr) {
    typedef typename G::VelT VelT;
    constexpr bool S16 = G::S16, SEG = G::SEG, FA = G::FA;
    constexpr int RPT = G::RPT, SW = G::SW;
    const taa_params_t& P = U.param[fd.param_idx];
    const int W = fd.W, H = fd.H;
    const uint32_t pitch = (uint32_t)fd.pitch;
    const int ty = scalar(tile / fd.tiles_x), tx = tile - ty * fd.tiles_x;
    const int x0 = fd.x_begin + tx * G::TW - G::RA, y0 = ty * G::TH - G::RA;  // the region's first texel
    const int tid = (int)threadIdx.x, rx = tid & 31, rg = (tid >> 5) * RPT;
    const float gamma = scalar_now(P.mVarClipGamma), fW = (float)W, fH = (float)H;
    const Image color(fd.color, fd.pitch, W, H, G::TB), depths(fd.depth, fd.pitch, W, H, 4), velocity(fd.velocity, fd.pitch, W, H, (int)sizeof(VelT)),
        history(fd.history, fd.pitch, W, H, G::TB), hdepth(fd.hdepth, fd.pitch, W, H, 4);
    VelT* const sv = reinterpret_cast<VelT*>(sm.win);
    float* const sd = reinterpret_cast<float*>(sv + G::NS);
    // the mask's: linear depth, unit normal, material id (its luma is the staged Y)
    float *const sl = sd + G::NS, *const nx = sl + G::NS, *const ny = nx + G::NS, *const nz = ny + G::NS;
    uint32_t* const mat = reinterpret_cast<uint32_t*>(nz + G::NS);
    const uint32_t fl = SEG ? (uint32_t)scalar_now((int)P.mRayTraceAugmentFlags) : 0u, spl = SEG ? (uint32_t)sg->pitch_l : 0u;
    const float near = U.mCamNearPlane, far = U.mCamFarPlane;
    const Image materials(SEG ? (const void*)sg->material : nullptr, SEG ? sg->pitch_l : 1, SEG ? W : 1, SEG ? H : 1, 4),
        normals(SEG ? (const void*)sg->uv_normal : nullptr, SEG ? sg->pitch_l : 1, SEG ? W : 1, SEG ? H : 1, 16),
        prev_materials(SEG ? (const void*)sg->prev_material : nullptr, SEG ? sg->pitch_l : 1, SEG ? W : 1, SEG ? H : 1, 4);

    float2 own[G::PLAIN ? RPT : 1];  // the thread's texels' velocities
    if constexpr (G::PLAIN) {
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            const uint32_t i = (uint32_t)clampi(y0 + rg + k, 0, H - 1) * pitch + (uint32_t)clampi(x0 + rx, 0, W - 1);
            if constexpr (S16) {
                own[k] = vel_xy(velocity.ld1(i * 4u, 0u));
            } else {
                const uint2 v = velocity.ld2(i * 8u, 0u);
                own[k] = make_float2(__uint_as_float(v.x), __uint_as_float(v.y));
            }
        }
    }

    // ---- 1. stage colour, depth and velocity of the region and one texel around it, clamped to the edge
    {
        auto store = [&](int i, f3 a, f3 b, uint2 d, VelT v0, VelT v1) {
            a = rgb_to_ycocg(a), b = rgb_to_ycocg(b);
            *reinterpret_cast<float4*>(sm.c01 + i) = make_float4(a.x, a.y, b.x, b.y);
            *reinterpret_cast<float2*>(sm.c2 + i) = make_float2(a.z, b.z);
            if constexpr (G::PLAIN) return;
            *reinterpret_cast<uint2*>(sd + i) = d;
            sv[i] = v0;
            sv[i + 1] = v1;
        };
        // a pair's mask inputs: material ids, normal angles (taa.comp:570-579)
        auto store_mask = [&](int i, uint2 d, uint2 m, uint2 a, uint2 b) {
            if (fl & TAA_RTFLAG_DPT) *reinterpret_cast<float2*>(sl + i) = make_float2(linearize_depth(__uint_as_float(d.x), near, far), linearize_depth(__uint_as_float(d.y), near, far));
            *reinterpret_cast<uint2*>(mat + i) = m;
            if (fl & TAA_RTFLAG_NRM) {
                auto normal = [](uint2 q) {
                    float sz, cz, sw, cw;
                    seg_sincos(__uint_as_float(q.x), sz, cz);
                    seg_sincos(__uint_as_float(q.y), sw, cw);
                    return f3{cz * cw, sz * cw, sw};
                };
                const f3 p = normal(a), q = normal(b);
                *reinterpret_cast<float2*>(nx + i) = make_float2(p.x, q.x);
                *reinterpret_cast<float2*>(ny + i) = make_float2(p.y, q.y);
                *reinterpret_cast<float2*>(nz + i) = make_float2(p.z, q.z);
            }
        };
        auto rgb16 = [](uint32_t a, uint32_t b) { return f3{lo16(a), hi16(a), lo16(b)}; };
        auto rgb32 = [](u32x4 t) { return f3{__uint_as_float(t.x), __uint_as_float(t.y), __uint_as_float(t.z)}; };
        auto vel32 = [](uint32_t a, uint32_t b) { return make_float2(__uint_as_float(a), __uint_as_float(b)); };
        auto tables = [&] {  // uv of the columns and rows (taa.comp:131), while the loads are under way
            if (tid < G::SW) sm.ux[tid] = ((float)clampi(x0 - 1 + tid, 0, W - 1) + 0.5f) / fW;
            else if (tid >= 64 && tid < 64 + G::SH) sm.uy[tid - 64] = ((float)clampi(y0 - 1 + tid - 64, 0, H - 1) + 0.5f) / fH;
        };
        const int sy = tid / G::SC, sx = 2 * (tid - sy * G::SC);
        const bool inside = x0 >= 1 && y0 >= 1 && x0 + G::RW + 1 <= W && y0 + G::RH + 1 <= H;
        constexpr int kPass = G::SC * G::SR * 2;
        if (inside) {  // the pass in the scalar offset
            const uint32_t o = (uint32_t)sy * pitch + (uint32_t)sx;
            u32x4 c[G::SP * (S16 ? 1 : 2)], v32[S16 ? 1 : G::SP];
            uint2 d[G::SP], v16[G::SP], m[SEG ? G::SP : 1], na[SEG ? G::SP : 1], nb[SEG ? G::SP : 1];
            const uint32_t om = (uint32_t)sy * spl + (uint32_t)sx;
#pragma unroll
            for (int p = 0; p < G::SP; ++p) {  // (an offset past the image reads nothing: no load in a branch)
                const bool have = tid < G::SC * G::SR && sy + p * G::SR < G::SH;
                const uint32_t s = (uint32_t)(y0 - 1 + p * G::SR) * pitch + (uint32_t)(x0 - 1);
                if constexpr (S16) {
                    c[p] = color.ld4(have ? o * 8u : ~15u, s * 8u);
                    v16[p] = velocity.ld2(have ? o * 4u : ~15u, s * 4u);
                } else {
                    c[2 * p] = color.ld4(have ? o * 16u : ~15u, s * 16u);
                    c[2 * p + 1] = color.ld4(have ? o * 16u + 16u : ~15u, s * 16u);
                    v32[p] = velocity.ld4(have ? o * 8u : ~15u, s * 8u);
                }
                d[p] = depths.ld2(have ? o * 4u : ~15u, s * 4u);
                if constexpr (SEG) {
                    const uint32_t t = (uint32_t)(y0 - 1 + p * G::SR) * spl + (uint32_t)(x0 - 1);
                    m[p] = materials.ld2(have ? om * 4u : ~15u, t * 4u);
                    na[p] = normals.ld2(have ? om * 16u + 8u : ~15u, t * 16u);
                    nb[p] = normals.ld2(have ? om * 16u + 24u : ~15u, t * 16u);
                }
            }
            tables();
#pragma unroll
            for (int p = 0; p < G::SP; ++p) {
                if (tid >= G::SC * G::SR || sy + p * G::SR >= G::SH) break;
                const int i = 2 * tid + p * kPass;
                if constexpr (S16) store(i, rgb16(c[p].x, c[p].y), rgb16(c[p].z, c[p].w), d[p], v16[p].x, v16[p].y);
                else store(i, rgb32(c[2 * p]), rgb32(c[2 * p + 1]), d[p], vel32(v32[p].x, v32[p].y), vel32(v32[p].z, v32[p].w));
                if constexpr (SEG) store_mask(i, d[p], m[p], na[p], nb[p]);
            }
        } else {  // a tile over the image's border: texel by texel, clamped
            tables();
#pragma unroll 1
            for (int p = 0; p < G::SP; ++p) {
                if (tid >= G::SC * G::SR || sy + p * G::SR >= G::SH) break;
                const uint32_t r = (uint32_t)clampi(y0 - 1 + sy + p * G::SR, 0, H - 1) * pitch;
                const uint32_t g0 = r + (uint32_t)clampi(x0 - 1 + sx, 0, W - 1), g1 = r + (uint32_t)clampi(x0 + sx, 0, W - 1);
                const uint2 d = make_uint2(depths.ld1(g0 * 4u, 0u), depths.ld1(g1 * 4u, 0u));
                if constexpr (SEG) {
                    const uint32_t rm = (uint32_t)clampi(y0 - 1 + sy + p * G::SR, 0, H - 1) * spl;
                    const uint32_t m0 = rm + (uint32_t)clampi(x0 - 1 + sx, 0, W - 1), m1 = rm + (uint32_t)clampi(x0 + sx, 0, W - 1);
                    store_mask(2 * tid + p * kPass, d, make_uint2(materials.ld1(m0 * 4u, 0u), materials.ld1(m1 * 4u, 0u)),
                               normals.ld2(m0 * 16u + 8u, 0u), normals.ld2(m1 * 16u + 8u, 0u));
                }
                if constexpr (S16) {
                    const uint2 a = color.ld2(g0 * 8u, 0u), b = color.ld2(g1 * 8u, 0u);
                    store(2 * tid + p * kPass, rgb16(a.x, a.y), rgb16(b.x, b.y), d, velocity.ld1(g0 * 4u, 0u), velocity.ld1(g1 * 4u, 0u));
                } else {
                    const uint2 a = velocity.ld2(g0 * 8u, 0u), b = velocity.ld2(g1 * 8u, 0u);
                    store(2 * tid + p * kPass, rgb32(color.ld4(g0 * 16u, 0u)), rgb32(color.ld4(g1 * 16u, 0u)), d, vel32(a.x, a.y), vel32(b.x, b.y));
                }
            }
        }
        __syncthreads();
    }

    // ---- 2. closest depth, history position and previous depth of the thread's texels
    ProdTexel q[RPT];
    int4 bases = make_int4(0x7fffffff, 0x7fffffff, 0x7fffffff, 0x7fffffff);
    if constexpr (G::PLAIN) {  // SAMPLE_TEX(uCurrentVelocity, uv) (taa.comp:421)
        const float uvx = sm.ux[rx + 1];
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            const float2 v = own[k];
            q[k].expected = q[k].pd = 0.0f;
            q[k].hu = uvx - v.x;
            q[k].hv = sm.uy[rg + k + 1] - v.y;
            q[k].masked = false;
            history_base<FA>(q[k], W, H, bases);
        }
    } else {
        const int base = rg * SW + rx;
        struct Row {
            float d, cd;  // the first smallest depth of the row's three in scan order (strict <), the centre's
            int i;        // its position
        };
        float sum = 0.0f;
        auto read_row = [&](int t) {
            const int i = base + t * SW;
            const float dl = sd[i], dc = sd[i + 1], dr = sd[i + 2];
            const bool c1 = dc < dl;
            const float d1 = c1 ? dc : dl;
            const bool c2 = dr < d1;
            sum += (dl + dc) + dr;
            return Row{c2 ? dr : d1, dc, i + (c2 ? 2 : c1 ? 1 : 0)};
        };
        const float uvx = sm.ux[rx + 1];
        Row ra = read_row(0), rb = read_row(1);
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            const float uvy = sm.uy[rg + k + 1];
            const Row rc = read_row(k + 2);
            // findClosestUvAndZ_3x3 (taa.comp:371-389): the rows' minima in scan order, strict <
            const bool c1 = rb.d < ra.d;
            const float d1 = c1 ? rb.d : ra.d;
            int best = rc.d < d1 ? rc.i : c1 ? rb.i : ra.i;
            if (!(sum == sum)) {  // a NaN among the depths read so far: the scan itself, in which only a NaN first tap stays
                best = base + k * SW;
                float d = sd[best];
#pragma unroll 1
                for (int j = 1; j < 9; ++j) {
                    const int i = base + (k + j / 3) * SW + j % 3;
                    const float e = sd[i];
                    if (e < d) d = e, best = i;
                }
            }
            const float2 v = vel_xy(sv[best]);
            q[k].expected = rb.cd;
            q[k].hu = uvx - v.x;
            q[k].hv = uvy - v.y;
            // the previous depth under the history position (taa.comp:818)
            const int dx = med3<0>(to_int(q[k].hu * fW), W - 1), dy = med3<0>(to_int(q[k].hv * fH), H - 1);
            q[k].pd = __uint_as_float(hdepth.ld1(((uint32_t)dy * pitch + (uint32_t)dx) * 4u, 0u));
            q[k].masked = false;
            history_base<FA>(q[k], W, H, bases);
            ra = rb, rb = rc;
        }
    }
    // ---- 3. segmentation mask (calc_segmentation_value, taa.comp:589-702): the tests in reverse, so that the first that holds stays
    if constexpr (SEG) {
        uint32_t prev[RPT], old[RPT];
        bool inside[RPT];
        const bool own_col = x0 + rx < fd.x_end && (!G::CAS || (rx >= 1 && rx < 31));
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            prev[k] = old[k] = 0u;
            inside[k] = own_col && (k > 0 || !G::CAS || rg > 0) && (k < RPT - 1 || !G::CAS || rg < G::RH - RPT) && y0 + rg + k < H;
            const int x = clampi(x0 + rx, 0, W - 1), y = clampi(y0 + rg + k, 0, H - 1);
            if (fl & TAA_RTFLAG_DIS) {  // the previous material under the history position; 0 outside the image
                const int tx = to_int(q[k].hu * fW), ty = to_int(q[k].hv * fH);
                prev[k] = prev_materials.ld1(tx >= 0 && ty >= 0 && tx < W && ty < H ? ((uint32_t)ty * spl + (uint32_t)tx) * 4u : ~15u, 0u);
            }
            if (fl & TAA_RTFLAG_CNT) old[k] = gload<uint32_t>(sg->prev_segmask, ((uint32_t)y * (uint32_t)sg->pitch + (uint32_t)x) * 4u) >> 16;
        }
        const uint32_t count = fl & TAA_RTFLAG_CNT ? (uint32_t)P.mRayTraceHistoryCount << 16 : 0u;
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            const int l = (rg + k + 1) * SW + rx + 1;
            float nrm = 0.0f, dpt = 0.0f, matv = 0.0f, lum = 0.0f;
            // sobel (taa.comp:582-587) and length() over the eight neighbours
            auto sobel = [&](auto&& at) {
                const float t0 = at(-SW - 1), t1 = at(-SW), t2 = at(-SW + 1), t3 = at(-1), t4 = at(1), t5 = at(SW - 1), t6 = at(SW), t7 = at(SW + 1);
                const float gx = t0 - t5 + 2.0f * t1 - 2.0f * t6 + t2 - t7;
                const float gy = t0 - t2 + 2.0f * t3 - 2.0f * t4 + t5 - t7;
                return sqrtf(gx * gx + gy * gy);
            };
            if (fl & TAA_RTFLAG_NRM) {
                const f3 c = {nx[l], ny[l], nz[l]};
                auto dn = [&](int o) { return c.x * nx[l + o] + c.y * ny[l + o] + c.z * nz[l + o]; };
                nrm = 1.0f - fmaxf(0.0f, fminf(fminf(fminf(dn(-1), dn(1)), dn(-SW)), dn(SW)));
            }
            if (fl & TAA_RTFLAG_DPT) dpt = sobel([&](int o) { return sl[l + o]; });
            const uint32_t id = mat[l];
            if ((fl & TAA_RTFLAG_MID) && (id != mat[l - 1] || id != mat[l + 1] || id != mat[l - SW] || id != mat[l + SW])) matv = 1.0f;
            if (fl & TAA_RTFLAG_LUM) lum = sobel([&](int o) { return sm.c01[l + o].x; });
            const float total = nrm * P.mRayTraceAugment_WNrm + dpt * P.mRayTraceAugment_WDpt + matv * P.mRayTraceAugment_WMId + lum * P.mRayTraceAugment_WLum;
            uint32_t v = old[k] > 0u ? 2u | ((old[k] - 1u) << 16) : 0u;
            if (total >= P.mRayTraceAugment_Thresh) v = 2u | count;
            if (prev[k] != id && (prev[k] & 0x80000000u) != 0u) v = 2u | count;
            if ((fl & TAA_RTFLAG_OUT) && (q[k].hu < 0.0f || q[k].hv < 0.0f || q[k].hu >= 1.0f || q[k].hv >= 1.0f)) v = 1u;
            if (fl & TAA_RTFLAG_ALL) v = 2u;
            const int x = x0 + rx, y = y0 + rg + k;
            if ((fl & TAA_RTFLAG_FXD) && (x < 100 || y < 100 || x >= W - 100 || y >= H - 100)) v = 1u;
            q[k].masked = (v & 3u) != 0u;
            if (inside[k]) gstore<uint32_t>(sg->segmask, ((uint32_t)y * (uint32_t)sg->pitch + (uint32_t)x) * 4u, v);
        }
    }
    // ---- 4. box and current colour of texel k (called for k = 0, 1, ... in turn): its 3x3 texels, the upper six from the call before
    f3 n[9];
    auto read3 = [&](int t, int j) {
        const int i = (rg + t) * SW + rx;
#pragma unroll
        for (int x = 0; x < 3; ++x) n[j + x] = {sm.c01[i + x].x, sm.c01[i + x].y, sm.c2[i + x]};
    };
    auto box = [&](int k, f3& c, f3& e, f3& cur, bool& found) {
        if (k == 0) read3(0, 0), read3(1, 3);
        read3(k + 2, 6);
        cur = n[4];
        found = true;
        // centre, then the others in scan order (taa.comp:199-213, 272-281)
        if constexpr (FA) {
            const int order[8] = {0, 1, 2, 3, 5, 6, 7, 8};
            f3 m1 = n[4], m2 = n[4] * n[4];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const f3 t = n[order[j]];
                m1 = m1 + t;
                m2 = {__builtin_fmaf(t.x, t.x, m2.x), __builtin_fmaf(t.y, t.y, m2.y), __builtin_fmaf(t.z, t.z, m2.z)};
            }
            fast_box(m1, m2, gamma, c, e);
#pragma unroll
            for (int j = 0; j < 6; ++j) n[j] = n[j + 3];
            return;
        }
        f3 m1 = n[4] + n[0] + n[1] + n[2] + n[3] + n[5] + n[6] + n[7] + n[8];
        f3 m2 = n[4] * n[4] + n[0] * n[0] + n[1] * n[1] + n[2] * n[2] + n[3] * n[3] + n[5] * n[5] + n[6] * n[6] + n[7] * n[7] + n[8] * n[8];
        div9_moments(m1, m2);
        const f3 mean = m1, var = m2 - mean * mean;
        const f3 sigma = sqrt3({fmaxf(0.0f, var.x), fmaxf(0.0f, var.y), fmaxf(0.0f, var.z)});
        const f3 mn = mean - gamma * sigma, mx = mean + gamma * sigma;
        c = 0.5f * (mx + mn);  // clipAabb's centre and half size (taa.comp:326-327)
        e = 0.5f * (mx - mn) + f3{1e-7f, 1e-7f, 1e-7f};
#pragma unroll
        for (int j = 0; j < 6; ++j) n[j] = n[j + 3];
    };
    finish<G>(fd, U, P, history, x0, y0, q, bases, sm.win, sm.box, box);
}

struct ResolveArgs {
    FrameDesc fd;
    taa_uniforms_t U;
};

// occupancy hint (waves per SIMD): what the LDS of the tile allows
template <class G>
constexpr int exact_waves() {
    return G::RPT == 1 ? 4 : G::S16 ? 6 : 5;
}

template <class G>
__global__ __launch_bounds__(G::NT) __attribute__((amdgpu_waves_per_eu(exact_waves<G>()))) void k_resolve_exact(const ResolveArgs a) {
    __shared__ typename G::Smem sm;
    resolve_exact<G>(a.fd, a.U, xcd_tile((int)blockIdx.x, a.fd.tiles_x * a.fd.tiles_y), sm);
}

// the frames of a batch, walked like the other batched kernels
template <class G>
__global__ __launch_bounds__(G::NT) __attribute__((amdgpu_waves_per_eu(exact_waves<G>()))) void k_resolve_exact_batch(const BatchEntry* __restrict__ entries, int n_entries, int total) {
    __shared__ typename G::Smem sm;
    const int t = batch_tile(total);
    if (t < 0) return;
    const BatchEntry& e = batch_entry(entries, n_entries, t);
    resolve_exact<G>(e.fd, e.U, t - e.tile_begin, sm);
}

// f(geometry) for a frame's form
template <bool PLAIN, int NT, int RPT, class F>
void for_form(bool cas, bool s16, F&& f) {
    if (cas) s16 ? f(ExactGeo<true, true, false, false, PLAIN, NT, RPT>()) : f(ExactGeo<true, false, false, false, PLAIN, NT, RPT>());
    else s16 ? f(ExactGeo<false, true, false, false, PLAIN, NT, RPT>()) : f(ExactGeo<false, false, false, false, PLAIN, NT, RPT>());
}

// the resolve with the segmentation mask of mRayTraceAugment (FA: the FP16 path's arithmetic where no selection depends on it)
template <bool CAS, bool S16, bool FA>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) void k_resolve_mask(const ResolveArgs a, const SegDesc sg) {
    using G = ExactGeo<CAS, S16, true, FA>;
    __shared__ typename G::Smem sm;
    resolve_exact<G>(a.fd, a.U, xcd_tile((int)blockIdx.x, a.fd.tiles_x * a.fd.tiles_y), sm, &sg);
}

template <bool FA>
void launch_mask_t(const ResolveArgs& a, const SegDesc& sg, hipStream_t st) {
    const dim3 g(a.fd.tiles_x * a.fd.tiles_y);
    const bool s16 = a.fd.color_fmt == TAA_FMT_RGBA16F;
    if (a.fd.cas_on) {
        if (s16) hipLaunchKernelGGL((k_resolve_mask<true, true, FA>), g, dim3(256), 0, st, a, sg);
        else hipLaunchKernelGGL((k_resolve_mask<true, false, FA>), g, dim3(256), 0, st, a, sg);
    } else {
        if (s16) hipLaunchKernelGGL((k_resolve_mask<false, true, FA>), g, dim3(256), 0, st, a, sg);
        else hipLaunchKernelGGL((k_resolve_mask<false, false, FA>), g, dim3(256), 0, st, a, sg);
    }
}

}  // namespace

bool mask_form(const FrameDesc& fd, const taa_uniforms_t& U) {
    FrameDesc p = fd;
    tile_production(p, kProd256x2);
    return !fd.up && (long long)p.tiles_x * p.tiles_y >= 700 && prod_params(fd, U, true);
}

int launch_mask(const FrameDesc& fd, const taa_uniforms_t& U, const SegDesc& sg, int arith, void* stream) {
    hipStream_t st = static_cast<hipStream_t>(stream);
    ResolveArgs a;
    a.fd = fd;
    a.U = U;
    tile_production(a.fd, kProd256x2);
    if (arith == TAA_ARITH_FP16) launch_mask_t<true>(a, sg, st);
    else launch_mask_t<false>(a, sg, st);
    return (int)hipGetLastError();
}

int launch_exact(const FrameDesc& fd, const taa_uniforms_t& U, bool plain, void* stream) {
    hipStream_t st = static_cast<hipStream_t>(stream);
    ResolveArgs a;
    a.fd = fd;
    a.U = U;
    const bool cas = fd.cas_on != 0, s16 = fd.color_fmt == TAA_FMT_RGBA16F;
    auto launch = [&](auto g) {
        hipLaunchKernelGGL((k_resolve_exact<decltype(g)>), dim3(fd.tiles_x * fd.tiles_y), dim3(decltype(g)::NT), 0, st, a);
    };
    if (!plain) for_form<false, 256, 2>(cas, s16, launch);
    else if (fd.rows != kProd512x1) for_form<true, 256, 2>(cas, s16, launch);
    else if (s16) launch(ExactGeo<false, true, false, false, true, 512, 1>());  // (chosen without CAS only)
    else launch(ExactGeo<false, false, false, false, true, 512, 1>());
    return (int)hipGetLastError();
}

int launch_exact_batch(const BatchEntry* e, int n, int total, bool plain, bool cas, bool s16, void* stream) {
    hipStream_t st = static_cast<hipStream_t>(stream);
    auto launch = [&](auto g) {
        hipLaunchKernelGGL((k_resolve_exact_batch<decltype(g)>), dim3(batch_grid(total)), dim3(256), 0, st, e, n, total);
    };
    if (plain) for_form<true, 256, 2>(cas, s16, launch);
    else for_form<false, 256, 2>(cas, s16, launch);
    return (int)hipGetLastError();
}

}  // namespace taastar
