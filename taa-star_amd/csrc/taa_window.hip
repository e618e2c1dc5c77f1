// gfx950 throughput kernel of the temporal resolve on FP16 storage (TAA_ARITH_FP16, RGBA16F), and the
// reference's default block in the exact arithmetic on that storage.
//
// Arithmetic: texels stay fp16 and enter the history filter through mixed fp16 x fp32 FMAs; moments,
// rectification and the blend run in fp32 with contraction and the hardware reciprocal / square root.
// Everything that selects a texel or rejects one -- the closest-depth tap, historyUv = uv - v, the
// filter's base texel, the depth-test texel, the out-of-screen and depth decisions -- is computed exactly
// as in the FP32 path.
//
// What bounds it: the vector-memory path, exposed latency and VALU issue together. A vector load of 8 or
// 16 bytes a lane costs a CU 16 clocks whatever it hits; gathering every texel's 4x4 footprint takes
// eight of them a wave, against 4.5-5 clocks for an LDS read. So a workgroup first finds the positions of all its
// texels (1, 2), then loads the rectangle their footprints cover into LDS once, two texels a lane (3), and
// filters from there (4): the L1's busy time at 4K falls from 168,000 to 106,000 clocks. A tile whose
// footprints lie too far apart for the window (48 columns, the region's height + 16 rows) reads them from memory; a scene in which
// neighbouring objects move 24 texels apart everywhere runs 149 us a 4K frame so, 12 more than the tile kernel that held footprints in registers.
// A thread owns consecutive rows of one column, so the 3x3 sums and the closest-depth search share its rows
// (a row's three texels are summed and compared once, not three times), the CAS takes its upper and
// lower neighbours from registers, and row offsets are scalar: 1,440 VALU instructions a wave of 4 x 64 texels against
// 1,770 on the tile kernel this replaced. Staging is two texels a lane too; the window and the resolved texels lie over
// LDS that earlier phases are done with, so five workgroups of 32 x 32 texels share a CU.
// 3840x2160 with CAS: 106.5 us a frame (365 MB of images, 411 MB of HBM traffic) against 125.6 before (378 MB), five
// waves per SIMD either way; twelve sessions in one batch 361 against 425 us; the reference's default block at
// 2560x1440 43.3 against 70.5 us (its switches fixed, bilinear footprints gathered directly), and that block in the exact
// arithmetic, which differs in the bilinear weights, the blend and the CAS, 25.3 against 55.3 us at 1920x1080.
// Measured and not kept: strips of rows marched by one wave, neighbours by lane shifts and no LDS (4K 141 us: rows
// shared by two strips come from beyond the L2 twice, four waves per SIMD leave the loads exposed); 512 threads of
// two rows (4K 115); tiles walked in column order over 2, 3, 4 or 9 tile rows (no gain).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "taa_device.hpp"
#include "taa_fast_math.hpp"
#include "taa_internal.hpp"
#include "taa_wave.hpp"

namespace taastar {
namespace {

// FORM (WindowForm): kProd and kDefault are the production feature set and the reference's default
// block with every switch fixed, kVar the variance box with Catmull-Rom history, kGeneral either box
// and history, kExt and kExtRgba the per-texel options on RG and RGBA velocity, kDefaultExact the default block in
// the exact FP32 arithmetic.
template <int NT_, int RPT_, bool CAS_, bool INSP_, int FORM_>
struct WinGeo {
    static constexpr bool CAS = CAS_, INSP = INSP_;
    static constexpr int FORM = FORM_;
    static constexpr bool EX = FORM == kDefaultExact;  // exact FP32 arithmetic (taa.comp's operations, no inspect image)
    static constexpr bool PROD = FORM == kProd, DEF = FORM == kDefault || EX;
    static constexpr bool EXT = FORM >= kExt, V4 = FORM >= kExtRgba;
    static constexpr int VAR = FORM <= kVar ? 1 : DEF ? 0 : kAny;     // variance box, else minimum / maximum
    static constexpr int CR = FORM <= kVar ? 1 : DEF ? 0 : kAny;      // Catmull-Rom history, else bilinear
    static constexpr int YCOCG = PROD ? 1 : DEF ? 0 : kAny, CLOSEST = YCOCG, CULL = YCOCG, LOTTES = YCOCG, OUTSIDE = YCOCG;
    static constexpr int RECT = PROD ? 2 : DEF ? 1 : kAny;            // clip, clamp
    static constexpr int OPTIONS = DEF ? 0 : EXT ? kAny : 0;          // anti-ghosting, velocity alpha, near-clamp, debug image
    typedef typename std::conditional<V4, uint2, uint32_t>::type VelT;
    typedef typename std::conditional<V4, uint4, uint2>::type DepthVel;  // staged: depth bits, velocity bits
    // A workgroup of NT threads resolves a region of 32 columns x RH rows, RPT rows of one column a thread; with
    // fused CAS its outermost ring belongs to the neighbouring tiles.
    static constexpr int NT = NT_, RPT = RPT_, RW = 32, RH = NT / 32 * RPT, RA = CAS ? 1 : 0, TW = RW - 2 * RA, TH = RH - 2 * RA;
    // staged inputs: the region and one texel around it, two texels of a row a thread, SR rows a pass
    static constexpr int SW = RW + 2, SH = RH + 2, NS = SW * SH, SC = SW / 2, SR = NT / SC, SP = (SH + SR - 1) / SR;
    // RPT 1, for frames that leave the device part empty, and bilinear history have no window: a texel's footprint is read
    // from memory as soon as its position is known, which saves two barriers and a round trip
    static constexpr bool WIN = RPT > 1 && CR != 0;
    static constexpr int FN = CR == 0 ? 2 : 4;  // rows and columns of a footprint
    // history window: rows of WP texels, two of them a thread, WR rows a pass
    static constexpr int WP = 48, WC = WP / 2, WR = NT / WC, WN = (RH + 3 + WR - 1) / WR;
    static constexpr int WH = RH + 16;  // rows it holds
    static constexpr int kDv = NS * (int)sizeof(DepthVel), kWin = WIN ? WP * WH * 8 : 0;
    struct Smem {
        alignas(16) unsigned char win[kWin > kDv ? kWin : kDv];  // depth and velocity until the window replaces them
        alignas(16) float2 c01[NS];                              // Y, Co; in the end the resolved texels for the fused CAS
        alignas(8) float c2[NS];                                 // Cg
        uint2 own[WIN || !CAS ? 1 : RW * RH];  // without the window LDS is no limit: a place of their own saves a barrier
        __device__ uint2* res() { return WIN ? reinterpret_cast<uint2*>(c01) : own; }
        float ux[SW], uy[SH];
        alignas(16) int4 box[NT / 64];
    };
};

__device__ __forceinline__ float2 vel_xy(uint32_t v) { return make_float2(lo16(v), hi16(v)); }
__device__ __forceinline__ float2 vel_xy(uint2 v) { return make_float2(lo16(v.x), hi16(v.x)); }
__device__ __forceinline__ float4 vel_xyzw(uint32_t v) { return make_float4(lo16(v), hi16(v), 0.0f, 1.0f); }
__device__ __forceinline__ float4 vel_xyzw(uint2 v) { return make_float4(lo16(v.x), hi16(v.x), lo16(v.y), hi16(v.y)); }

// a resolve texel between its history position and its blend
struct Texel0 {
    float fx, fy, expected, pd, hu, hv;
    int k;  // its footprint's first texel in the window
    int kx, ky, ix, iy, dtx, dty, closest;
    bool outside, used_velocity, moved, calm;
};

template <class G>
__device__ __forceinline__ void resolve_window(const FrameDesc& fd, const taa_uniforms_t& U, int tile, typename G::Smem& sm) {
    typedef typename G::VelT VelT;
    typedef typename G::DepthVel DepthVel;
    constexpr bool EXT = G::EXT, INSP = G::INSP;
    constexpr int RPT = G::RPT, SW = G::SW;
    const taa_params_t& P = U.param[fd.param_idx];
    const int W = fd.W, H = fd.H;
    const uint32_t pitch = (uint32_t)fd.pitch;
    const int ty = scalar(tile / fd.tiles_x), tx = tile - ty * fd.tiles_x;
    const int x0 = fd.x_begin + tx * G::TW - G::RA, y0 = ty * G::TH - G::RA;  // the region's first texel
    const int tid = (int)threadIdx.x, rx = tid & 31, rg = (tid >> 5) * RPT;

    // parameters read here, ahead of their phases; one row a thread (all workgroups start at once) has its first loads under way sooner
    // without waiting for them
    auto pin = [](auto v) {
        if constexpr (G::RPT > 1) return scalar_now(v);
        else return v;
    };
    auto pinned_flag = [&](int v) { return pin(v) != 0; };
    const int sample_mode = G::CLOSEST == kAny ? pin(P.mVelocitySampleMode) : G::CLOSEST * 2;
    const bool ycocg = opt(G::YCOCG, pinned_flag(P.mUseYCoCg));
    const bool closest_mode = sample_mode == 2;
    const int rect = G::RECT == kAny ? pin(P.mColorClampingOrClipping) : G::RECT;
    const bool lottes = opt(G::LOTTES, pinned_flag(P.mLumaWeightingLottes));
    const bool reject_out = opt(G::OUTSIDE, pinned_flag(P.mRejectOutside));
    const bool depth_cull = opt(G::CULL, pinned_flag(P.mDepthCulling));
    const bool reset = pinned_flag(U.mResetHistory);
    const bool var_clip = opt(G::VAR, pinned_flag(P.mVarianceClipping));
    const bool cr_hist = G::CR == kAny ? pin(P.mInterpolationMode) == 2 : G::CR != 0;
    const bool ghost = opt(G::OPTIONS, pinned_flag(P.mDynamicAntiGhosting));
    const bool vel_alpha = opt(G::OPTIONS, pinned_flag(P.mVelBasedAlpha)), near_clamp = opt(G::OPTIONS, pinned_flag(P.mReduceBlendNearClamp));
    const bool longest = EXT && sample_mode == 1;
    const int use_velocity = G::DEF ? 1 : EXT ? pin(P.mUseVelocityVectors) : 2;
    const float gamma = pin(P.mVarClipGamma), a_plain = pin(P.mAlpha), a_max = pin(P.mMaxAlpha),
                a_min = pin(P.mMinAlpha), a_reject = pin(P.mRejectionAlpha), peak = pin(__uint_as_float(fd.cas_peak_bits));
    const float near = pin(U.mCamNearPlane), far = pin(U.mCamFarPlane), lin_thr = pin(U.pad1);
    const bool lin_depth = lin_thr > 0.0f;
    const float fW = (float)W, fH = (float)H;
    const Image color(fd.color, fd.pitch, W, H, 8), depths(fd.depth, fd.pitch, W, H, 4), velocity(fd.velocity, fd.pitch, W, H, (int)sizeof(VelT)),
        history(fd.history, fd.pitch, W, H, 8), hdepth(fd.hdepth, fd.pitch, W, H, 4);
    // the outputs from one row above their first, so that the region's row -1 (a tile's ring, never written) has an offset too
    const size_t row_bytes = (size_t)pitch * 8u;
    const Image history_out((const char*)fd.history_out - row_bytes, fd.pitch, W, H + 1, 8), screen((const char*)fd.screen - row_bytes, fd.pitch, W, H + 1, 8);
    const uint32_t out_off = ((uint32_t)(y0 + 1 + rg) * pitch + (uint32_t)(x0 + rx)) * 8u;
    DepthVel* const dv = reinterpret_cast<DepthVel*>(sm.win);
    uint2* const win = reinterpret_cast<uint2*>(sm.win);

    // ---- 1. stage depth, velocity and colour of the region and one texel around it, clamped to the edge
    {
        auto store = [&](int i, uint2 c0, uint2 c1, uint2 d, const VelT& v0, const VelT& v1) {
            auto convert = [&](uint2 c) -> f3 {
                const f3 q = {lo16(c.x), hi16(c.x), lo16(c.y)};
                if (!ycocg) return q;
                const float t = 0.25f * (q.x + q.z);
                return {__builtin_fmaf(0.5f, q.y, t), 0.5f * (q.x - q.z), __builtin_fmaf(0.5f, q.y, -t)};
            };
            const f3 a = convert(c0), b = convert(c1);
            *reinterpret_cast<float4*>(sm.c01 + i) = make_float4(a.x, a.y, b.x, b.y);
            *reinterpret_cast<float2*>(sm.c2 + i) = make_float2(a.z, b.z);
            if constexpr (G::V4) {
                dv[i] = make_uint4(d.x, v0.x, v0.y, 0u);
                dv[i + 1] = make_uint4(d.y, v1.x, v1.y, 0u);
            } else {
                *reinterpret_cast<uint4*>(dv + i) = make_uint4(d.x, v0, d.y, v1);
            }
        };
        auto tables = [&] {  // uv of the columns and rows (taa.comp:131), while the loads are under way
            if (tid < G::SW) sm.ux[tid] = ((float)clampi(x0 - 1 + tid, 0, W - 1) + 0.5f) / fW;
            else if (tid >= 64 && tid < 64 + G::SH) sm.uy[tid - 64] = ((float)clampi(y0 - 1 + tid - 64, 0, H - 1) + 0.5f) / fH;
        };
        const int sy = tid / G::SC, sx = 2 * (tid - sy * G::SC);
        const bool inside = x0 >= 1 && y0 >= 1 && x0 + G::RW + 1 <= W && y0 + G::RH + 1 <= H;
        if (inside) {  // two texels a load, the pass in the scalar offset
            const uint32_t o = (uint32_t)sy * pitch + (uint32_t)sx;
            u32x4 c[G::SP];
            uint2 d[G::SP];
            VelT v[2 * G::SP];
#pragma unroll
            for (int p = 0; p < G::SP; ++p) {
                if (tid >= G::SC * G::SR || sy + p * G::SR >= G::SH) break;
                const uint32_t s = (uint32_t)(y0 - 1 + p * G::SR) * pitch + (uint32_t)(x0 - 1);
                c[p] = color.ld4(o * 8u, s * 8u);
                d[p] = depths.ld2(o * 4u, s * 4u);
                if constexpr (G::V4) {
                    const u32x4 q = velocity.ld4(o * 8u, s * 8u);
                    v[2 * p] = make_uint2(q.x, q.y);
                    v[2 * p + 1] = make_uint2(q.z, q.w);
                } else {
                    const uint2 q = velocity.ld2(o * 4u, s * 4u);
                    v[2 * p] = q.x;
                    v[2 * p + 1] = q.y;
                }
            }
            tables();
#pragma unroll
            for (int p = 0; p < G::SP; ++p) {
                if (tid >= G::SC * G::SR || sy + p * G::SR >= G::SH) break;
                store(2 * tid + p * G::SC * G::SR * 2, make_uint2(c[p].x, c[p].y), make_uint2(c[p].z, c[p].w), d[p], v[2 * p], v[2 * p + 1]);
            }
        } else {  // a tile over the image's border: texel by texel, clamped
            tables();
#pragma unroll 1
            for (int p = 0; p < G::SP; ++p) {
                if (tid >= G::SC * G::SR || sy + p * G::SR >= G::SH) break;
                const uint32_t r = (uint32_t)clampi(y0 - 1 + sy + p * G::SR, 0, H - 1) * pitch;
                const uint32_t g0 = r + (uint32_t)clampi(x0 - 1 + sx, 0, W - 1), g1 = r + (uint32_t)clampi(x0 + sx, 0, W - 1);
                VelT v0, v1;
                ld_vel(velocity, g0 * (uint32_t)sizeof(VelT), 0u, v0);
                ld_vel(velocity, g1 * (uint32_t)sizeof(VelT), 0u, v1);
                store(2 * tid + p * G::SC * G::SR * 2, color.ld2(g0 * 8u, 0u), color.ld2(g1 * 8u, 0u),
                      make_uint2(depths.ld1(g0 * 4u, 0u), depths.ld1(g1 * 4u, 0u)), v0, v1);
            }
        }
        __syncthreads();
    }

    // ---- 2. closest depth, history position and previous depth of the thread's texels; their footprints' box
    Texel0 q[RPT];
    int bx0 = 0x7fffffff, by0 = 0x7fffffff, bx1 = -0x7fffffff, by1 = -0x7fffffff;
    {
        const int base = rg * SW + rx;
        auto vel_of = [](const DepthVel& e) {
            if constexpr (G::V4) return make_uint2(e.y, e.z);
            else return e.y;
        };
        struct Row {
            float d, cd;      // the first smallest depth of the row's three in scan order (strict <), the centre's
            VelT v, cv, rv;   // the velocities under them, and the right one
            int k;            // column of the smallest (inspect image)
            uint32_t mov;     // bit 0: the centre moves, bit 1: a texel beside it does (anti-ghosting)
        };
        float sum = 0.0f;
        auto read_row = [&](int t) {
            Row r;
            const DepthVel c = dv[base + t * SW + 1];
            r.cd = __uint_as_float(c.x);
            r.cv = vel_of(c);
            if (closest_mode || ghost || longest) {
                const DepthVel l = dv[base + t * SW], e = dv[base + t * SW + 2];
                const float dl = __uint_as_float(l.x), dr = __uint_as_float(e.x);
                r.rv = vel_of(e);
                const bool c1 = r.cd < dl;
                const float d1 = c1 ? r.cd : dl;
                const bool c2 = dr < d1;
                r.d = c2 ? dr : d1;
                r.v = select(c2, r.rv, select(c1, r.cv, vel_of(l)));
                if constexpr (INSP) r.k = c2 ? 2 : c1 ? 1 : 0;
                sum += (dl + r.cd) + dr;
                r.mov = 0u;
                if (ghost) {
                    constexpr float eps = 1e-5f;
                    auto moves = [&](VelT v) {
                        const float4 a = vel_xyzw(v);
                        return (fabsf(a.x) > eps || fabsf(a.y) > eps) && fabsf(a.w) >= 0.5f;
                    };
                    r.mov = (moves(r.cv) ? 1u : 0u) | (moves(vel_of(l)) || moves(r.rv) ? 2u : 0u);
                }
            }
            return r;
        };
        const float uvx = sm.ux[rx + 1];
        Row ra = read_row(0), rb = read_row(1);
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            const float uvy = sm.uy[rg + k + 1];
            const Row rc = read_row(k + 2);
            VelT vs = rb.cv;
            int closest = -1;
            if (closest_mode) {  // findClosestUvAndZ_3x3 (taa.comp:371-389): the rows' minima in scan order, strict <
                const bool c1 = rb.d < ra.d;
                const float d1 = c1 ? rb.d : ra.d;
                const bool c2 = rc.d < d1;
                vs = select(c2, rc.v, select(c1, rb.v, ra.v));
                if constexpr (INSP) closest = c2 ? 6 + rc.k : c1 ? 3 + rb.k : ra.k;
                if (!(sum == sum)) {  // a NaN among the depths read so far: the scan itself, in which only a NaN first tap stays
                    const DepthVel e0 = dv[base + k * SW];
                    float d = __uint_as_float(e0.x);
                    vs = vel_of(e0);
                    closest = 0;
#pragma unroll 1
                    for (int j = 1; j < 9; ++j) {
                        const DepthVel e = dv[base + (k + j / 3) * SW + j % 3];
                        if (__uint_as_float(e.x) < d) d = __uint_as_float(e.x), vs = vel_of(e), closest = j;
                    }
                }
            }
            const float depth = rb.cd;
            float hu, hv2;
            q[k].expected = depth;
            q[k].used_velocity = true;
            if constexpr (!EXT) {
                const float2 v = vel_xy(vs);
                hu = __builtin_fmaf(v.x, -1.0f, uvx);  // uv - v (taa.comp:421)
                hv2 = __builtin_fmaf(v.y, -1.0f, uvy);
            } else {
                // movers only (mode 1) reads .w of the centre tap; RG formats read w = 1
                const float4 vc = vel_xyzw(rb.cv);
                q[k].used_velocity = !(use_velocity == 0 || (use_velocity == 1 && vc.w < 0.5f));
                float4 v = vel_xyzw(vs);
                if (longest) {  // taa.comp:398-412: the last tap's xy, not the longest
                    const float2 l = vel_xy(rc.rv);
                    v.x = l.x;
                    v.y = l.y;
                }
                hu = uvx - v.x;
                hv2 = uvy - v.y;
                q[k].expected = depth - v.z;
                if (!q[k].used_velocity) {  // reprojection through the matrices (taa.comp:424-431), IEEE divisions as the FP32 path
                    closest = -1;
                    const float* Mi = U.mInverseViewProjMatrix;
                    const float* Mh = U.mHistoryViewProjMatrix;
                    const float cs[4] = {uvx * 2.0f - 1.0f, uvy * 2.0f - 1.0f, depth, 1.0f};
                    float wv[4], hc[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) wv[r] = Mi[r] * cs[0] + Mi[4 + r] * cs[1] + Mi[8 + r] * cs[2] + Mi[12 + r] * cs[3];
#pragma unroll
                    for (int r = 0; r < 4; ++r) hc[r] = Mh[r] * wv[0] + Mh[4 + r] * wv[1] + Mh[8 + r] * wv[2] + Mh[12 + r] * wv[3];
                    hu = (hc[0] / hc[3]) * 0.5f + 0.5f;
                    hv2 = (hc[1] / hc[3]) * 0.5f + 0.5f;
                    q[k].expected = hc[2] / hc[3];
                }
                q[k].moved = (rb.mov & 1u) != 0u;
                q[k].calm = ((ra.mov | rc.mov) & 1u) == 0u && rb.mov == 0u;
            }
            q[k].closest = closest;
            q[k].hu = hu;
            q[k].hv = hv2;
            const float sX = hu * fW, sY = hv2 * fH;
            q[k].pd = 0.0f;
            q[k].dtx = q[k].dty = 0;
            if (depth_cull) {  // previous depth under the history position (taa.comp:818)
                q[k].dtx = to_int(sX);
                q[k].dty = to_int(sY);
                q[k].pd = __uint_as_float(hdepth.ld1(((uint32_t)med3<0>(q[k].dty, H - 1) * pitch + (uint32_t)med3<0>(q[k].dtx, W - 1)) * 4u, 0u));
            }
            const float tX = sX - 0.5f, tY = sY - 0.5f;
            const float fbx = floorf(tX), fby = floorf(tY);
            q[k].fx = tX - fbx;
            q[k].fy = tY - fby;
            if constexpr (INSP) {
                q[k].ix = to_int(fbx);
                q[k].iy = to_int(fby);
            }
            // the base pre-clamped (cr_base): every tap clamped to the edge still reads the texel the unclamped tap would
            q[k].kx = med3<-2>(to_int(fbx), W + 1);
            q[k].ky = med3<-2>(to_int(fby), H + 1);
            bx0 = min(bx0, q[k].kx), by0 = min(by0, q[k].ky), bx1 = max(bx1, q[k].kx), by1 = max(by1, q[k].ky);
            ra = rb, rb = rc;
        }
    }
    constexpr int FN = G::FN;
    uint2 foot[G::WIN ? 1 : RPT][FN * FN];  // without the window: the texels' footprints, FN rows of FN (or 2 of 2)
    if constexpr (!G::WIN) {
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            const int kx = q[k].kx, ky = q[k].ky;
            q[k].outside = reject_out && (q[k].hu < 0.0f || q[k].hv < 0.0f || q[k].hu >= 1.0f || q[k].hv >= 1.0f);
            const int n = cr_hist ? 4 : 2, first = cr_hist ? -1 : 0;
            // a row's texels in 16-byte loads, from a base that keeps them inside the image; a wave with a footprint over
            // its edge (or an image too small) reads them one by one, clamped
            const int bx = max(min(kx + first, W - n), 0), by = max(min(ky + first, H - n), 0);
            const uint32_t o = ((uint32_t)by * pitch + (uint32_t)bx) * 8u;
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                if (j >= n) break;
                const uint32_t s = (uint32_t)min(j, H - 1) * pitch * 8u;
                const u32x4 a = history.ld4(o, s);
                foot[k][FN * j] = make_uint2(a.x, a.y), foot[k][FN * j + 1] = make_uint2(a.z, a.w);
                if constexpr (FN == 4)
                    if (cr_hist) {
                        const u32x4 b = history.ld4(o + 16u, s);
                        foot[k][FN * j + 2] = make_uint2(b.x, b.y), foot[k][FN * j + 3] = make_uint2(b.z, b.w);
                    }
            }
            if (__builtin_amdgcn_ballot_w64(bx != kx + first) | __builtin_amdgcn_ballot_w64(by != ky + first) | (uint64_t)(W < n || H < n)) {
#pragma unroll
                for (int j = 0; j < FN; ++j) {
                    if (j >= n) break;
                    const uint32_t r = (uint32_t)clampi(ky + first + j, 0, H - 1) * pitch;
#pragma unroll
                    for (int i = 0; i < FN; ++i)
                        if (i < n) foot[k][FN * j + i] = history.ld2((r + (uint32_t)clampi(kx + first + i, 0, W - 1)) * 8u, 0u);
                }
#pragma unroll
                for (int j = 0; j < FN * FN; ++j)
                    if (G::CR != kAny || j < 6) asm volatile("" : "+v"(foot[k][j].x), "+v"(foot[k][j].y));  // waited for here
            }
        }
    }
    bool fits = false;
    if constexpr (G::WIN) {
        // (a texel outside the image has the position of the border texel it was staged from)
        const int4 wb = wave_min(make_int4(bx0, by0, -bx1, -by1));
        if ((tid & 63) == 0) sm.box[tid >> 6] = wb;
#pragma unroll
        for (int k = 0; k < RPT; ++k) q[k].outside = false;
        // positions outside the image: none in a wave whose bases all lie in 0 .. size - 2
        if (reject_out && (wb.x < 0 || wb.y < 0 || wb.z < 2 - W || wb.w < 2 - H)) {
#pragma unroll
            for (int k = 0; k < RPT; ++k) q[k].outside = q[k].hu < 0.0f || q[k].hv < 0.0f || q[k].hu >= 1.0f || q[k].hv >= 1.0f;
        }
        __syncthreads();
        int4 b = sm.box[0];
#pragma unroll
        for (int w = 1; w < G::NT / 64; ++w) {
            const int4 o = sm.box[w];
            b = make_int4(min(b.x, o.x), min(b.y, o.y), min(b.z, o.z), min(b.w, o.w));
        }
        // the window: taps k - 1 .. k + 2 of every footprint (bilinear ones use k, k + 1)
        const int wx0 = scalar(b.x) - 1, wy0 = scalar(b.y) - 1;
        const int ww = -scalar(b.z) - scalar(b.x) + 4, wh = -scalar(b.w) - scalar(b.y) + 4;
        fits = ww <= G::WP && wh <= G::WH;

        // ---- 3. the window's texels, clamped to the edge
        if (fits) {
            const int row = tid / G::WC, col = 2 * (tid - row * G::WC);
            u32x4 v[G::WN];
            if (wx0 >= 0 && wy0 >= 0 && wx0 + ww + 1 <= W && wy0 + wh <= H) {
                const uint32_t o = ((uint32_t)row * pitch + (uint32_t)col) * 8u;
                const uint32_t s0 = ((uint32_t)wy0 * pitch + (uint32_t)wx0) * 8u;
                // only what the footprints cover: a full rectangle of WP columns read 15% more from HBM (4K, 284 against 245 MB)
                const bool take = tid < G::WC * G::WR && col < ww;
#pragma unroll
                for (int p = 0; p < G::WN; ++p)
                    if (take && row + p * G::WR < wh) v[p] = history.ld4(o, s0 + (uint32_t)(p * G::WR) * pitch * 8u);
#pragma unroll
                for (int p = 0; p < G::WN; ++p)
                    if (take && row + p * G::WR < wh) *reinterpret_cast<u32x4*>(win + 2 * tid + p * G::WC * G::WR * 2) = v[p];
                for (int p = G::WN; p * G::WR < wh; ++p)
                    if (take && row + p * G::WR < wh)
                        *reinterpret_cast<u32x4*>(win + 2 * tid + p * G::WC * G::WR * 2) = history.ld4(o, s0 + (uint32_t)(p * G::WR) * pitch * 8u);
            } else {
#pragma unroll 1
                for (int p = 0; p * G::WR < wh; ++p) {
                    const uint32_t r = (uint32_t)clampi(wy0 + row + p * G::WR, 0, H - 1) * pitch;
                    const uint2 a = history.ld2((r + (uint32_t)clampi(wx0 + col, 0, W - 1)) * 8u, 0u);
                    const uint2 c = history.ld2((r + (uint32_t)clampi(wx0 + col + 1, 0, W - 1)) * 8u, 0u);
                    if (tid < G::WC * G::WR && row + p * G::WR < wh) *reinterpret_cast<u32x4*>(win + 2 * tid + p * G::WC * G::WR * 2) = u32x4{a.x, a.y, c.x, c.y};
                }
            }
        }
#pragma unroll
        for (int k = 0; k < RPT; ++k) q[k].k = fits ? (q[k].ky - 1 - wy0) * G::WP + q[k].kx - 1 - wx0 : 0;
        __syncthreads();
    }

    // ---- 4. box, history filter, rejection, rectification and blend
    const float a_span = a_min - a_max;
    const bool own_col = x0 + rx < fd.x_end && (!G::CAS || (rx >= 1 && rx < 31));
    uint2 hbs[RPT];
    f3 r1[3], r2[3];  // three columns' sums and sums of squares (minima and maxima) of rows k, k + 1, k + 2
    f3 cen[2];        // centre texels of rows k + 1, k + 2
    auto row_sums = [&](int t, f3& s, f3& ss, f3& c) {
        const int i = (rg + t) * SW + rx;
        const float2 a0 = sm.c01[i], a1 = sm.c01[i + 1], a2 = sm.c01[i + 2];
        const float b0 = sm.c2[i], b1 = sm.c2[i + 1], b2 = sm.c2[i + 2];
        c = {a1.x, a1.y, b1};
        if (var_clip) {
            s = {(a0.x + a1.x) + a2.x, (a0.y + a1.y) + a2.y, (b0 + b1) + b2};
            ss = {__builtin_fmaf(a2.x, a2.x, __builtin_fmaf(a1.x, a1.x, a0.x * a0.x)), __builtin_fmaf(a2.y, a2.y, __builtin_fmaf(a1.y, a1.y, a0.y * a0.y)),
                  __builtin_fmaf(b2, b2, __builtin_fmaf(b1, b1, b0 * b0))};
        } else {
            s = {fminf(a1.x, fminf(a0.x, a2.x)), fminf(a1.y, fminf(a0.y, a2.y)), fminf(b1, fminf(b0, b2))};
            ss = {fmaxf(a1.x, fmaxf(a0.x, a2.x)), fmaxf(a1.y, fmaxf(a0.y, a2.y)), fmaxf(b1, fmaxf(b0, b2))};
        }
    };
    {
        f3 unused;
        row_sums(0, r1[0], r2[0], unused);
        row_sums(1, r1[1], r2[1], cen[0]);
    }
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
        const int x = x0 + rx, y = y0 + rg + k;
        const bool owned = own_col && (k > 0 || !G::CAS || rg > 0) && (k < RPT - 1 || !G::CAS || rg < G::RH - RPT) && y < H;
        row_sums(k + 2, r1[2], r2[2], cen[1]);
        const f3 c = cen[0];
        f3 mean, sig, mn, mx;
        if (var_clip) {
            constexpr float inv9 = 1.0f / 9.0f;
            mean = ((r1[0] + r1[1]) + r1[2]) * inv9;
            const f3 m2 = ((r2[0] + r2[1]) + r2[2]) * inv9;
            sig = {sqrt_fast(fmaxf(__builtin_fmaf(-mean.x, mean.x, m2.x), 0.f)), sqrt_fast(fmaxf(__builtin_fmaf(-mean.y, mean.y, m2.y), 0.f)),
                   sqrt_fast(fmaxf(__builtin_fmaf(-mean.z, mean.z, m2.z), 0.f))};
        } else {
            mn = vmin(vmin(r1[0], r1[1]), r1[2]);
            mx = vmax(vmax(r2[0], r2[1]), r2[2]);
        }
        r1[0] = r1[1], r1[1] = r1[2], r2[0] = r2[1], r2[1] = r2[2], cen[0] = cen[1];

        // ---- history filter, fp32 accumulation: Catmull-Rom (taa.comp:441-514), separable, or bilinear (taa.comp:545-549)
        f3 hrgb;
        float ha = 0.0f;
        if (cr_hist) {
            const W4 wx = cr_weights(q[k].fx), wy = cr_weights(q[k].fy);
            hrgb = {0.f, 0.f, 0.f};
            auto add_row = [&](const uint2 (&e)[4], float w) {
                f3 row = {0.f, 0.f, 0.f};
                float rowa = 0.0f;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    row.x = __builtin_fmaf(lo16(e[i].x), wx.w[i], row.x);
                    row.y = __builtin_fmaf(hi16(e[i].x), wx.w[i], row.y);
                    row.z = __builtin_fmaf(lo16(e[i].y), wx.w[i], row.z);
                    if (ghost) rowa = __builtin_fmaf(hi16(e[i].y), wx.w[i], rowa);
                }
                hrgb.x = __builtin_fmaf(row.x, w, hrgb.x);
                hrgb.y = __builtin_fmaf(row.y, w, hrgb.y);
                hrgb.z = __builtin_fmaf(row.z, w, hrgb.z);
                if (ghost) ha = __builtin_fmaf(rowa, w, ha);
            };
            if constexpr (!G::WIN) {
#pragma unroll
                for (int j = 0; j < FN; ++j) {
                    const uint2 e[4] = {foot[k][FN * j], foot[k][FN * j + 1], foot[k][FN * j + 2 & (FN * FN - 1)], foot[k][FN * j + 3 & (FN * FN - 1)]};
                    add_row(e, wy.w[j]);
                }
            } else if (fits) {
                const uint2* w = win + q[k].k;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint2 e[4] = {w[j * G::WP], w[j * G::WP + 1], w[j * G::WP + 2], w[j * G::WP + 3]};
                    add_row(e, wy.w[j]);
                }
            } else if (__builtin_amdgcn_ballot_w64(q[k].kx < 1 || q[k].kx > W - 3 || q[k].ky < 1 || q[k].ky > H - 3) == 0) {
                // the tile's footprints lie too far apart for the window (motion that differs by more than its margin): from
                // memory, a row's two 16-byte loads at a time (two rows at a time cost registers everywhere: 3840x2160 113 us, not 108)
                uint32_t o = ((uint32_t)(q[k].ky - 1) * pitch + (uint32_t)(q[k].kx - 1)) * 8u;
#pragma unroll 1
                for (int j = 0; j < 4; ++j) {
                    const u32x4 a = history.ld4(o, 0u), b = history.ld4(o + 16u, 0u);
                    const uint2 e[4] = {make_uint2(a.x, a.y), make_uint2(a.z, a.w), make_uint2(b.x, b.y), make_uint2(b.z, b.w)};
                    add_row(e, j == 0 ? wy.w[0] : j == 1 ? wy.w[1] : j == 2 ? wy.w[2] : wy.w[3]);
                    o += pitch * 8u;
                }
            } else {  // ... and over the image's edge: texel by texel, clamped
#pragma unroll 1
                for (int j = 0; j < 4; ++j) {
                    const uint32_t r = (uint32_t)clampi(q[k].ky - 1 + j, 0, H - 1) * pitch;
                    uint2 e[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) e[i] = history.ld2((r + (uint32_t)clampi(q[k].kx - 1 + i, 0, W - 1)) * 8u, 0u);
                    add_row(e, j == 0 ? wy.w[0] : j == 1 ? wy.w[1] : j == 2 ? wy.w[2] : wy.w[3]);
                }
            }
        } else {
            uint2 e[4];
            if constexpr (!G::WIN) {
                e[0] = foot[k][0], e[1] = foot[k][1], e[2] = foot[k][FN], e[3] = foot[k][FN + 1];
            } else if (fits) {
                const uint2* w = win + q[k].k + G::WP + 1;
                e[0] = w[0], e[1] = w[1], e[2] = w[G::WP], e[3] = w[G::WP + 1];
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    e[j] = history.ld2(((uint32_t)clampi(q[k].ky + j / 2, 0, H - 1) * pitch + (uint32_t)clampi(q[k].kx + j % 2, 0, W - 1)) * 8u, 0u);
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) asm volatile("" : "+v"(e[j].x), "+v"(e[j].y));  // waited for here, not where the paths meet
            }
            const float fx = q[k].fx, fy = q[k].fy, ux = 1.0f - fx, uy = 1.0f - fy;
            auto mix = [](float a, float b, float u, float t) { return __builtin_fmaf(b, t, a * u); };
            auto quad = [&](float a, float b, float c, float d) { return mix(mix(a, b, ux, fx), mix(c, d, ux, fx), uy, fy); };
            if constexpr (G::EX) {  // bilinear4_quad
                auto exact = [&](float a, float b, float c, float d) { return (a * ux + b * fx) * uy + (c * ux + d * fx) * fy; };
                hrgb = {exact(lo16(e[0].x), lo16(e[1].x), lo16(e[2].x), lo16(e[3].x)), exact(hi16(e[0].x), hi16(e[1].x), hi16(e[2].x), hi16(e[3].x)),
                        exact(lo16(e[0].y), lo16(e[1].y), lo16(e[2].y), lo16(e[3].y))};
            } else
            hrgb = {quad(lo16(e[0].x), lo16(e[1].x), lo16(e[2].x), lo16(e[3].x)), quad(hi16(e[0].x), hi16(e[1].x), hi16(e[2].x), hi16(e[3].x)),
                    quad(lo16(e[0].y), lo16(e[1].y), lo16(e[2].y), lo16(e[3].y))};
            if (ghost) ha = quad(hi16(e[0].y), hi16(e[1].y), hi16(e[2].y), hi16(e[3].y));
        }
        const Texel0& p = q[k];
        
        f3 h = hrgb;
        if (ycocg) {
            const float t = 0.25f * (hrgb.x + hrgb.z);
            h = {__builtin_fmaf(0.5f, hrgb.y, t), 0.5f * (hrgb.x - hrgb.z), __builtin_fmaf(0.5f, hrgb.y, -t)};
        }
        // decisions as in the FP32 path (taa.comp:787-823)
        bool rejected = p.outside;
        int flags = p.used_velocity ? TAA_FLAG_USED_VELOCITY : 0;
        if (rejected) flags |= TAA_FLAG_OUTSIDE;
        if (ghost && p.calm && ha > 0.0f) {
            rejected = true;
            flags |= TAA_FLAG_GHOST_REJECT;
        }
        const bool write_mask = ghost && p.moved;  // history alpha: the dynamic mask (taa.comp:796-811)
        if (depth_cull) {
            const bool rej = lin_depth ? linear_depth_reject(p.pd, p.expected, near, far, lin_thr)
                                       : fabsf(p.pd - p.expected) > 0.1f * (1.0f - p.pd);
            if (rej) {
                rejected = true;
                flags |= TAA_FLAG_DEPTH_REJECT;
            }
        }
        // clamp to / clip towards the box (taa.comp:288-345)
        if (var_clip) {
            mn = {__builtin_fmaf(-gamma, sig.x, mean.x), __builtin_fmaf(-gamma, sig.y, mean.y), __builtin_fmaf(-gamma, sig.z, mean.z)};
            mx = {__builtin_fmaf(gamma, sig.x, mean.x), __builtin_fmaf(gamma, sig.y, mean.y), __builtin_fmaf(gamma, sig.z, mean.z)};
        }
        const f3 h_orig = h;
        if (rect == 2) {
            // clipAabb (taa.comp:323-345): ma = max_i |v_i| / e_i, clip when ma > 1, with one
            // reciprocal: ma = M / D for M = max_i |v_i| * prod_{j != i} e_j and D = e_x e_y e_z
            f3 bc2, e;
            if (var_clip) {
                bc2 = mean;
                e = {__builtin_fmaf(gamma, sig.x, 1e-7f), __builtin_fmaf(gamma, sig.y, 1e-7f), __builtin_fmaf(gamma, sig.z, 1e-7f)};
            } else {
                bc2 = f3{0.5f * (mx.x + mn.x), 0.5f * (mx.y + mn.y), 0.5f * (mx.z + mn.z)};
                e = {__builtin_fmaf(0.5f, mx.x - mn.x, 1e-7f), __builtin_fmaf(0.5f, mx.y - mn.y, 1e-7f), __builtin_fmaf(0.5f, mx.z - mn.z, 1e-7f)};
            }
            const f3 vc = h - bc2;
            const float exy = e.x * e.y, D = exy * e.z;
            const float M = fmaxf(fabsf(vc.x) * (e.y * e.z), fmaxf(fabsf(vc.y) * (e.x * e.z), fabsf(vc.z) * exy));
            if (M > D) {
                const float s = D * rcp_fast(M);
                h = {__builtin_fmaf(vc.x, s, bc2.x), __builtin_fmaf(vc.y, s, bc2.y), __builtin_fmaf(vc.z, s, bc2.z)};
            }
        } else if (rect == 1) {
            h = vmin(vmax(h, mn), mx);
        }
        // blend (taa.comp:850-900)
        auto luma = [&](const f3& c) { return ycocg ? c.x : 0.25f * (c.x + c.z) + 0.5f * c.y; };
        float pixel_speed = 0.0f;
        if (EXT) {
            const float vux = sm.ux[rx + 1] - p.hu, vuy = sm.uy[rg + k + 1] - p.hv;
            pixel_speed = sqrt_fast(vux * vux + vuy * vuy);  // taa.comp:434-435
        }
        float alpha = a_plain;
        if (vel_alpha) {  // taa.comp:855-859
            const float t = fminf(fmaxf(pixel_speed * P.mVelBasedAlphaFactor, 0.0f), 1.0f);
            alpha = fmaxf(alpha, __builtin_fmaf(t, P.mVelBasedAlphaMax - alpha, alpha));
        }
        if (lottes) {
            const float lc = luma(c), lh = luma(h);
            const float diff = fabsf(lc - lh) * rcp_fast(fmaxf(fmaxf(lc, lh), 0.2f));
            const float w = 1.0f - diff;
            alpha = __builtin_fmaf(w * w, a_span, a_max);
        }
        if (near_clamp) {  // taa.comp:873-894 (the Unreal-based form)
            const float mnl = luma(mn), mxl = luma(mx), hl = luma(h_orig);
            float dist = 2.0f * fabsf(fminf(hl - mnl, mxl - hl)) * rcp_fast(mxl - mnl);
            if (mxl - mnl < 0.001f) dist = 1.0f;
            alpha *= fminf(fmaxf(4.0f * dist, 0.0f), 1.0f);
        }
        if (rejected) alpha = a_reject;
        if (reset) alpha = 1.0f;
        f3 aa = {__builtin_fmaf(alpha, c.x - h.x, h.x), __builtin_fmaf(alpha, c.y - h.y, h.y), __builtin_fmaf(alpha, c.z - h.z, h.z)};
        if (reset) aa = c;  // exactly the current colour, whatever the history holds
        if constexpr (G::EX) aa = {gmix(h.x, c.x, alpha), gmix(h.y, c.y, alpha), gmix(h.z, c.z, alpha)};
        if (ycocg) {
            const float t = aa.x - aa.z;
            aa = {t + aa.y, aa.x + aa.z, t - aa.y};
        }
        // fp16 bits of the result, converted once for the history, the screen and the CAS rows
        const uint2 hb = make_uint2(pack_sat(aa.x, aa.y), pack_sat(aa.z, 0.0f));
        if (owned) {
            const uint32_t gi = (uint32_t)y * pitch + (uint32_t)x;
            // history alpha = the dynamic mask (0 or 1: 0x3c00 in fp16); the screen's alpha is 1
            history_out.st2(make_uint2(hb.x, write_mask ? hb.y | 0x3c000000u : hb.y), out_off, (uint32_t)k * pitch * 8u);
            if constexpr (!G::CAS) screen.st2(make_uint2(hb.x, hb.y | 0x3c000000u), out_off, (uint32_t)k * pitch * 8u);
            if (G::OPTIONS != 0 && fd.debug) {  // taa.comp:912-942 (mode 8: no mask here, category 0)
                float4 g = make_float4(0.f, 0.f, 0.f, 0.f);
                const float wm = write_mask ? 1.0f : 0.0f;
                switch (P.mDebugMode) {
                    case 0: g = make_float4(mx.x - mn.x, mx.y - mn.y, mx.z - mn.z, 0.f); break;
                    case 1: { const float t = (mx.x - mn.x) * (mx.y - mn.y) * (mx.z - mn.z); g = make_float4(t, t, t, 0.f); break; }
                    case 2: {
                        const f3 d = h - h_orig;
                        g = make_float4(rejected ? 1.f : 0.f, sqrt_fast(d.x * d.x + d.y * d.y + d.z * d.z), 0.f, 0.f);
                        break;
                    }
                    case 3: g = make_float4(alpha, alpha, alpha, 0.f); break;
                    case 4: { VelT v; ld_vel(velocity, gi * (uint32_t)sizeof(VelT), 0u, v); g = vel_xyzw(v); } break;
                    case 5: g = make_float4(pixel_speed, 0.f, 0.f, 0.f); break;
                    case 6: g = make_float4(aa.x, aa.y, aa.z, 1.0f); break;
                    case 7: g = make_float4(aa.x, aa.y, aa.z, wm); break;
                    case 8: g = make_float4(0.f, 0.f, 1.f, 0.f); break;
                    default: break;
                }
                const float ds = P.mDebugScale;
                g = make_float4(g.x * ds * P.mDebugMask[0], g.y * ds * P.mDebugMask[1], g.z * ds * P.mDebugMask[2],
                                g.w * ds * P.mDebugMask[3]);
                if (P.mDebugCenter) g = make_float4(g.x * 0.5f + 0.5f, g.y * 0.5f + 0.5f, g.z * 0.5f + 0.5f, g.w * 0.5f + 0.5f);
                st_rgba16(fd.debug, gi, g);
            }
            if constexpr (INSP) {
                if (rejected) flags |= TAA_FLAG_REJECTED;
                int32_t w[TAA_INSPECT_WORDS];
                w[TAA_INSPECT_HIST_TC_X] = p.ix;
                w[TAA_INSPECT_HIST_TC_Y] = p.iy;
                w[TAA_INSPECT_CLOSEST_TAP] = p.closest;
                w[TAA_INSPECT_FLAGS] = flags;
                w[TAA_INSPECT_COLMIN + 0] = __float_as_int(mn.x);
                w[TAA_INSPECT_COLMIN + 1] = __float_as_int(mn.y);
                w[TAA_INSPECT_COLMIN + 2] = __float_as_int(mn.z);
                w[TAA_INSPECT_COLMAX + 0] = __float_as_int(mx.x);
                w[TAA_INSPECT_COLMAX + 1] = __float_as_int(mx.y);
                w[TAA_INSPECT_COLMAX + 2] = __float_as_int(mx.z);
                w[TAA_INSPECT_BLEND] = __float_as_int(alpha);
                w[TAA_INSPECT_DEPTH_TC_X] = p.dtx;
                w[TAA_INSPECT_DEPTH_TC_Y] = p.dty;
                w[TAA_INSPECT_HIST_UV_X] = __float_as_int(p.hu);
                w[TAA_INSPECT_HIST_UV_Y] = __float_as_int(p.hv);
                w[15] = 0;
                st_inspect(fd.inspect, gi, w);
            }
        }
        hbs[k] = hb;
    }

    // ---- 5. fused CAS: left and right neighbours from LDS, upper and lower ones of the thread's own column where it
    // has them; at the image's border the missing neighbour is the texel itself
    if constexpr (G::CAS) {
        if constexpr (G::WIN) __syncthreads();  // every thread is done with the staged colours
        uint2* const res = sm.res();
#pragma unroll
        for (int k = 0; k < RPT; ++k) res[(rg + k) * 32 + rx] = hbs[k];
        __syncthreads();
        const int x = x0 + rx;
        const bool border = x0 < 0 || y0 < 0 || x0 + G::RW >= W || y0 + G::RH >= H;
        if (!own_col) return;
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            const int ry = rg + k, y = y0 + ry;
            if ((k == 0 && rg == 0) || (k == RPT - 1 && rg == G::RH - RPT) || y >= H) continue;
            const uint2 c = hbs[k];
            uint2 l = res[ry * 32 + rx - 1], r = res[ry * 32 + rx + 1];
            uint2 u = k > 0 ? hbs[k - 1] : res[(ry - 1) * 32 + rx], d = k < RPT - 1 ? hbs[k + 1] : res[(ry + 1) * 32 + rx];
            if (border) {
                if (x == 0) l = c;
                if (x == W - 1) r = c;
                if (y == 0) u = c;
                if (y == H - 1) d = c;
            }
            if constexpr (G::EX) {
                auto rgb = [](uint2 t) { return f3{lo16(t.x), hi16(t.x), lo16(t.y)}; };
                const f3 o = cas_filter(rgb(u), rgb(l), rgb(c), rgb(r), rgb(d), peak);
                screen.st2(make_uint2(pack_sat(o.x, o.y), pack_sat(o.z, 1.0f)), out_off, (uint32_t)k * pitch * 8u);
            } else {
                screen.st2(cas_filter_h2(u, l, c, r, d, peak), out_off, (uint32_t)k * pitch * 8u);
            }
        }
    }
}

// Occupancy hints (waves per SIMD): what the workgroup's LDS allows and the form fits without spills.
constexpr int window_waves(int rpt, int form, bool insp) {
    const int ext = form == kExt || form == kExtRgba ? 1 : 0;
    return insp ? 1 : rpt == 2 ? 6 - ext : 5 - ext;
}

struct FastArgs {
    FrameDesc fd;
    taa_uniforms_t U;
};

template <int NT, int RPT, bool CAS, bool INSP, int FORM>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(window_waves(RPT, FORM, INSP)))) void k_resolve_window(const FastArgs a) {
    using G = WinGeo<NT, RPT, CAS, INSP, FORM>;
    __shared__ typename G::Smem sm;
    resolve_window<G>(a.fd, a.U, xcd_tile((int)blockIdx.x, a.fd.tiles_x * a.fd.tiles_y), sm);
}

template <int NT, int RPT, bool CAS, int FORM>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(window_waves(RPT, FORM, false)))) void k_resolve_window_batch(const BatchEntry* __restrict__ entries, int n_entries, int total) {
    using G = WinGeo<NT, RPT, CAS, false, FORM>;
    __shared__ typename G::Smem sm;
    const int t = batch_tile(total);
    if (t < 0) return;
    const BatchEntry& e = batch_entry(entries, n_entries, t);
    resolve_window<G>(e.fd, e.U, t - e.tile_begin, sm);
}

template <int NT, int RPT, bool CAS, bool INSP>
void launch_window_f(const FastArgs& a, int form, hipStream_t st) {
    const dim3 n(a.fd.tiles_x * a.fd.tiles_y);
    switch (form) {
        case kProd: hipLaunchKernelGGL((k_resolve_window<NT, RPT, CAS, INSP, kProd>), n, dim3(NT), 0, st, a); break;
        case kVar: hipLaunchKernelGGL((k_resolve_window<NT, RPT, CAS, INSP, kVar>), n, dim3(NT), 0, st, a); break;
        case kGeneral: hipLaunchKernelGGL((k_resolve_window<NT, RPT, CAS, INSP, kGeneral>), n, dim3(NT), 0, st, a); break;
        case kExt: hipLaunchKernelGGL((k_resolve_window<NT, RPT, CAS, INSP, kExt>), n, dim3(NT), 0, st, a); break;
        case kExtRgba: hipLaunchKernelGGL((k_resolve_window<NT, RPT, CAS, INSP, kExtRgba>), n, dim3(NT), 0, st, a); break;
        case kDefaultExact:
            if constexpr (!INSP && RPT < 4) hipLaunchKernelGGL((k_resolve_window<NT, RPT, CAS, INSP, kDefaultExact>), n, dim3(NT), 0, st, a);
            break;
        default: hipLaunchKernelGGL((k_resolve_window<NT, RPT, CAS, INSP, kDefault>), n, dim3(NT), 0, st, a); break;
    }
}

template <int NT, int RPT, bool CAS>
void launch_window_batch_f(const BatchEntry* e, int n, int total, int form, hipStream_t st) {
    const dim3 grid(batch_grid(total));
    switch (form) {
        case kProd: hipLaunchKernelGGL((k_resolve_window_batch<NT, RPT, CAS, kProd>), grid, dim3(NT), 0, st, e, n, total); break;
        case kVar: hipLaunchKernelGGL((k_resolve_window_batch<NT, RPT, CAS, kVar>), grid, dim3(NT), 0, st, e, n, total); break;
        case kGeneral: hipLaunchKernelGGL((k_resolve_window_batch<NT, RPT, CAS, kGeneral>), grid, dim3(NT), 0, st, e, n, total); break;
        case kExt: hipLaunchKernelGGL((k_resolve_window_batch<NT, RPT, CAS, kExt>), grid, dim3(NT), 0, st, e, n, total); break;
        case kExtRgba: hipLaunchKernelGGL((k_resolve_window_batch<NT, RPT, CAS, kExtRgba>), grid, dim3(NT), 0, st, e, n, total); break;
        case kDefaultExact:
            if constexpr (RPT < 4) hipLaunchKernelGGL((k_resolve_window_batch<NT, RPT, CAS, kDefaultExact>), grid, dim3(NT), 0, st, e, n, total);
            break;
        default: hipLaunchKernelGGL((k_resolve_window_batch<NT, RPT, CAS, kDefault>), grid, dim3(NT), 0, st, e, n, total); break;
    }
}

template <bool CAS, bool INSP>
void launch_window_r(const FastArgs& a, int form, hipStream_t st) {
    switch (a.fd.rows) {
        case 1: launch_window_f<CAS ? 512 : 256, 1, CAS, INSP>(a, form, st); break;
        case 2: launch_window_f<256, 2, CAS, INSP>(a, form, st); break;
        default: launch_window_f<256, 4, CAS, INSP>(a, form, st); break;
    }
}

template <bool CAS>
void launch_window_batch_r(const BatchEntry* e, int n, int total, int rows, int form, hipStream_t st) {
    switch (rows) {
        case 1: launch_window_batch_f<CAS ? 512 : 256, 1, CAS>(e, n, total, form, st); break;
        case 2: launch_window_batch_f<256, 2, CAS>(e, n, total, form, st); break;
        default: launch_window_batch_f<256, 4, CAS>(e, n, total, form, st); break;
    }
}

}  // namespace

int launch_window(const FrameDesc& fd, const taa_uniforms_t& U, int form, void* stream) {
    hipStream_t st = static_cast<hipStream_t>(stream);
    FastArgs a;
    a.fd = fd;
    a.U = U;
    const bool insp = fd.inspect != nullptr;
    if (fd.cas_on) {
        if (insp) launch_window_r<true, true>(a, form, st);
        else launch_window_r<true, false>(a, form, st);
    } else {
        if (insp) launch_window_r<false, true>(a, form, st);
        else launch_window_r<false, false>(a, form, st);
    }
    return (int)hipGetLastError();
}

int launch_window_batch(const BatchEntry* d_entries, int n_entries, int total, int rows, bool cas, int form, void* stream) {
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (cas) launch_window_batch_r<true>(d_entries, n_entries, total, rows, form, st);
    else launch_window_batch_r<false>(d_entries, n_entries, total, rows, form, st);
    return (int)hipGetLastError();
}

}  // namespace taastar
