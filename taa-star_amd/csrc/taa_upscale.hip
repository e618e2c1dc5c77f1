// gfx950 upsampling resolve (input size no larger than the output) with the production feature set:
// variance box, clip, YCoCg, Catmull-Rom history, closest-depth RG velocity of the colour's precision,
// depth culling, Lottes, outside rejection. Exact FP32 arithmetic, operation for operation that of the
// general kernel (taa_kernels.hip), or with FA the FP16 path's where no selection depends on it.
//
// What bounds it: VALU issue. The kernel this replaced for these sizes spent 2,850 clocks a wave and SIMD on a texel
// (1920x1080 to 3840x2160, FP16: 183 us), a third of them on what its neighbours computed too. So what depends on an
// input texel only -- the 3x3 moments, their square roots and divisions, the clip box -- is computed once an input
// texel (2), a quarter of the output's at twice the size; the horizontal lerps of the nine bilinear depth samples of the
// closest-depth search once an output column and input row; and the axes of the samples once a row and a column (1). The
// history's footprints are filtered from an LDS window (4, 5) as in taa_window.hip: 16 LDS reads of 8 or 12 bytes a
// texel instead of 8 or 16 vector loads of 16, and 54 to 82 VGPRs where holding footprints took 111 to 139. A thread's
// rows share its column's tables and feed the CAS from registers.
// us a frame with CAS, before and now: FP16 on FP16 storage 1920x1080 to 3840x2160 183 and 114, 1280x720 to 1920x1080
// 47.4 and 37.8, 320x180 to 640x360 10.5 and 9.6; exact on FP32 storage 1281x721 to 1921x1081 66 and 55; exact on FP16
// storage 1920x1080 to 3840x2160 235 and 156.
// Measured and not kept: FP32 window texels of 16 bytes (1281x721: 59 us; LDS for four workgroups a CU instead of
// six); depth samples as float4 rows (four-row tiles of the 4K frame 132 us against 121); window loads inside a branch
// (each waits for the one before it, 59 us against 55).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "taa_device.hpp"
#include "taa_fast_math.hpp"
#include "taa_internal.hpp"
#include "taa_wave.hpp"

namespace taastar {
namespace {

// A workgroup of 256 threads resolves a region of 32 columns x 8 RPT rows, RPT rows of one column a thread; with fused
// CAS its outermost ring belongs to the neighbouring tiles.
template <int RPT_, bool CAS_, bool S16_, bool FA_>
struct UpGeo {
    static constexpr bool CAS = CAS_, S16 = S16_, FA = FA_;
    static constexpr int NT = 256, RPT = RPT_, RW = 32, RH = NT / 32 * RPT, RA = CAS ? 1 : 0, TW = RW - 2 * RA, TH = RH - 2 * RA;
    typedef typename std::conditional<S16, uint32_t, float2>::type VelT;  // staged velocity: the image's texel
    typedef typename std::conditional<S16, uint2, float4>::type Tex;      // a colour texel; a resolved texel for the CAS
    static constexpr int TB = (int)sizeof(Tex);
    // history window: rows of WP texels (FP32 ones without their alpha), 16 bytes of the image a lane, WR rows a pass
    struct Rgb {
        float x, y, z;
    };
    typedef typename std::conditional<S16, uint2, Rgb>::type Win;
    static constexpr int WP = kUpWindowCols, WH = RH + kUpWindowRows, WL = WP * TB / 16, WR = NT / WL, WN = (RH + 3 + WR - 1) / WR;
    struct Tables {  // per column (0 .. 31) and row (32 ..) of the region
        float uv[RW + RH];        // its uv
        int a[3][RW + RH];        // bilinear axis of SAMPLE_TEX at uv + (q - 1) input texels: the first tap's position in the
        float t[3][RW + RH];      // staged rectangle, the second tap's weight
        int pick[RW + RH];        // position of getCurrentUpsampledColor's input texel, -1: none
        int lo[RW + RH];          // position of the input texel int(uv * input size)
        alignas(16) int4 box[NT / 64];
    };
};

// a resolve texel between its history position and its blend
struct UpTexel {
    float fx, fy, expected, pd, hu, hv;
    f3 cur;
    bool found, outside;
    int kx, ky, k;
};

__device__ __forceinline__ float2 up_vel(uint32_t v) { return make_float2(lo16(v), hi16(v)); }
__device__ __forceinline__ float2 up_vel(float2 v) { return v; }

template <class G>
__device__ __forceinline__ void resolve_upscale(const FrameDesc& fd, const taa_uniforms_t& U, int tile, unsigned char* lds, typename G::Tables& tb) {
    typedef typename G::VelT VelT;
    typedef typename G::Tex Tex;
    constexpr bool S16 = G::S16, FA = G::FA;
    constexpr int RPT = G::RPT, RW = G::RW, RH = G::RH;
    const taa_params_t& P = U.param[fd.param_idx];
    const int W = fd.W, H = fd.H, Wl = fd.Wl, Hl = fd.Hl;
    const uint32_t pitch = (uint32_t)fd.pitch, pl = (uint32_t)fd.pitch_l;
    const int ty = scalar(tile / fd.tiles_x), tx = tile - ty * fd.tiles_x;
    const int x0 = fd.x_begin + tx * G::TW - G::RA, y0 = ty * G::TH - G::RA;  // the region's first texel
    const int tid = (int)threadIdx.x, rx = tid & 31, rg = (tid >> 5) * RPT;
    const float gamma = scalar_now(P.mVarClipGamma), a_max = scalar_now(P.mMaxAlpha), a_min = scalar_now(P.mMinAlpha),
                a_reject = scalar_now(P.mRejectionAlpha), peak = scalar_now(__uint_as_float(fd.cas_peak_bits));
    const float near = scalar_now(U.mCamNearPlane), far = scalar_now(U.mCamFarPlane), lin_thr = scalar_now(U.pad1);
    const bool reset = flag(U.mResetHistory), upsampling = flag(U.mUpsampling);
    const float fW = (float)W, fH = (float)H, fWl = (float)Wl, fHl = (float)Hl;
    const Image color(fd.color, fd.pitch_l, Wl, Hl, G::TB), depths(fd.depth, fd.pitch_l, Wl, Hl, 4),
        velocity(fd.velocity, fd.pitch_l, Wl, Hl, (int)sizeof(VelT)), history(fd.history, fd.pitch, W, H, G::TB), hdepth(fd.hdepth, fd.pitch_l, Wl, Hl, 4);

    // ---- 1. tables of the region's columns and rows (one axis an offset and wave), and the rectangle of input texels
    // under the region, three more on every side: every input texel that a resolved texel reads lies within two of its
    // own int(uv * input size) (the neighbourhood at +-1, the bilinear taps at uv +- one input texel, the upsampled
    // sample within the output texel), and that position grows with the output column and row
    int ox, oy, w, h;
    {
        const int q = scalar(tid >> 6), j = tid & 63;
        const bool col = j < 32, used = j < RW + RH;
        const int c = col ? clampi(x0 + j, 0, W - 1) : clampi(y0 + j - 32, 0, H - 1);
        const float n_out = col ? fW : fH, n_in = col ? fWl : fHl;
        const int n = col ? Wl : Hl;
        const float uv = ((float)c + 0.5f) / n_out;  // tc_to_uv (taa.comp:131)
        const int lo = to_int(uv * n_in);
        ox = __builtin_amdgcn_readlane(lo, 0) - 3;
        oy = __builtin_amdgcn_readlane(lo, 32) - 3;
        w = __builtin_amdgcn_readlane(lo, 31) - ox + 4;
        h = __builtin_amdgcn_readlane(lo, 31 + RH) - oy + 4;
        const int o = col ? ox : oy;
        if (q < 3) {
            const float to_u = col ? fd.to_u[0] : fd.to_u[1];  // 1 / input size
            int first;
            const BilinearAxis ba = bilinear_axis(n, uv + to_u * (float)(q - 1), &first);
            if (used) {
                tb.a[q][j] = first - o;
                tb.t[q][j] = ba.t;
                if (q == 0) {
                    tb.uv[j] = uv;
                    tb.lo[j] = lo - o;
                }
            }
        } else {
            const float ju = U.mJitterNdc[0] * 0.5f * P.mUnjitterFactor, jv = U.mJitterNdc[1] * 0.5f * P.mUnjitterFactor;
            const float tj = (col ? ju : jv) * n_in * -1.0f;
            const int p = upsample_pick(n_in, n_out, col ? fd.up_scale[0] : fd.up_scale[1], tj, c, n, col);
            if (used) tb.pick[j] = p < 0 ? -1 : p - o;
        }
    }
    const int n = w * h, bw = w - 6, nb = bw * (h - 6);
    // LDS: the rectangle's horizontal depth samples, colour, depth and velocity, then the history window in their place;
    // behind both the boxes of the rectangle's inner texels
    float* const hs = reinterpret_cast<float*>(lds);  // a row of the rectangle: three samples of each of the region's 32 columns
    float2* const c01 = reinterpret_cast<float2*>(hs + 96 * h);
    VelT* const sv = reinterpret_cast<VelT*>(c01 + n);
    float* const c2 = reinterpret_cast<float*>(sv + n);
    float* const sd = c2 + n;
    typename G::Win* const win = reinterpret_cast<typename G::Win*>(lds);
    float4* const box0 = reinterpret_cast<float4*>(lds + up_box_offset(w, h, G::RPT, S16));  // clip centre, first half size
    float2* const box1 = reinterpret_cast<float2*>(box0 + nb);                               // the other two
    {
        // a texel a lane, whole rows of the rectangle a pass: a lane keeps its column
        const float inv_w = rcp_fast((float)w);
        const int per = scalar((int)(((float)G::NT + 0.5f) * inv_w)), sy = (int)(((float)tid + 0.5f) * inv_w), sx = tid - __mul24(sy, w);
        const uint32_t gx = (uint32_t)med3<0>(ox + sx, Wl - 1);  // (quotients: the fraction stays 0.5 / w off a whole number)
        constexpr int U2 = RPT == 4 ? 3 : 2;
        for (int first = 0; first < h; first += U2 * per) {
            const int r0 = scalar_now(first);  // (kept from becoming a running value of every address)
            Tex c[U2];
            uint32_t d[U2];
            VelT v[U2];
#pragma unroll
            for (int p = 0; p < U2; ++p) {
                const uint32_t g = (uint32_t)med3<0>(oy + r0 + p * per + sy, Hl - 1) * pl + gx;
                d[p] = depths.ld1(g * 4u, 0u);
                if constexpr (S16) {
                    c[p] = color.ld2(g * 8u, 0u);
                    v[p] = velocity.ld1(g * 4u, 0u);
                } else {
                    const u32x4 t = color.ld4(g * 16u, 0u);
                    c[p] = make_float4(__uint_as_float(t.x), __uint_as_float(t.y), __uint_as_float(t.z), 0.0f);
                    const uint2 u = velocity.ld2(g * 8u, 0u);
                    v[p] = make_float2(__uint_as_float(u.x), __uint_as_float(u.y));
                }
            }
#pragma unroll
            for (int p = 0; p < U2; ++p) {
                const int i = (r0 + p * per) * w + tid;
                if (sy >= per || r0 + p * per + sy >= h) continue;
                f3 t;
                if constexpr (S16) t = {lo16(c[p].x), hi16(c[p].x), lo16(c[p].y)};
                else t = {c[p].x, c[p].y, c[p].z};
                t = rgb_to_ycocg(t);
                c01[i] = make_float2(t.x, t.y);
                c2[i] = t.z;
                sd[i] = __uint_as_float(d[p]);
                sv[i] = v[p];
            }
        }
    }
    __syncthreads();

    // ---- 2. once per input texel what its output texels share: the clip box, and per output column the horizontal
    // lerps of the bilinear depth samples (the same operations on the same values as texel by texel)
    {
        const float inv_bw = rcp_fast((float)bw);
        for (int i = tid; i < nb; i += G::NT) {
            const int by = (int)(((float)i + 0.5f) * inv_bw), bx = i - by * bw;
            const int l = (by + 3) * w + bx + 3;
            auto at = [&](int o) { return f3{c01[l + o].x, c01[l + o].y, c2[l + o]}; };
            const f3 c[9] = {at(0), at(-w - 1), at(-w), at(-w + 1), at(-1), at(1), at(w - 1), at(w), at(w + 1)};
            f3 p, e;
            if constexpr (FA) {
                f3 m1 = c[0], m2 = c[0] * c[0];
#pragma unroll
                for (int k = 1; k < 9; ++k) {
                    m1 = m1 + c[k];
                    m2 = {__builtin_fmaf(c[k].x, c[k].x, m2.x), __builtin_fmaf(c[k].y, c[k].y, m2.y), __builtin_fmaf(c[k].z, c[k].z, m2.z)};
                }
                constexpr float inv9 = 1.0f / 9.0f;
                const f3 mean = m1 * inv9;
                const f3 sigma = {sqrt_fast(fmaxf(__builtin_fmaf(-mean.x, mean.x, m2.x * inv9), 0.0f)),
                                  sqrt_fast(fmaxf(__builtin_fmaf(-mean.y, mean.y, m2.y * inv9), 0.0f)),
                                  sqrt_fast(fmaxf(__builtin_fmaf(-mean.z, mean.z, m2.z * inv9), 0.0f))};
                const f3 mn = {__builtin_fmaf(-gamma, sigma.x, mean.x), __builtin_fmaf(-gamma, sigma.y, mean.y), __builtin_fmaf(-gamma, sigma.z, mean.z)};
                const f3 mx = {__builtin_fmaf(gamma, sigma.x, mean.x), __builtin_fmaf(gamma, sigma.y, mean.y), __builtin_fmaf(gamma, sigma.z, mean.z)};
                p = {0.5f * (mx.x + mn.x), 0.5f * (mx.y + mn.y), 0.5f * (mx.z + mn.z)};  // clip_aabb_fast's centre and half size
                e = {__builtin_fmaf(0.5f, mx.x - mn.x, 1e-7f), __builtin_fmaf(0.5f, mx.y - mn.y, 1e-7f), __builtin_fmaf(0.5f, mx.z - mn.z, 1e-7f)};
            } else {
                const f3 m1 = c[0] + c[1] + c[2] + c[3] + c[4] + c[5] + c[6] + c[7] + c[8];
                const f3 m2 = c[0] * c[0] + c[1] * c[1] + c[2] * c[2] + c[3] * c[3] + c[4] * c[4] + c[5] * c[5] + c[6] * c[6] + c[7] * c[7] + c[8] * c[8];
                const f3 mean = {div9(m1.x), div9(m1.y), div9(m1.z)};
                const f3 var = f3{div9(m2.x), div9(m2.y), div9(m2.z)} - mean * mean;
                const f3 sigma = {sqrtf(fmaxf(0.0f, var.x)), sqrtf(fmaxf(0.0f, var.y)), sqrtf(fmaxf(0.0f, var.z))};
                const f3 mn = mean - gamma * sigma, mx = mean + gamma * sigma;
                p = 0.5f * (mx + mn);  // clipAabb's centre and half size (taa.comp:326-327)
                e = 0.5f * (mx - mn) + f3{1e-7f, 1e-7f, 1e-7f};
            }
            box0[i] = make_float4(p.x, p.y, p.z, e.x);
            box1[i] = make_float2(e.y, e.z);
        }
        int a[3];
        float t[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) a[q] = tb.a[q][rx], t[q] = tb.t[q][rx];
        for (int r = tid >> 5; r < h; r += G::NT / 32) {
            const float* d = sd + r * w;
            auto lerp = [&](int q) { return d[a[q]] * (1.0f - t[q]) + d[a[q] + 1] * t[q]; };
            #pragma unroll
            for (int q = 0; q < 3; ++q) hs[r * 96 + q * 32 + rx] = lerp(q);
        }
    }
    __syncthreads();

    // ---- 3. closest depth, history position, previous depth and current sample of the thread's texels
    UpTexel q[RPT];
    int bx0 = 0x7fffffff, by0 = 0x7fffffff, bx1 = -0x7fffffff, by1 = -0x7fffffff;
    {
        const float uvx = tb.uv[rx];
        const int lox = tb.lo[rx], pickx = tb.pick[rx];
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            const int r = 32 + rg + k;
            const float uvy = tb.uv[r];
            float ds[9];
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const float* p = hs + __mul24(tb.a[j][r], 96) + rx;
                const float t = tb.t[j][r], u = 1.0f - t;
#pragma unroll
                for (int i = 0; i < 3; ++i) ds[3 * j + i] = p[i * 32] * u + p[i * 32 + 96] * t;
            }
            float dmin = ds[0];  // findClosestUvAndZ_3x3 (taa.comp:371-389): scan order, strict <
            int best = 0;
#pragma unroll
            for (int j = 1; j < 9; ++j) {
                const bool c = ds[j] < dmin;
                dmin = c ? ds[j] : dmin;
                best = c ? j : best;
            }
            const int vj = (best * 11) >> 5, vi = best - 3 * vj;
            const int ax = tb.a[vi][rx], ay = tb.a[vj][r];
            const float vtx = tb.t[vi][rx], vty = tb.t[vj][r], vux = 1.0f - vtx, vuy = 1.0f - vty;
            const VelT* v = sv + __mul24(ay, w) + ax;
            const float2 va = up_vel(v[0]), vb = up_vel(v[1]), vc = up_vel(v[w]), vd = up_vel(v[w + 1]);
            const float hu = uvx - ((va.x * vux + vb.x * vtx) * vuy + (vc.x * vux + vd.x * vtx) * vty);
            const float hv = uvy - ((va.y * vux + vb.y * vtx) * vuy + (vc.y * vux + vd.y * vtx) * vty);
            const int l = __mul24(tb.lo[r], w) + lox;
            q[k].expected = sd[l];
            q[k].hu = hu;
            q[k].hv = hv;
            // the previous depth under the history position (taa.comp:818)
            q[k].pd = __uint_as_float(hdepth.ld1(((uint32_t)med3<0>(to_int(hv * fHl), Hl - 1) * pl + (uint32_t)med3<0>(to_int(hu * fWl), Wl - 1)) * 4u, 0u));
            // current colour: the texel itself, or getCurrentUpsampledColor's (taa.comp:222-257, 750-755)
            const int picky = tb.pick[r];
            q[k].found = !upsampling || (pickx >= 0 && picky >= 0);
            const int li = upsampling && q[k].found ? __mul24(picky, w) + pickx : l;
            const float2 cc = c01[li];
            q[k].cur = {cc.x, cc.y, c2[li]};
            // history position: base texel and fraction (taa.comp:456-462)
            const float sX = hu * fW, sY = hv * fH;
            const float fbx = floorf(sX - 0.5f), fby = floorf(sY - 0.5f);
            if constexpr (FA) {
                q[k].fx = (sX - 0.5f) - fbx;
                q[k].fy = (sY - 0.5f) - fby;
            } else {
                q[k].fx = sX - (fbx + 0.5f);
                q[k].fy = sY - (fby + 0.5f);
            }
            q[k].kx = med3<-2>(to_int(fbx), W + 1);  // cr_base
            q[k].ky = med3<-2>(to_int(fby), H + 1);
            bx0 = min(bx0, q[k].kx), by0 = min(by0, q[k].ky), bx1 = max(bx1, q[k].kx), by1 = max(by1, q[k].ky);
        }
    }
    const int4 wb = wave_min(make_int4(bx0, by0, -bx1, -by1));
    if ((tid & 63) == 0) tb.box[tid >> 6] = wb;
#pragma unroll
    for (int k = 0; k < RPT; ++k) q[k].outside = false;
    // positions outside the image: none in a wave whose bases all lie in 0 .. size - 2
    if (wb.x < 0 || wb.y < 0 || wb.z < 2 - W || wb.w < 2 - H) {
#pragma unroll
        for (int k = 0; k < RPT; ++k) q[k].outside = q[k].hu < 0.0f || q[k].hv < 0.0f || q[k].hu >= 1.0f || q[k].hv >= 1.0f;
    }
    __syncthreads();
    int4 b = tb.box[0];
#pragma unroll
    for (int i = 1; i < G::NT / 64; ++i) {
        const int4 o = tb.box[i];
        b = make_int4(min(b.x, o.x), min(b.y, o.y), min(b.z, o.z), min(b.w, o.w));
    }
    // ---- 4. the history window: taps k - 1 .. k + 2 of every footprint, clamped to the edge
    const int wx0 = scalar(b.x) - 1, wy0 = scalar(b.y) - 1;
    const int ww = -scalar(b.z) - scalar(b.x) + 4, wh = -scalar(b.w) - scalar(b.y) + 4;
    const bool fits = ww <= G::WP && wh <= G::WH;
    typedef typename G::Win Win;
    auto put = [&](int i, u32x4 t) {  // the i-th 16 bytes of the window's texels
        if constexpr (S16) reinterpret_cast<u32x4*>(win)[i] = t;
        else win[i] = Win{__uint_as_float(t.x), __uint_as_float(t.y), __uint_as_float(t.z)};
    };
    auto tap = [&](int x, int y) {  // one texel of the history, clamped
        const uint32_t o = ((uint32_t)clampi(y, 0, H - 1) * pitch + (uint32_t)clampi(x, 0, W - 1)) * (uint32_t)G::TB;
        if constexpr (S16) {
            return history.ld2(o, 0u);
        } else {
            const u32x4 t = history.ld4(o, 0u);
            return Win{__uint_as_float(t.x), __uint_as_float(t.y), __uint_as_float(t.z)};
        }
    };
    if (fits) {
        constexpr int L = 16 / G::TB;  // texels a lane
        const int row = tid / G::WL, col = L * (tid - row * G::WL);
        if (wx0 >= 0 && wy0 >= 0 && wx0 + ww + L - 1 <= W && wy0 + wh <= H) {
            const uint32_t o = ((uint32_t)row * pitch + (uint32_t)col) * (uint32_t)G::TB;
            const uint32_t s0 = ((uint32_t)wy0 * pitch + (uint32_t)wx0) * (uint32_t)G::TB;
            const bool take = tid < G::WL * G::WR && col < ww;
            u32x4 v[G::WN];  // (no load in a branch: the others would wait for it. An offset past the image reads nothing)
#pragma unroll
            for (int p = 0; p < G::WN; ++p)
                v[p] = history.ld4(take && row + p * G::WR < wh ? o : ~15u, s0 + (uint32_t)(p * G::WR) * pitch * (uint32_t)G::TB);
#pragma unroll
            for (int p = 0; p < G::WN; ++p)
                if (take && row + p * G::WR < wh) put(tid + p * G::WL * G::WR, v[p]);
            for (int p = G::WN; p * G::WR < wh; ++p)
                if (take && row + p * G::WR < wh)
                    put(tid + p * G::WL * G::WR, history.ld4(o, s0 + (uint32_t)(p * G::WR) * pitch * (uint32_t)G::TB));
        } else {
#pragma unroll 1
            for (int p = 0; p * G::WR < wh; ++p) {
                Win t[L];
#pragma unroll
                for (int i = 0; i < L; ++i) t[i] = tap(wx0 + col + i, wy0 + row + p * G::WR);
                if (tid < G::WL * G::WR && row + p * G::WR < wh) {
#pragma unroll
                    for (int i = 0; i < L; ++i) win[L * (tid + p * G::WL * G::WR) + i] = t[i];
                }
            }
        }
    }
#pragma unroll
    for (int k = 0; k < RPT; ++k) q[k].k = fits ? (q[k].ky - 1 - wy0) * G::WP + q[k].kx - 1 - wx0 : 0;
    __syncthreads();

    // ---- 5. history filter, rejection, clip and blend
    const uint32_t out_off = ((uint32_t)(y0 + rg) * pitch + (uint32_t)(x0 + rx)) * (uint32_t)G::TB;
    const bool own_col = x0 + rx < fd.x_end && (!G::CAS || (rx >= 1 && rx < 31));
    auto store = [&](void* im, const Tex& t, int k) { gstore<Tex>(im, out_off + (uint32_t)k * pitch * (uint32_t)G::TB, t); };
    const int lox = tb.lo[rx] - 3;
    Tex res[RPT];
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
        const int y = y0 + rg + k;
        const bool owned = own_col && (k > 0 || !G::CAS || rg > 0) && (k < RPT - 1 || !G::CAS || rg < RH - RPT) && y < H;
        const UpTexel& p = q[k];
        f3 acc = {0.f, 0.f, 0.f};
        W4 wx, wy;
        if constexpr (FA) {
            wx = cr_weights(p.fx), wy = cr_weights(p.fy);
        } else {
            auto weights = [](float f) {  // taa.comp:464-467 in source order
                const float f2 = f * f, f3_ = f2 * f;
                return W4{{-0.5f * f3_ + f2 - 0.5f * f, 1.5f * f3_ - 2.5f * f2 + 1.0f, -1.5f * f3_ + 2.0f * f2 + 0.5f * f, 0.5f * f3_ - 0.5f * f2}};
            };
            wx = weights(p.fx), wy = weights(p.fy);
        }
        auto add_row = [&](const Win (&e)[4], float wj, bool first) {
            if constexpr (FA) {
                f3 row = {0.f, 0.f, 0.f};
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    f3 t;
                    if constexpr (S16) t = {lo16(e[i].x), hi16(e[i].x), lo16(e[i].y)};
                    else t = {e[i].x, e[i].y, e[i].z};
                    row = {__builtin_fmaf(t.x, wx.w[i], row.x), __builtin_fmaf(t.y, wx.w[i], row.y), __builtin_fmaf(t.z, wx.w[i], row.z)};
                }
                acc = {__builtin_fmaf(row.x, wj, acc.x), __builtin_fmaf(row.y, wj, acc.y), __builtin_fmaf(row.z, wj, acc.z)};
            } else {  // texel * w_x * w_y summed tap by tap (taa.comp:480-495)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    f3 t;
                    if constexpr (S16) t = {mul_f16<false>(e[i].x, wx.w[i]), mul_f16<true>(e[i].x, wx.w[i]), mul_f16<false>(e[i].y, wx.w[i])};
                    else t = f3{e[i].x, e[i].y, e[i].z} * wx.w[i];
                    t = t * wj;
                    acc = i == 0 && first ? t : acc + t;
                }
            }
        };
        if (fits) {
            const Win* t = win + p.k;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const Win e[4] = {t[j * G::WP], t[j * G::WP + 1], t[j * G::WP + 2], t[j * G::WP + 3]};
                add_row(e, wy.w[j], j == 0);
            }
        } else {  // the tile's footprints lie too far apart for the window: texel by texel from memory
#pragma unroll 1
            for (int j = 0; j < 4; ++j) {
                Win e[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) e[i] = tap(p.kx - 1 + i, p.ky - 1 + j);
                const float wj = j == 0 ? wy.w[0] : j == 1 ? wy.w[1] : j == 2 ? wy.w[2] : wy.w[3];
                if (FA || j > 0) add_row(e, wj, false);
                else add_row(e, wj, true);
            }
        }
        f3 hc = rgb_to_ycocg(acc);
        // rejection (taa.comp:787-823)
        bool rejected = p.outside;
        if (lin_thr > 0.0f ? linear_depth_reject(p.pd, p.expected, near, far, lin_thr) : fabsf(p.pd - p.expected) > 0.1f * (1.0f - p.pd)) rejected = true;
        // clipAabb (taa.comp:323-345) in the box of the texel's input texel
        {
            const int i = __mul24(tb.lo[32 + rg + k] - 3, bw) + lox;
            const float4 b0 = box0[i];
            const float2 b1 = box1[i];
            const f3 c = {b0.x, b0.y, b0.z}, e = {b0.w, b1.x, b1.y}, v = hc - c;
            if constexpr (FA) {  // one reciprocal: ma = M / D
                const float exy = e.x * e.y, D = exy * e.z;
                const float M = fmaxf(fabsf(v.x) * (e.y * e.z), fmaxf(fabsf(v.y) * (e.x * e.z), fabsf(v.z) * exy));
                if (M > D) {
                    const float s = D * rcp_fast(M);
                    hc = {__builtin_fmaf(v.x, s, c.x), __builtin_fmaf(v.y, s, c.y), __builtin_fmaf(v.z, s, c.z)};
                }
            } else {
                const f3 u = v / e;
                const float ma = fmaxf(fabsf(u.x), fmaxf(fabsf(u.y), fabsf(u.z)));
                if (ma > 1.0f) hc = c + v / ma;
            }
        }
        // blend (taa.comp:850-900)
        f3 cur = p.cur;
        if (!p.found) cur = {0.f, 0.f, 0.f};
        const float lc = cur.x, lh = hc.x;
        const float ld = fmaxf(fmaxf(lc, lh), 0.2f);
        const float diff = FA ? fabsf(lc - lh) * rcp_fast(ld) : fabsf(lc - lh) / ld;
        const float wl = 1.0f - diff;
        float ab = gmix(a_max, a_min, wl * wl);
        if (!p.found) ab = ab * 0.0f;  // alpha * beta: beta is 0 where no sample was found, unless rejected or reset
        if (rejected) ab = a_reject;
        if (reset) ab = 1.0f;
        f3 aa;
        if constexpr (FA)
            aa = {__builtin_fmaf(ab, cur.x - hc.x, hc.x), __builtin_fmaf(ab, cur.y - hc.y, hc.y), __builtin_fmaf(ab, cur.z - hc.z, hc.z)};
        else
            aa = {gmix(hc.x, cur.x, ab), gmix(hc.y, cur.y, ab), gmix(hc.z, cur.z, ab)};
        aa = ycocg_to_rgb(aa);
        if constexpr (S16) {
            const uint32_t rgb0 = pack_sat(aa.z, 0.0f);
            res[k] = make_uint2(pack_sat(aa.x, aa.y), rgb0);
            if (owned) {
                store(fd.history_out, res[k], k);
                if constexpr (!G::CAS) store(fd.screen, make_uint2(res[k].x, rgb0 | 0x3c000000u), k);
            }
        } else {
            res[k] = make_float4(aa.x, aa.y, aa.z, 0.0f);
            if (owned) {
                store(fd.history_out, res[k], k);
                if constexpr (!G::CAS) store(fd.screen, make_float4(aa.x, aa.y, aa.z, 1.0f), k);
            }
        }
    }

    // ---- 6. fused CAS: left and right neighbours from LDS, upper and lower ones of the thread's own column where it
    // has them; at the image's border the missing neighbour is the texel itself
    if constexpr (G::CAS) {
        __syncthreads();  // every thread is done with the window
        Tex* const rs = reinterpret_cast<Tex*>(lds);
#pragma unroll
        for (int k = 0; k < RPT; ++k) rs[(rg + k) * 32 + rx] = res[k];
        __syncthreads();
        const int x = x0 + rx;
        const bool border = x0 < 0 || y0 < 0 || x0 + RW >= W || y0 + RH >= H;
        if (!own_col) return;
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            const int ry = rg + k, y = y0 + ry;
            if ((k == 0 && rg == 0) || (k == RPT - 1 && rg == RH - RPT) || y >= H) continue;
            const Tex c = res[k];
            Tex l = rs[ry * 32 + rx - 1], r = rs[ry * 32 + rx + 1];
            Tex u = k > 0 ? res[k > 0 ? k - 1 : 0] : rs[(ry - 1) * 32 + rx], d = k < RPT - 1 ? res[k < RPT - 1 ? k + 1 : 0] : rs[(ry + 1) * 32 + rx];
            if (border) {
                if (x == 0) l = c;
                if (x == W - 1) r = c;
                if (y == 0) u = c;
                if (y == H - 1) d = c;
            }
            if constexpr (FA && S16) {
                store(fd.screen, cas_filter_h2(u, l, c, r, d, peak), k);
            } else {
                auto rgb = [](const Tex& t) {
                    if constexpr (S16) return f3{lo16(t.x), hi16(t.x), lo16(t.y)};
                    else return f3{t.x, t.y, t.z};
                };
                const f3 o = FA ? cas_filter_fma(rgb(u), rgb(l), rgb(c), rgb(r), rgb(d), peak) : cas_filter(rgb(u), rgb(l), rgb(c), rgb(r), rgb(d), peak);
                if constexpr (S16) store(fd.screen, make_uint2(pack_sat(o.x, o.y), pack_sat(o.z, 1.0f)), k);
                else store(fd.screen, make_float4(o.x, o.y, o.z, 1.0f), k);
            }
        }
    }
}

struct ResolveArgs {
    FrameDesc fd;
    taa_uniforms_t U;
};

constexpr int kUpWaves = 4;  // occupancy hint (waves per SIMD): registers leave six and more, LDS four to seven
constexpr int kLdsOfFive = 160 * 1024 / 5;

template <int RPT, bool CAS, bool S16, bool FA>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kUpWaves))) void k_resolve_upscale(const ResolveArgs a) {
    using G = UpGeo<RPT, CAS, S16, FA>;
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ typename G::Tables tb;
    resolve_upscale<G>(a.fd, a.U, xcd_tile((int)blockIdx.x, a.fd.tiles_x * a.fd.tiles_y), lds, tb);
}

// the frames of a batch, walked like the other batched kernels
template <int RPT, bool CAS, bool S16, bool FA>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kUpWaves))) void k_resolve_upscale_batch(const BatchEntry* __restrict__ entries, int n_entries, int total) {
    using G = UpGeo<RPT, CAS, S16, FA>;
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ typename G::Tables tb;
    const int t = batch_tile(total);
    if (t < 0) return;
    const BatchEntry& e = batch_entry(entries, n_entries, t);
    resolve_upscale<G>(e.fd, e.U, t - e.tile_begin, lds, tb);
}

template <int RPT, bool CAS, bool S16, bool FA>
void launch_t(const ResolveArgs& a, int lds, hipStream_t st) {
    hipLaunchKernelGGL((k_resolve_upscale<RPT, CAS, S16, FA>), dim3(a.fd.tiles_x * a.fd.tiles_y), dim3(256), (size_t)lds, st, a);
}
template <int RPT, bool CAS, bool S16, bool FA>
void launch_batch_t(const BatchEntry* e, int n, int total, int lds, hipStream_t st) {
    hipLaunchKernelGGL((k_resolve_upscale_batch<RPT, CAS, S16, FA>), dim3(batch_grid(total)), dim3(256), (size_t)lds, st, e, n, total);
}

// f<RPT, CAS, S16, FA>(args...) for run-time values
#define TAA_UP_SWITCH(F, ...)                                                                                              \
    do {                                                                                                                   \
        const int form = (cas ? 4 : 0) | (s16 ? 2 : 0) | (fa ? 1 : 0);                                                     \
        switch (form) {                                                                                                    \
            case 0: rows == 4 ? F<4, false, false, false>(__VA_ARGS__) : F<2, false, false, false>(__VA_ARGS__); break;    \
            case 1: rows == 4 ? F<4, false, false, true>(__VA_ARGS__) : F<2, false, false, true>(__VA_ARGS__); break;      \
            case 2: rows == 4 ? F<4, false, true, false>(__VA_ARGS__) : F<2, false, true, false>(__VA_ARGS__); break;      \
            case 3: rows == 4 ? F<4, false, true, true>(__VA_ARGS__) : F<2, false, true, true>(__VA_ARGS__); break;        \
            case 4: rows == 4 ? F<4, true, false, false>(__VA_ARGS__) : F<2, true, false, false>(__VA_ARGS__); break;      \
            case 5: rows == 4 ? F<4, true, false, true>(__VA_ARGS__) : F<2, true, false, true>(__VA_ARGS__); break;        \
            case 6: rows == 4 ? F<4, true, true, false>(__VA_ARGS__) : F<2, true, true, false>(__VA_ARGS__); break;        \
            default: rows == 4 ? F<4, true, true, true>(__VA_ARGS__) : F<2, true, true, true>(__VA_ARGS__); break;         \
        }                                                                                                                  \
    } while (0)

}  // namespace

bool upscale_form(const FrameDesc& fd, const taa_uniforms_t& U) {
    const long long out = (long long)fd.W * fd.H, in = (long long)fd.Wl * fd.Hl;
    return fd.Wl <= fd.W && fd.Hl <= fd.H && out * 10 >= in * (fd.color_fmt == TAA_FMT_RGBA16F ? 14 : 16) && prod_params(fd, U);
}

int upscale_lds(const FrameDesc& fd, int rows) {
    // 31 output columns span 31 Wl / W input texels, their floors at most one more, seven with the border; 1/16 covers
    // the rounding of uv * size (below 0.01 texels at 32768)
    const int w = (int)((31LL * 16 * fd.Wl + fd.W) / (16LL * fd.W)) + 8, h = (int)(((8LL * rows - 1) * 16 * fd.Hl + fd.H) / (16LL * fd.H)) + 8;
    return up_box_offset(w, h, rows, fd.color_fmt == TAA_FMT_RGBA16F) + 24 * (w - 6) * (h - 6);
}

int upscale_rows(long long n4, int lds4) { return n4 >= 5 * 256 && lds4 <= kLdsOfFive - (int)sizeof(UpGeo<4, true, true, true>::Tables) ? 4 : 2; }

int launch_upscale(const FrameDesc& fd, const taa_uniforms_t& U, int arith, void* stream) {
    hipStream_t st = static_cast<hipStream_t>(stream);
    ResolveArgs a;
    a.fd = fd;
    a.U = U;
    const bool cas = fd.cas_on != 0, s16 = fd.color_fmt == TAA_FMT_RGBA16F, fa = arith == TAA_ARITH_FP16;
    tile_upscale(a.fd, 4);
    const int rows = upscale_rows((long long)a.fd.tiles_x * a.fd.tiles_y, upscale_lds(fd, 4));
    tile_upscale(a.fd, rows);
    const int lds = upscale_lds(fd, rows);
    TAA_UP_SWITCH(launch_t, a, lds, st);
    return (int)hipGetLastError();
}

int launch_upscale_batch(const BatchEntry* e, int n, int total, int rows, int lds, bool cas, bool s16, int arith, void* stream) {
    hipStream_t st = static_cast<hipStream_t>(stream);
    const bool fa = arith == TAA_ARITH_FP16;
    TAA_UP_SWITCH(launch_batch_t, e, n, total, lds, st);
    return (int)hipGetLastError();
}

}  // namespace taastar
