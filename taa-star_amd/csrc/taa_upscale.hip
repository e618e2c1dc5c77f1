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
// history's footprints are filtered from an LDS window (taa_production.hpp) as in taa_window.hip: 16 LDS reads of 8 or 12 bytes a
// texel instead of 8 or 16 vector loads of 16, and 53 to 85 VGPRs where holding footprints took 111 to 139. A thread's
// rows share its column's tables and feed the CAS from registers.
// us a frame with CAS, before and now: FP16 on FP16 storage 1920x1080 to 3840x2160 183 and 114, 1280x720 to 1920x1080
// 47.3 and 33.4, 320x180 to 640x360 10.5 and 9.0; exact on FP32 storage 1281x721 to 1921x1081 66 and 54; exact on FP16
// storage 1920x1080 to 3840x2160 235 and 156.
// Measured and not kept: FP32 window texels of 16 bytes (1281x721: 59 us; LDS for four workgroups a CU instead of
// six); depth samples as float4 rows (four-row tiles of the 4K frame 132 us against 121); window loads inside a branch
// (each waits for the one before it, 59 us against 55).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "taa_device.hpp"
#include "taa_fast_math.hpp"
#include "taa_internal.hpp"
#include "taa_production.hpp"
#include "taa_wave.hpp"

namespace taastar {
namespace {

template <int NT, int RPT, bool CAS, bool S16, bool FA>
struct UpGeo : ProdGeo<NT, RPT, CAS, S16, FA> {
    typedef ProdGeo<NT, RPT, CAS, S16, FA> Base;
    static constexpr int RW = Base::RW, RH = Base::RH;
    struct Tables {  // per column (0 .. 31) and row (32 ..) of the region
        float uv[RW + RH];        // its uv
        int a[3][RW + RH];        // bilinear axis of SAMPLE_TEX at uv + (q - 1) input texels: the first tap's position in the
        float t[3][RW + RH];      // staged rectangle, the second tap's weight
        int pick[RW + RH];        // position of getCurrentUpsampledColor's input texel, -1: none
        int lo[RW + RH];          // position of the input texel int(uv * input size)
        alignas(16) int4 box[NT / 64];
    };
};

template <class G>
__device__ __forceinline__ void resolve_upscale(const FrameDesc& fd, const taa_uniforms_t& U, int tile, unsigned char* lds, typename G::Tables& tb) {
    typedef typename G::VelT VelT;
    typedef typename G::Tex Tex;
    constexpr bool S16 = G::S16, FA = G::FA;
    constexpr int RPT = G::RPT, RW = G::RW, RH = G::RH;
    const taa_params_t& P = U.param[fd.param_idx];
    const int W = fd.W, H = fd.H, Wl = fd.Wl, Hl = fd.Hl;
    const uint32_t pl = (uint32_t)fd.pitch_l;
    const int ty = scalar(tile / fd.tiles_x), tx = tile - ty * fd.tiles_x;
    const int x0 = fd.x_begin + tx * G::TW - G::RA, y0 = ty * G::TH - G::RA;  // the region's first texel
    const int tid = (int)threadIdx.x, rx = tid & 31, rg = (tid >> 5) * RPT;
    const float gamma = scalar_now(P.mVarClipGamma);
    const bool upsampling = flag(U.mUpsampling);
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
        } else if (q == 3) {
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
    float4* const box0 = reinterpret_cast<float4*>(lds + up_box_offset(w, h, RH, S16));  // clip centre, first half size
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
                fast_box(m1, m2, gamma, p, e);
            } else {
                f3 m1 = c[0] + c[1] + c[2] + c[3] + c[4] + c[5] + c[6] + c[7] + c[8];
                f3 m2 = c[0] * c[0] + c[1] * c[1] + c[2] * c[2] + c[3] * c[3] + c[4] * c[4] + c[5] * c[5] + c[6] * c[6] + c[7] * c[7] + c[8] * c[8];
                div9_moments(m1, m2);
                const f3 mean = m1, var = m2 - mean * mean;
                const f3 sigma = sqrt3({fmaxf(0.0f, var.x), fmaxf(0.0f, var.y), fmaxf(0.0f, var.z)});
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
    ProdTexel q[RPT];
    f3 cur[RPT];
    bool found[RPT];
    int4 bases = make_int4(0x7fffffff, 0x7fffffff, 0x7fffffff, 0x7fffffff);
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
            const float2 va = vel_xy(v[0]), vb = vel_xy(v[1]), vc = vel_xy(v[w]), vd = vel_xy(v[w + 1]);
            const float hu = uvx - ((va.x * vux + vb.x * vtx) * vuy + (vc.x * vux + vd.x * vtx) * vty);
            const float hv = uvy - ((va.y * vux + vb.y * vtx) * vuy + (vc.y * vux + vd.y * vtx) * vty);
            const int l = __mul24(tb.lo[r], w) + lox;
            q[k].expected = sd[l];
            q[k].hu = hu;
            q[k].hv = hv;
            q[k].masked = false;
            // the previous depth under the history position (taa.comp:818)
            q[k].pd = __uint_as_float(hdepth.ld1(((uint32_t)med3<0>(to_int(hv * fHl), Hl - 1) * pl + (uint32_t)med3<0>(to_int(hu * fWl), Wl - 1)) * 4u, 0u));
            // current colour: the texel itself, or getCurrentUpsampledColor's (taa.comp:222-257, 750-755)
            const int picky = tb.pick[r];
            found[k] = !upsampling || (pickx >= 0 && picky >= 0);
            const int li = upsampling && found[k] ? __mul24(picky, w) + pickx : l;
            const float2 cc = c01[li];
            cur[k] = {cc.x, cc.y, c2[li]};
            history_base<FA>(q[k], W, H, bases);
        }
    }
    // the clip box of the texel's input texel, and its current colour
    const int lox = tb.lo[rx] - 3;
    auto box = [&](int k, f3& c, f3& e, f3& now, bool& have) {
        const int i = __mul24(tb.lo[32 + rg + k] - 3, bw) + lox;
        const float4 b0 = box0[i];
        const float2 b1 = box1[i];
        c = {b0.x, b0.y, b0.z}, e = {b0.w, b1.x, b1.y};
        have = found[k];
        now = have ? cur[k] : f3{0.f, 0.f, 0.f};
    };
    finish<G>(fd, U, P, history, x0, y0, q, bases, lds, tb.box, box);
}

struct ResolveArgs {
    FrameDesc fd;
    taa_uniforms_t U;
};

constexpr int kUpWaves = 4;  // occupancy hint (waves per SIMD): registers leave six and more, LDS four to seven

template <class G>
__global__ __launch_bounds__(G::NT) __attribute__((amdgpu_waves_per_eu(kUpWaves))) void k_resolve_upscale(const ResolveArgs a) {
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ typename G::Tables tb;
    resolve_upscale<G>(a.fd, a.U, xcd_tile((int)blockIdx.x, a.fd.tiles_x * a.fd.tiles_y), lds, tb);
}

// the frames of a batch, walked like the other batched kernels
template <class G>
__global__ __launch_bounds__(G::NT) __attribute__((amdgpu_waves_per_eu(kUpWaves))) void k_resolve_upscale_batch(const BatchEntry* __restrict__ entries, int n_entries, int total) {
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ typename G::Tables tb;
    const int t = batch_tile(total);
    if (t < 0) return;
    const BatchEntry& e = batch_entry(entries, n_entries, t);
    resolve_upscale<G>(e.fd, e.U, t - e.tile_begin, lds, tb);
}

// f(geometry) for the variant's geometry
template <int NT, int RPT, class F>
void for_form(bool cas, bool s16, bool fa, F&& f) {
    if (cas) {
        if (s16) fa ? f(UpGeo<NT, RPT, true, true, true>()) : f(UpGeo<NT, RPT, true, true, false>());
        else fa ? f(UpGeo<NT, RPT, true, false, true>()) : f(UpGeo<NT, RPT, true, false, false>());
    } else {
        if (s16) fa ? f(UpGeo<NT, RPT, false, true, true>()) : f(UpGeo<NT, RPT, false, true, false>());
        else fa ? f(UpGeo<NT, RPT, false, false, true>()) : f(UpGeo<NT, RPT, false, false, false>());
    }
}
template <class F>
void for_geometry(int variant, bool cas, bool s16, bool fa, F&& f) {
    switch (variant) {
        case kProd512x1: for_form<512, 1>(cas, s16, fa, f); break;
        case kProd512x2: for_form<512, 2>(cas, s16, fa, f); break;
        case kProd256x4: for_form<256, 4>(cas, s16, fa, f); break;
        default: for_form<256, 2>(cas, s16, fa, f); break;
    }
}

}  // namespace

bool upscale_form(const FrameDesc& fd, const taa_uniforms_t& U) {
    if (fd.Wl > fd.W || fd.Hl > fd.H || !prod_params(fd, U)) return false;
    const long long out = (long long)fd.W * fd.H, in = (long long)fd.Wl * fd.Hl;
    if (fd.color_fmt == TAA_FMT_RGBA16F) return out * 10 >= in * 14;
    FrameDesc p = fd;
    tile_production(p, kProd256x2);
    const long long n16 = (long long)p.tiles_x * p.tiles_y;
    return out * 10 >= in * (n16 < 2500 ? 18 : 16) && (fd.cas_on || n16 >= 600);
}

int upscale_lds(const FrameDesc& fd, int variant) {
    // 31 output columns span 31 Wl / W input texels, their floors at most one more, seven with the border; 1/16 covers
    // the rounding of uv * size (below 0.01 texels at 32768)
    const int rows = production_rows(variant);
    const int w = (int)((31LL * 16 * fd.Wl + fd.W) / (16LL * fd.W)) + 8, h = (int)(((rows - 1LL) * 16 * fd.Hl + fd.H) / (16LL * fd.H)) + 8;
    return up_box_offset(w, h, rows, fd.color_fmt == TAA_FMT_RGBA16F) + 24 * (w - 6) * (h - 6);
}

int upscale_variant(long long n16, long long n32, int lds) {
    const int tables = (int)sizeof(UpGeo<256, 4, true, true, true>::Tables), cu = 160 * 1024;
    if (n16 < 800) return kProd512x1;
    if (n32 < 5 * 256 || lds + tables > cu / 3) return kProd256x2;
    return lds + tables <= cu / 5 ? kProd256x4 : kProd512x2;
}

int launch_upscale(const FrameDesc& fd, const taa_uniforms_t& U, int arith, void* stream) {
    hipStream_t st = static_cast<hipStream_t>(stream);
    ResolveArgs a;
    a.fd = fd;
    a.U = U;
    tile_production(a.fd, kProd256x2);
    const long long n16 = (long long)a.fd.tiles_x * a.fd.tiles_y;
    tile_production(a.fd, kProd256x4);
    tile_production(a.fd, upscale_variant(n16, (long long)a.fd.tiles_x * a.fd.tiles_y, upscale_lds(fd, kProd256x4)));
    const size_t lds = (size_t)upscale_lds(fd, a.fd.rows);
    for_geometry(a.fd.rows, fd.cas_on != 0, fd.color_fmt == TAA_FMT_RGBA16F, arith == TAA_ARITH_FP16, [&](auto g) {
        hipLaunchKernelGGL((k_resolve_upscale<decltype(g)>), dim3(a.fd.tiles_x * a.fd.tiles_y), dim3(decltype(g)::NT), lds, st, a);
    });
    return (int)hipGetLastError();
}

int launch_upscale_batch(const BatchEntry* e, int n, int total, int variant, int lds, bool cas, bool s16, int arith, void* stream) {
    hipStream_t st = static_cast<hipStream_t>(stream);
    for_geometry(variant, cas, s16, arith == TAA_ARITH_FP16, [&](auto g) {
        hipLaunchKernelGGL((k_resolve_upscale_batch<decltype(g)>), dim3(batch_grid(total)), dim3(decltype(g)::NT), (size_t)lds, st, e, n, total);
    });
    return (int)hipGetLastError();
}

}  // namespace taastar
