// The last phases of the kernels with the production feature set (taa_exact.hip, taa_upscale.hip): history window,
// Catmull-Rom filter, rejection, clip, blend and CAS of a workgroup's region. Exact FP32 arithmetic in the
// order of taa.comp, or with FA the FP16 path's.
#pragma once

#include <type_traits>

#include "taa_device.hpp"
#include "taa_fast_math.hpp"
#include "taa_internal.hpp"
#include "taa_wave.hpp"

namespace taastar {
namespace {

// A workgroup of NT threads resolves a region of 32 columns x NT / 32 * RPT rows, RPT rows of one column a thread; with fused
// CAS its outermost ring belongs to the neighbouring tiles.
template <int NT_, int RPT_, bool CAS_, bool S16_, bool FA_>
struct ProdGeo {
    static constexpr bool CAS = CAS_, S16 = S16_, FA = FA_;
    static constexpr bool PLAIN = false;  // without depth culling, Lottes weighting and outside rejection
    static constexpr int NT = NT_, RPT = RPT_, RW = 32, RH = NT / 32 * RPT, RA = CAS ? 1 : 0, TW = RW - 2 * RA, TH = RH - 2 * RA;
    typedef typename std::conditional<S16, uint32_t, float2>::type VelT;  // staged velocity: the image's texel
    typedef typename std::conditional<S16, uint2, float4>::type Tex;      // a colour texel; a resolved texel for the CAS
    static constexpr int TB = (int)sizeof(Tex);
    // history window: rows of WP texels (FP32 ones without their alpha), 16 bytes of the image a lane, WR rows a pass
    struct Rgb {
        float x, y, z;
    };
    typedef typename std::conditional<S16, uint2, Rgb>::type Win;
    // one row a thread, for frames that leave the device part empty, has no window: a texel's footprint is read from memory as soon
    // as its position is known, which saves two barriers and a round trip
    static constexpr bool WIN = RPT > 1;
    static constexpr int WP = kProdWindowCols, WH = RH + kProdWindowRows, WL = WP * TB / 16, WR = NT / WL, WN = (RH + 3 + WR - 1) / WR;
};

// a resolve texel between its history position and its blend
struct ProdTexel {
    float fx, fy, expected, pd, hu, hv;
    bool outside, masked;  // masked: rejected by the segmentation mask
    int kx, ky, k;
};

__device__ __forceinline__ float2 vel_xy(uint32_t v) { return make_float2(lo16(v), hi16(v)); }
__device__ __forceinline__ float2 vel_xy(float2 v) { return v; }

// m1 / 9 and m2 / 9 of a neighbourhood's sum and sum of squares, and the square roots of three values >= 0: div9 and the
// compiler's sqrtf, operation for operation, with one test for the six (three) instead of one each for the values
// that their steps do not cover. For div9 these are -0, which a sum of squares is not, and infinities: a sum that overflows, or
// holds one, has an infinite sum of squares. For the square root, values that it would scale up first.
// (About 40 and 60 issue clocks a wave less.)
__device__ __forceinline__ void div9_moments(f3& m1, f3& m2) {
    auto q = [](float x) {
        const float y = 1.0f / 9.0f, q0 = x * y;
        return __builtin_fmaf(__builtin_fmaf(-q0, 9.0f, x), y, q0);
    };
    const bool other = fmaxf(fmaxf(m2.x, m2.y), m2.z) == __builtin_inff() ||
                       min(min(__float_as_int(m1.x), __float_as_int(m1.y)), __float_as_int(m1.z)) == (int)0x80000000;
    if (other) {
        m1 = {div9(m1.x), div9(m1.y), div9(m1.z)};
        m2 = {div9(m2.x), div9(m2.y), div9(m2.z)};
    } else {
        m1 = {q(m1.x), q(m1.y), q(m1.z)};
        m2 = {q(m2.x), q(m2.y), q(m2.z)};
    }
}
__device__ __forceinline__ f3 sqrt3(f3 v) {
    auto root = [](float x) {  // the hardware's within one ulp, then the neighbour whose residual says so
        const float s = __builtin_amdgcn_sqrtf(x);
        const float down = __uint_as_float(__float_as_uint(s) - 1u), up = __uint_as_float(__float_as_uint(s) + 1u);
        const float a = __builtin_fmaf(-down, s, x), b = __builtin_fmaf(-up, s, x);
        const float t = a <= 0.0f ? down : s;
        return b > 0.0f ? up : t;
    };
    auto bits = [](float x) { return __float_as_uint(x) - 1u; };  // zero last
    if (min(min(bits(v.x), bits(v.y)), bits(v.z)) < __float_as_uint(0x1p-96f) - 1u) return {sqrtf(v.x), sqrtf(v.y), sqrtf(v.z)};
    return {root(v.x), root(v.y), root(v.z)};
}

// clip centre and half size of the FP16 path's box (clip_aabb_fast) from the 3x3 sums and sums of squares
__device__ __forceinline__ void fast_box(f3 m1, f3 m2, float gamma, f3& c, f3& e) {
    constexpr float inv9 = 1.0f / 9.0f;
    const f3 mean = m1 * inv9;
    const f3 sigma = {sqrt_fast(fmaxf(__builtin_fmaf(-mean.x, mean.x, m2.x * inv9), 0.0f)), sqrt_fast(fmaxf(__builtin_fmaf(-mean.y, mean.y, m2.y * inv9), 0.0f)),
                      sqrt_fast(fmaxf(__builtin_fmaf(-mean.z, mean.z, m2.z * inv9), 0.0f))};
    const f3 mn = {__builtin_fmaf(-gamma, sigma.x, mean.x), __builtin_fmaf(-gamma, sigma.y, mean.y), __builtin_fmaf(-gamma, sigma.z, mean.z)};
    const f3 mx = {__builtin_fmaf(gamma, sigma.x, mean.x), __builtin_fmaf(gamma, sigma.y, mean.y), __builtin_fmaf(gamma, sigma.z, mean.z)};
    c = {0.5f * (mx.x + mn.x), 0.5f * (mx.y + mn.y), 0.5f * (mx.z + mn.z)};
    e = {__builtin_fmaf(0.5f, mx.x - mn.x, 1e-7f), __builtin_fmaf(0.5f, mx.y - mn.y, 1e-7f), __builtin_fmaf(0.5f, mx.z - mn.z, 1e-7f)};
}

// history position of a texel: base texel and fraction (taa.comp:456-462), the base widening the bounds of the thread's
template <bool FA>
__device__ __forceinline__ void history_base(ProdTexel& q, int W, int H, int4& bases) {
    const float sX = q.hu * (float)W, sY = q.hv * (float)H;
    const float fbx = floorf(sX - 0.5f), fby = floorf(sY - 0.5f);
    if constexpr (FA) {
        q.fx = (sX - 0.5f) - fbx;
        q.fy = (sY - 0.5f) - fby;
    } else {
        q.fx = sX - (fbx + 0.5f);
        q.fy = sY - (fby + 0.5f);
    }
    q.kx = med3<-2>(to_int(fbx), W + 1);  // cr_base
    q.ky = med3<-2>(to_int(fby), H + 1);
    bases = make_int4(min(bases.x, q.kx), min(bases.y, q.ky), min(bases.z, -q.kx), min(bases.w, -q.ky));
}

// q: the thread's texels; bases: the least of their kx, ky, -kx, -ky; lds: the window's space, free after the first barrier here;
// box(k, c, e, cur, found): clip centre and half size of texel k, its current colour (zero unless found)
template <class G, class Box>
__device__ __forceinline__ void finish(const FrameDesc& fd, const taa_uniforms_t& U, const taa_params_t& P, const Image& history, int x0, int y0,
                                       ProdTexel (&q)[G::RPT], int4 bases, unsigned char* lds, int4* boxes, Box&& box) {
    typedef typename G::Tex Tex;
    constexpr bool S16 = G::S16, FA = G::FA;
    constexpr int RPT = G::RPT, RW = G::RW, RH = G::RH;
    const int W = fd.W, H = fd.H;
    const uint32_t pitch = (uint32_t)fd.pitch;
    const int tid = (int)threadIdx.x, rx = tid & 31, rg = (tid >> 5) * RPT;
    const float a_max = P.mMaxAlpha, a_min = P.mMinAlpha, a_reject = P.mRejectionAlpha, peak = __uint_as_float(fd.cas_peak_bits);
    const float near = U.mCamNearPlane, far = U.mCamFarPlane, lin_thr = U.pad1;
    const bool reset = U.mResetHistory != 0;
    typedef typename G::Win Win;
    Win* const win = reinterpret_cast<Win*>(lds);
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
    bool fits = false;
    Win foot[G::WIN ? 1 : RPT][16];  // without the window: the texels' footprints
    if constexpr (!G::WIN) {
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            q[k].outside = !G::PLAIN && (q[k].hu < 0.0f || q[k].hv < 0.0f || q[k].hu >= 1.0f || q[k].hv >= 1.0f);
            // from a base that keeps the footprint inside the image; a wave with one over its edge (or an image too small) reads
            // the texels one by one, clamped
            const int kx = q[k].kx - 1, ky = q[k].ky - 1, bx = max(min(kx, W - 4), 0), by = max(min(ky, H - 4), 0);
            const uint32_t o = ((uint32_t)by * pitch + (uint32_t)bx) * (uint32_t)G::TB;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t s = (uint32_t)min(j, H - 1) * pitch * (uint32_t)G::TB;
                if constexpr (S16) {
                    const u32x4 a = history.ld4(o, s), b = history.ld4(o + 16u, s);
                    foot[k][4 * j] = make_uint2(a.x, a.y), foot[k][4 * j + 1] = make_uint2(a.z, a.w);
                    foot[k][4 * j + 2] = make_uint2(b.x, b.y), foot[k][4 * j + 3] = make_uint2(b.z, b.w);
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const u32x4 t = history.ld4(o + 16u * i, s);
                        foot[k][4 * j + i] = Win{__uint_as_float(t.x), __uint_as_float(t.y), __uint_as_float(t.z)};
                    }
                }
            }
            if (__builtin_amdgcn_ballot_w64(bx != kx) | __builtin_amdgcn_ballot_w64(by != ky) | (uint64_t)(W < 4 || H < 4)) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int i = 0; i < 4; ++i) foot[k][4 * j + i] = tap(kx + i, ky + j);
#pragma unroll
                for (int j = 0; j < 16; ++j) {  // waited for here, not where the paths meet
                    if constexpr (S16) asm volatile("" : "+v"(foot[k][j].x), "+v"(foot[k][j].y));
                    else asm volatile("" : "+v"(foot[k][j].x), "+v"(foot[k][j].y), "+v"(foot[k][j].z));
                }
            }
        }
    } else {
        const int4 wb = wave_min(bases);
        if ((tid & 63) == 0) boxes[tid >> 6] = wb;
#pragma unroll
        for (int k = 0; k < RPT; ++k) q[k].outside = false;
        // positions outside the image: none in a wave whose bases all lie in 0 .. size - 2
        if (!G::PLAIN && (wb.x < 0 || wb.y < 0 || wb.z < 2 - W || wb.w < 2 - H)) {
#pragma unroll
            for (int k = 0; k < RPT; ++k) q[k].outside = q[k].hu < 0.0f || q[k].hv < 0.0f || q[k].hu >= 1.0f || q[k].hv >= 1.0f;
        }
        __syncthreads();
        int4 b = boxes[0];
#pragma unroll
        for (int i = 1; i < G::NT / 64; ++i) {
            const int4 o = boxes[i];
            b = make_int4(min(b.x, o.x), min(b.y, o.y), min(b.z, o.z), min(b.w, o.w));
        }
        // the history window: taps k - 1 .. k + 2 of every footprint, clamped to the edge
        const int wx0 = scalar(b.x) - 1, wy0 = scalar(b.y) - 1;
        const int ww = -scalar(b.z) - scalar(b.x) + 4, wh = -scalar(b.w) - scalar(b.y) + 4;
        fits = ww <= G::WP && wh <= G::WH;
        if (fits) {
            constexpr int L = 16 / G::TB;  // texels a lane
            const int row = tid / G::WL, col = L * (tid - row * G::WL);
            if (wx0 >= 0 && wy0 >= 0 && wx0 + ww + L - 1 <= W && wy0 + wh <= H) {
                const uint32_t o = ((uint32_t)row * pitch + (uint32_t)col) * (uint32_t)G::TB;
                const uint32_t s0 = ((uint32_t)wy0 * pitch + (uint32_t)wx0) * (uint32_t)G::TB;
                const bool take = tid < G::WL * G::WR && col < ww;
                u32x4 v[G::WN];  // (no load in a branch: the others would wait for it. An offset past the image reads nothing)
#pragma unroll
                for (int p = 0; p < G::WN; ++p) {
                    const uint32_t s = p * G::WR < wh ? s0 + (uint32_t)(p * G::WR) * pitch * (uint32_t)G::TB : 0u;  // a row of the image
                    v[p] = history.ld4(take && row + p * G::WR < wh ? o : ~15u, s);
                }
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
    }

    // history filter, rejection, clip and blend
    const uint32_t out_off = ((uint32_t)(y0 + rg) * pitch + (uint32_t)(x0 + rx)) * (uint32_t)G::TB;
    const bool own_col = x0 + rx < fd.x_end && (!G::CAS || (rx >= 1 && rx < 31));
    auto store = [&](void* im, const Tex& t, int k) { gstore<Tex>(im, out_off + (uint32_t)k * pitch * (uint32_t)G::TB, t); };
    Tex res[RPT];
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
        const int y = y0 + rg + k;
        const bool owned = own_col && (k > 0 || !G::CAS || rg > 0) && (k < RPT - 1 || !G::CAS || rg < RH - RPT) && y < H;
        const ProdTexel& p = q[k];
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
        if constexpr (!G::WIN) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const Win e[4] = {foot[k][4 * j], foot[k][4 * j + 1], foot[k][4 * j + 2], foot[k][4 * j + 3]};
                add_row(e, wy.w[j], j == 0);
            }
        } else if (fits) {
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
        bool rejected = p.outside || p.masked;
        if (G::PLAIN) {
        } else if (lin_thr > 0.0f ? linear_depth_reject(p.pd, p.expected, near, far, lin_thr) : fabsf(p.pd - p.expected) > 0.1f * (1.0f - p.pd)) rejected = true;
        // clipAabb (taa.comp:323-345) towards the box's centre c, half size e
        f3 cur;
        bool found;
        {
            f3 c, e;
            box(k, c, e, cur, found);
            const f3 v = hc - c;
            if constexpr (FA) {  // one reciprocal: ma = M / D
                const float exy = e.x * e.y, D = exy * e.z;
                const float M = fmaxf(fabsf(v.x) * (e.y * e.z), fmaxf(fabsf(v.y) * (e.x * e.z), fabsf(v.z) * exy));
                if (M > D) {
                    const float s = D * rcp_fast(M);
                    hc = {__builtin_fmaf(v.x, s, c.x), __builtin_fmaf(v.y, s, c.y), __builtin_fmaf(v.z, s, c.z)};
                }
            } else {
                // no quotient exceeds 1 where |v| <= e (which only e >= 0 does): the divisions are for the other texels
                if (!(fabsf(v.x) <= e.x && fabsf(v.y) <= e.y && fabsf(v.z) <= e.z)) {
                    const f3 u = v / e;
                    const float ma = fmaxf(fabsf(u.x), fmaxf(fabsf(u.y), fabsf(u.z)));
                    if (ma > 1.0f) hc = c + v / ma;
                }
            }
        }
        // blend (taa.comp:850-900)
        const float lc = cur.x, lh = hc.x;
        const float ld = fmaxf(fmaxf(lc, lh), 0.2f);
        const float diff = FA ? fabsf(lc - lh) * rcp_fast(ld) : fabsf(lc - lh) / ld;
        const float wl = 1.0f - diff;
        float ab = G::PLAIN ? P.mAlpha : gmix(a_max, a_min, wl * wl);
        if (!found) ab = ab * 0.0f;  // alpha * beta: beta is 0 where no sample was found, unless rejected or reset
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

    // fused CAS: left and right neighbours from LDS, upper and lower ones of the thread's own column where it
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

}  // namespace
}  // namespace taastar
