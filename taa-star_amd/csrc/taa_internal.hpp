// Internal types shared by the gfx950 kernels (taa_kernels.hip) and the host runtime
// (taa_api.cpp). Not part of the C ABI.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include "taastar/taa_abi.h"
#include "taastar/taa_velocity.h"

namespace taastar {

// One frame as the kernels see it. Mirrors the descriptor set of taa.comp
// (shaders/taa.comp:24-38) plus the tiling of this launch.
struct FrameDesc {
    const void* color;        // uCurrentFrame
    const float* depth;       // uCurrentDepth
    const void* history;      // uHistoryFrame
    const float* hdepth;      // uHistoryDepth
    void* screen;             // uResultScreen (sharpened when cas_on)
    void* debug;              // uDebug (RGBA16F) or null
    const void* velocity;     // uCurrentVelocity
    void* history_out;        // uResultHistory
    void* inspect;            // parity-test intermediates or null
    int32_t W, H, pitch;
    int32_t color_fmt, vel_fmt;
    int32_t x_begin, x_end;   // columns owned by this launch (split screen), [x_begin, x_end)
    int32_t tiles_x, tiles_y; // output tiles covering [x_begin, x_end) x [0, H)
    int32_t param_idx;        // which Parameters block of the uniforms applies
    int32_t cas_on;
    uint32_t cas_peak_bits;   // const1[0] of CasSetup
    int32_t Wl, Hl, pitch_l;  // input (render) size of colour, depth, velocity, previous depth
    int32_t up;               // upsampling path: input size != output size, or mUpsampling
    int32_t rows;             // window and upscale kernels: rows of a column a thread resolves
    float to_u[2], up_scale[2];  // upscale kernel: 1 / input size, output size / input size (x, y)
};

// The segmentation mask's extra images (taa_segmentation_images_t), pitch resolved.
struct SegDesc {
    const uint32_t* material;
    const uint32_t* prev_material;
    const float* uv_normal;
    const uint32_t* prev_segmask;
    uint32_t* segmask;
    int32_t pitch;    // the masks' row pitch (output size)
    int32_t pitch_l;  // the renderer's images' row pitch (input size)
};

// One frame of a batched launch: frame + device copy of its uniforms + first flattened tile.
struct BatchEntry {
    FrameDesc fd;
    taa_uniforms_t U;         // the frame's uniforms, inline so the kernel reads them with scalar loads
    int32_t tile_begin;       // prefix sum of tiles of the entries before this one
    int32_t pad;
    uint64_t pad2;            // entries are whole 16-byte words
};

// Tile shapes the kernels are instantiated for (output tile, 256 threads per workgroup).
struct TileShapeDef {
    int tw, th, pad;
};
constexpr int kNumShapes = 4;
// Shapes used without fused CAS (resolve region == output tile)
constexpr TileShapeDef kShapesPlain[kNumShapes] = {{16, 16, 1}, {32, 8, 1}, {64, 4, 1}, {32, 16, 1}};
// Shapes used with fused CAS (resolve region == output tile + 1-px apron)
constexpr TileShapeDef kShapesCas[kNumShapes] = {{14, 14, 1}, {30, 14, 1}, {30, 30, 1}, {62, 14, 1}};
constexpr int kDefaultShapePlain = 0;
constexpr int kDefaultShapeCas = 2;
// tile shapes of the resolve with the segmentation mask: its LDS also holds the mask's inputs,
// so the small 14x14 CAS tile keeps more workgroups resident (1080p FP32 with the reference's
// default flags: 102 us against 105 us for 30x14 and 151 us for 30x30)
constexpr int kSegShapeCas = 0;
constexpr int kSegShapePlain = kDefaultShapePlain;
// tile shapes of the upsampling resolve (its LDS holds the staged input rectangle); its production
// form (fewer registers) takes 30x14 CAS tiles: 1080p -> 4K in the FP16 arithmetic 0.205 ms against
// 0.232 ms with 14x14 (30x30 and 62x14: 0.261 and 0.267 ms); the general form stays at 14x14. The production
// form is left the sizes that upscale_form() refuses
constexpr int kUpShapeCas = 0;
constexpr int kUpShapeCasProd = 1;
constexpr int kUpShapePlain = kDefaultShapePlain;

inline int tiles_for(int extent, int t) { return (extent + t - 1) / t; }

// Launchers (taa_kernels.hip). All return hipError_t as int.
int launch_resolve(const FrameDesc& fd, const taa_uniforms_t& U, int shape, int arith, void* stream);
// whether launch_resolve runs the exact kernel's production form for this frame (variance clip box,
// clip, YCoCg, Catmull-Rom history, closest-depth RG velocity of the colour's precision, depth
// culling, Lottes, outside rejection; no debug or inspect image): the general kernel's arithmetic
// with the other branches compiled out
bool exact_prod_form(const FrameDesc& fd, const taa_uniforms_t& U);
// the same for its plain form: the production set without closest-depth velocity, depth culling, Lottes weighting and
// outside rejection (each texel's own velocity, mAlpha)
bool exact_plain_form(const FrameDesc& fd, const taa_uniforms_t& U);
// the same switches, whatever the sizes: launch_upscale (or, for the sizes it does not take, launch_resolve_up's
// production form) runs when they hold; with seg, the same with mRayTraceAugment set (the masked resolve's
// production form, whose mask keeps its own parameters)
bool prod_params(const FrameDesc& fd, const taa_uniforms_t& U, bool seg = false);
// the upsampling (TAAU) path: exact FP32 arithmetic, or with TAA_ARITH_FP16 the FP16 path's where no
// selection depends on it; tiled by its form's shape (kUpShapeCas / kUpShapeCasProd / kUpShapePlain),
// whatever fd.tiles_x / tiles_y say
int launch_resolve_up(const FrameDesc& fd, const taa_uniforms_t& U, int arith, void* stream);
// the resolve with the segmentation mask (exact FP32 arithmetic, or with TAA_ARITH_FP16 the FP16 path's
// where no selection depends on it); fd.up: the upsampling path's kernel, which reads the mask's
// inputs from global memory. Tiled by its own shape, whatever fd.tiles_x / tiles_y say
int launch_resolve_seg(const FrameDesc& fd, const taa_uniforms_t& U, const SegDesc& sg, int arith, void* stream);
// Workgroups of a batched launch: one per tile, rounded to whole XCD slots; the batch kernels take
// exactly this grid and resolve one tile per workgroup (batch_tile). Measured on the 64-session
// mix, one workgroup per tile with the hardware dispatcher balancing the XCDs is faster (55.7 vs
// 48.1 Gpix/s) than an occupancy-sized persistent grid with static strides; and a kernel body
// without a loop over tiles keeps the single-frame kernel's register budget (the loop cost the
// FP16 batch kernel 12 VGPRs and a wave per SIMD: 62.6 against 70.9 Gpix/s on the 48-stream mix).
inline int batch_grid(int total_tiles) { return (total_tiles + 7) & ~7; }

// prod: every frame has the production feature set (exact_prod_form): the production form
int launch_batch(const BatchEntry* d_entries, int n_entries, int total_tiles, int shape, bool cas,
                 bool s16, int arith, bool prod, void* stream);
// the upsampling frames of a batch (the upsampling resolve in the batch's arithmetic, kUpShapeCas /
// kUpShapePlain tiles, kUpShapeCasProd with prod: every frame has the production feature set,
// prod_params)
int launch_batch_up(const BatchEntry* d_entries, int n_entries, int total_tiles, bool cas, bool s16, int arith, bool prod,
                    void* stream);

// Throughput kernel (taa_fast.hip): variance clip + Catmull-Rom + simple/closest-depth velocity
// with RG velocity, fp16-fed mixed arithmetic. fast_path_supported() says whether a parameter
// block is one it implements (else *why, when given, names the first reason it is not);
// everything else runs the FP32 kernel.
bool fast_path_supported(const FrameDesc& fd, const taa_uniforms_t& U, int param_idx, const char** why = nullptr);
// the form of the FP16 kernel a supported block runs: 0 the production form (variance box,
// Catmull-Rom history, RG velocity), 1 the general form (min/max box or bilinear history), 2 the
// extended form (matrix reprojection, 3x3-longest velocity, anti-ghosting, velocity-based alpha,
// near-clamp, debug image) with RG velocity, 3 the extended form with RGBA velocity (a batched
// launch's frames must all have RGBA velocity or none)
int fast_path_form(const FrameDesc& fd, const taa_uniforms_t& U, int param_idx);
int launch_resolve_fast(const FrameDesc& fd, const taa_uniforms_t& U, int shape, void* stream);
int launch_batch_fast(const BatchEntry* d_entries, int n_entries, int total_tiles, int shape, bool cas, int form, void* stream);

// The FP16-storage form of that kernel (taa_window.hip): a workgroup resolves a region of 32 columns x
// 32 rows (fd.rows 4: 256 threads, four rows of a column each) or 16 rows (2: 256 threads, two rows
// each; 1: 512 threads, one row each, and without CAS, where there is no ring, 256 threads and 8 rows, whose smaller
// workgroups spread evenly: 720x405 6.5 us against 9.0), of which fused CAS keeps the inner part.
inline void tile_window(FrameDesc& fd, int rows) {
    const int ring = fd.cas_on ? 2 : 0;
    fd.rows = rows;
    fd.tiles_x = tiles_for(fd.x_end - fd.x_begin, 32 - ring);
    fd.tiles_y = tiles_for(fd.H, (rows == 4 ? 32 : rows == 1 && !ring ? 8 : 16) - ring);
}
// rows a thread of a class whose tile shape was tuned or selected (kShapesCas / kShapesPlain index)
constexpr int kWindowRows[kNumShapes] = {1, 2, 4, 2};
// Rows a thread for a launch of n16 workgroups on 16-row regions, n32 on 32-row ones (us a frame, FP16 storage
// and arithmetic, three states in turn, rows 1 / 2 / 4). A launch that leaves the device part empty takes the most
// threads: CAS 640x360 7.7 / 7.9 / 9.8, without CAS 800x450 7.3 / 8.0 / 10.2; in the range 480x270 to 720x405 with CAS
// the tile kernel before this one took 0.3 to 0.7 less, but CAS 800x450 (891 workgroups)
// 9.9 / 9.6 / 11.1. With CAS the 32-row region resolves 14% ring texels instead of 22% and wins once its workgroups
// fill the device (five on each of 256 CUs): 1280x720 16.9 / 16.7 / 19.6, 1600x900 23.9 / 23.0 / 22.8, 3840x2160
// 119 / 115 / 106. Without CAS there is no ring (2560x1440 55.1 / 45.6 / 47.8), and the reference's default block
// (bilinear history, no window) is lighter in registers (2560x1440 45.4 / 43.3 / 45.9): both stay at two rows.
int window_rows(long long n16, long long n32, bool cas, int form);
// its forms: kProd and kDefault fix every option (the production feature set; the reference's default
// block with RGBA velocity), the others read theirs per launch
enum WindowForm { kProd = 0, kVar = 1, kGeneral = 2, kExt = 3, kExtRgba = 4, kDefault = 5, kDefaultExact = 6 };
int window_form(const FrameDesc& fd, const taa_uniforms_t& U, int param_idx);
// whether kDefaultExact takes a frame of the exact arithmetic: the reference's default block on RGBA16F storage with RGBA16F
// velocity, no debug or inspect image. The general kernel read its switches per launch (118 VGPRs) and resolved a row of
// its tile at a time; 1920x1080 with CAS takes 25.3 us now against 55.3, 640x360 6.6 against 7.9 (the cost of a launch),
// 3840x2160 92 against 194
bool default_exact_form(const FrameDesc& fd, const taa_uniforms_t& U, int param_idx);
int launch_window(const FrameDesc& fd, const taa_uniforms_t& U, int form, void* stream);
int launch_window_batch(const BatchEntry* d_entries, int n_entries, int total, int rows, bool cas, int form, void* stream);

// The kernels with the production feature set (taa_exact.hip, taa_upscale.hip): a workgroup resolves a region of 32
// columns x 16 rows (512 threads of one row of a column, or 256 of two) or 32 rows (512 of two, 256 of four), of which
// fused CAS keeps the inner part. fd.rows holds the variant.
enum ProdVariant { kProd512x1 = 1, kProd256x2 = 2, kProd512x2 = 3, kProd256x4 = 4 };
inline int production_rows(int variant) { return variant >= kProd512x2 ? 32 : 16; }
inline void tile_production(FrameDesc& fd, int variant) {
    const int ring = fd.cas_on ? 2 : 0;
    fd.rows = variant;
    fd.to_u[0] = 1.0f / (float)fd.Wl, fd.to_u[1] = 1.0f / (float)fd.Hl;
    fd.up_scale[0] = (float)fd.W / (float)fd.Wl, fd.up_scale[1] = (float)fd.H / (float)fd.Hl;
    fd.tiles_x = tiles_for(fd.x_end - fd.x_begin, 32 - ring);
    fd.tiles_y = tiles_for(fd.H, production_rows(variant) - ring);
}
constexpr int kProdWindowCols = 48, kProdWindowRows = 12;  // the history window: columns, rows beyond the region's
// The exact kernel at one size (kProd256x2 regions), for launches of at least exact_workgroups() of them (us, general kernel's
// production form and this one: with CAS 640x360 (572) FP32 storage 8.9 and 10.8, FP16 9.2 and 10.1, 960x540 (1248) 17.9 and
// 15.6, 18.9 and 15.1; without CAS FP32 960x540 (1020) 12.7 and 13.8, 1280x720 (1800) 19.6 and 19.6, FP16 640x360 (460) 7.8
// and 8.1, 960x540 13.2 and 12.2): below, most of a workgroup's time is the chain of its loads and barriers, which the
// general kernel's small tiles keep shorter.
int launch_exact(const FrameDesc& fd, const taa_uniforms_t& U, bool plain, void* stream);
int launch_exact_batch(const BatchEntry* d_entries, int n_entries, int total, bool plain, bool cas, bool s16, void* stream);
// The masked resolve with the production feature set at one size, exact or FP16 arithmetic, and whether it takes a frame: from 700
// workgroups (us, k_resolve_seg and this one, with CAS: FP32 storage 640x360 (572) 16.4 and 15.7, 320x180 7.9 and 11.2, FP16
// storage and arithmetic 640x360 11.3 and 13.0, 1280x720 33 and 25; without CAS FP32 640x360 (460) 13.6 and 14.5, 1280x720 44 and 34).
bool mask_form(const FrameDesc& fd, const taa_uniforms_t& U);
int launch_mask(const FrameDesc& fd, const taa_uniforms_t& U, const SegDesc& sg, int arith, void* stream);
// The plain form is taken at every size (general kernel and this one, FP32 storage: 320x180 with CAS 7.8 and 7.0), without CAS on
// kProd512x1 regions below 800 workgroups (640x360 7.8, two rows a thread 8.3; 960x540 (1020) 13.1 and 11.9).
inline int plain_variant(long long n16, bool cas) { return !cas && n16 < 800 ? kProd512x1 : kProd256x2; }
inline long long exact_workgroups(bool cas, bool s16) { return cas || s16 ? 900 : 1500; }
// The upsampling resolve, inputs no larger than the output.
// LDS of a tile over a w x h rectangle of input texels, in front of the rectangle's boxes (24 bytes each): the staged
// rectangle and its horizontal depth samples, then in the same place the history window and the resolved texels
#if defined(__HIPCC__)
__host__ __device__
#endif
inline int up_box_offset(int w, int h, int rows, bool s16) {
    const int tex = s16 ? 8 : 12, staged = 384 * h + (s16 ? 20 : 24) * w * h, window = kProdWindowCols * (rows + kProdWindowRows) * tex;
    const int resolved = 32 * rows * (s16 ? 8 : 16);
    const int most = staged > window ? staged : window;
    return ((most > resolved ? most : resolved) + 15) & ~15;
}
// Whether it takes this frame: with 1.4 (FP16 storage) or 1.6 (FP32 storage; 1.8 below 2500 workgroups, and without CAS
// from 600 on: 480x270 at 1.5 times the input 7.0 and 7.9 us) output texels an input texel, where sharing
// an input texel's box among them pays for the larger LDS (us, the general kernel's production form and this one: FP16
// 3840x2160 at 1.15 times the input's size 197 and 210, at 1.2 196 and 182; FP32 1920x1080 at 1.25 68 and 66, at 1.3 68 and
// 60, 3840x2160 at 1.25 256 and 263).
bool upscale_form(const FrameDesc& fd, const taa_uniforms_t& U);
// LDS bytes of any tile of the frame (without the tables)
int upscale_lds(const FrameDesc& fd, int variant);
// The variant of a launch of n16 and n32 workgroups on 16- and 32-row regions, the latter's tiles of lds bytes of LDS
// (us, FP16 storage and arithmetic unless said otherwise): small launches take the most threads (640x360 from 320x180 9.0,
// 256 threads of two rows 9.5). 32 rows have 14% ring texels instead of 22%, once they fill the device: 512 threads of two rows where three
// workgroups' LDS fits a CU (1280x720 to 1920x1080 33.4, 16 rows 37.0; exact on FP32 storage 51.7 and 54.5; at a scale of
// 1.2, where it does not, 45.6 and 43.0), 256 of four where five do, which is at scales of about 2 and more (640x360 to
// 1920x1080 29.8, 512 threads 31.2; 1280x720 to 3840x2160 110 and 122).
int upscale_variant(long long n16, long long n32, int lds);
int launch_upscale(const FrameDesc& fd, const taa_uniforms_t& U, int arith, void* stream);
int launch_upscale_batch(const BatchEntry* d_entries, int n_entries, int total, int variant, int lds, bool cas, bool s16, int arith, void* stream);

// Edge-AA fallback on category-1 texels of a segmentation mask (taa_post.hip).
int launch_edge_aa(const void* src, const uint32_t* mask, void* dst, int W, int H, int pitch, int seg_pitch, int fmt,
                   float subpix, float thr, float thr_min, void* stream);
// sharpen_cas.comp on its own (taa_post.hip).
int launch_cas(const void* src, void* dst, int W, int H, int pitch, int fmt, uint32_t peak_bits, void* stream);

// TAA_OK, or the status taa_batch_submit returns for a frame with these uniforms (taa_api.cpp).
int check_batch_uniforms(const taa_uniforms_t* u);

// Record `msg` as the calling thread's taa_last_error() and return `code` (taa_api.cpp).
int set_last_error(int code, const char* msg);

// taa_resolve_frame with the intermediate screen of split screen with CAS in `scratch` (a device
// buffer of scratch_bytes; TAA_ERR_CAPACITY when the frame needs more) instead of the library's
// per-device buffer; every other case is taa_resolve_frame itself (taa_api.cpp).
int resolve_frame_with_scratch(const taa_uniforms_t* uniforms, const taa_frame_images_t* images, const taa_cas_consts_t* cas,
                               int arith, void* stream, void* scratch, size_t scratch_bytes);
// Bytes that intermediate screen takes for these images (pitch x height texels of the colour format).
size_t split_cas_scratch_bytes(const taa_frame_images_t* images);

// Velocity producer (taa_velocity.hip): one launch over width x height; ids may be NULL.
int launch_velocity(const taa_reproject_t& r, const float* depth, const uint32_t* ids, void* velocity, int fmt, int W,
                    int H, int pitch, void* stream);

}  // namespace taastar
