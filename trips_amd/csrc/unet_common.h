// Pieces shared by the forward and backward kernels of the reconstruction net (gfx950).
#pragma once
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <algorithm>

#include "../../include/trips_unet.h"
#include "splat_internal.h"

namespace trips
{
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kConvTileH   = 8;
constexpr int kConvTileW   = 32;
constexpr int kConvPatchH  = kConvTileH + 2;
constexpr int kConvPatchW  = kConvTileW + 2;
constexpr int kBelowH      = kConvTileH / 2 + 2;  // rows / columns of the level below that an upsampled patch touches
constexpr int kBelowW      = kConvTileW / 2 + 2;
constexpr int kFinalPixelsPerBlock = 256;   // pixels a workgroup of the 1x1 convolution's backward takes at a time
constexpr int kUnetMaxImageChannels = 16;  // channels of the splat images (the descriptor widths of the splat: 3, 4, 6, 8, 16)
constexpr int kFinalPartFloats     = 4 * (kUnetMaxImageChannels + 64) + 4;  // its partial sums: [4 outputs][<= 16 image + <= 64 block channels], 4 biases
constexpr int kMaxGridImages = 32768;  // images of a batch that one launch takes (the y and z dimensions of a grid end at 65535)
constexpr int kLdsChanPad  = 8;  // halves added to every LDS row so that 16 lanes reading 16 bytes hit 64 distinct banks

// position n of a pixel's pre-activations (see LevelPlan): its channel, and whether it is the mask's
__host__ __device__ __forceinline__ int preact_channel(int n) { return (n >> 3) * 4 + (n & 3); }
__host__ __device__ __forceinline__ bool preact_is_mask(int n) { return (n & 4) != 0; }

// source row / column and weight of torch's bilinear upsampling with scale_factor 2, align_corners = false
// (area_pixel_compute_source_index: src = max(0, (dst + 0.5) * 0.5 - 0.5))
__device__ __forceinline__ void up2_source(int dst, int in_size, int& i0, int& i1, float& lambda)
{
    float src = (float(dst) + 0.5f) * 0.5f - 0.5f;
    src       = src < 0.f ? 0.f : src;
    i0        = (int)src;
    i0        = i0 < in_size - 1 ? i0 : in_size - 1;
    i1        = i0 + 1 < in_size ? i0 + 1 : in_size - 1;
    lambda    = src - float(i0);
}

// The 2 x 2 pixels that bilinear 2x upsampling (align_corners = false) makes between four neighbouring pixels of the
// coarser level, v[0..3] = (upper left, upper right, lower left, lower right), eight channels in packed fp16. The
// weights (products of 1/4 and 3/4) are exact, and a sum of products stays in fp16's range wherever its result does;
// the separable form, along x, then along y, needs differences of neighbours, which need not (its 12 packed operations
// instead of 16 made no difference in time).
// `top` / `left`: the lower / right pixels are the image's first row / column, whose source is that of the coarser level
// alone.
__device__ __forceinline__ void upsample_quad(half8 a, half8 b, half8 c, half8 d, bool top, bool left, half8 (&v)[4])
{
    const _Float16 w1 = _Float16(0.0625f), w3 = _Float16(0.1875f), w9 = _Float16(0.5625f);
    const half8 W1 = {w1, w1, w1, w1, w1, w1, w1, w1}, W3 = {w3, w3, w3, w3, w3, w3, w3, w3}, W9 = {w9, w9, w9, w9, w9, w9, w9, w9};
    auto mix = [](half8 a, half8 wa, half8 b, half8 wb, half8 c, half8 wc, half8 d, half8 wd)
    { return __builtin_elementwise_fma(d, wd, __builtin_elementwise_fma(c, wc, __builtin_elementwise_fma(b, wb, a * wa))); };
    v[0] = mix(a, W9, b, W3, c, W3, d, W1);
    v[1] = mix(a, W3, b, W9, c, W1, d, W3);
    v[2] = mix(a, W3, b, W1, c, W9, d, W3);
    v[3] = mix(a, W1, b, W3, c, W3, d, W9);
    if (top || left)
    {
        const _Float16 q1 = _Float16(0.25f), q3 = _Float16(0.75f);
        const half8 Q1 = {q1, q1, q1, q1, q1, q1, q1, q1}, Q3 = {q3, q3, q3, q3, q3, q3, q3, q3};
        if (top)
        {
            v[2] = __builtin_elementwise_fma(b, Q1, a * Q3);
            v[3] = __builtin_elementwise_fma(b, Q3, a * Q1);
        }
        if (left)
        {
            v[1] = __builtin_elementwise_fma(c, Q1, a * Q3);
            v[3] = top ? a : __builtin_elementwise_fma(c, Q3, a * Q1);
        }
    }
}

// Work split of the weight-gradient kernel for a (padded input channels, padded pre-activations) shape: how many ways the
// wavefronts split the 16-channel input blocks, the 16-channel pre-activation blocks and, where there are more wavefronts
// than blocks, the rows of a tile.
constexpr int kWgradThreads = 512;
// Pre-activations of a workgroup: 64 at most, so that a tile in flight has registers beside the sums (64 inputs x 128 in one
// workgroup spilled and took four times as long per tile as 64 x 64). 32 x 128 fits, and where every workgroup has tiles to
// walk it saves assembling the patch twice: 1920 x 1080, 272 -> 206 us; with 300 tiles 21 -> 23, with 30 9 -> 13.
constexpr int wgrad_tile(int cin, int npad, long long tiles) { return npad == 128 && cin == 32 && tiles >= 512 ? 128 : npad % 64 == 0 ? 64 : 32; }
constexpr int wgrad_cbw(int cin) { return cin / 16 < 4 ? cin / 16 : 4; }
constexpr int wgrad_nbw(int cin, int npad)
{
    return (kWgradThreads / 64) / wgrad_cbw(cin) < npad / 16 ? (kWgradThreads / 64) / wgrad_cbw(cin) : npad / 16;
}
constexpr int wgrad_row_split(int cin, int npad) { return (kWgradThreads / 64) / (wgrad_cbw(cin) * wgrad_nbw(cin, npad)); }

// ---- host-side plan of a network: per level the padded GEMM sizes and where its buffers live ----
inline int round_up(int v, int m) { return (v + m - 1) / m * m; }

// Rows of a level: [B][H][W][row_stride] fp16, what the next finer block reads of this one. Positions [0, C) are zero,
// [C, 2C) the level's image, [2C, 2C + cout) the block's outputs: the positions that these channels have in the finer
// block's input, whose first C are its own image. row_stride = 2C + cout rounded up to 8, the rest zero.
// Pre-activations and their gradients: [B][H][W][npad] fp16, the features and the masks of four channels side by side:
// position 8 (ch / 4) + 4 (mask) + ch % 4, so that one 16-byte access serves the gate of four channels.
struct LevelPlan
{
    int H, W, cin_real, cin_pad, cout, npad, row_stride;
    size_t wpack_off, bias_off, rows_off;  // bytes into the forward workspace
    size_t saved_rows_off, saved_pre_off;  // bytes into the saved state (training)
    // bytes into the backward workspace
    size_t wt_off;      // packed transposed weights [9][cin_pad][npad] fp16
    size_t dpre_off;    // gradient of the pre-activations [B][H][W][npad] fp16
    size_t din_off;     // gradient of the block input [B][H][W][cin_pad] fp16, where it leaves its kernel
    size_t part_off;    // partial weight gradients [groups][9][npad][cin_pad] fp32
    size_t sliced_off;  // partial sums of the partials [16][9][npad][cin_pad] fp32
    size_t bias_part_off;  // per-workgroup sums of the pre-activation gradients [groups][npad] fp32
    int wgrad_tile;     // pre-activations of a workgroup of the weight-gradient kernel
    long long tiles;    // 8 x 32 tiles of all images of the batch
    int groups;         // persistent workgroups of the weight-gradient kernel for each of its npad / wgrad_tile shares
    int wgrad_resident; // ... and how many of them share a CU
};

// Whether the data gradient of a block and the adjoint of the upsampling below it run as one kernel
// (conv_bwd_data_up_kernel): where there is a level below and the weights of a wavefront's outputs fit its registers
// (64 x 64 takes 144 of a lane's 256; 96 would take 216).
inline bool bwd_data_up_fits(int npad, int cin_pad, bool below) { return below && npad <= 64 && cin_pad <= 64; }

struct NetPlan
{
    LevelPlan lv[TRIPS_UNET_MAX_LEVELS];
    size_t bytes;           // forward workspace
    size_t fin_off;         // forward workspace: packed weights of the 1x1 output convolution
    size_t saved_bytes;     // saved state
    size_t backward_bytes;  // backward workspace
    size_t wgrad_off;       // backward workspace: the levels' partial weight and bias gradients (plan_wgrad)
    size_t final_part_off;  // backward workspace: per-workgroup sums of the 1x1 convolution's weight and bias gradients
    int final_groups;       // persistent workgroups of the finest level's first backward kernel, for all images of the batch
};

inline int check_unet_desc(const TripsUnetDesc* d)
{
    if (!d) return set_error(TRIPS_ERR_INVALID_ARG, "desc is NULL");
    if (d->abi_version != TRIPS_ABI_VERSION)
        return set_error(TRIPS_ERR_INVALID_ARG, "abi_version %d, library has %d", d->abi_version, TRIPS_ABI_VERSION);
    if (d->num_levels < 1 || d->num_levels > TRIPS_UNET_MAX_LEVELS)
        return set_error(TRIPS_ERR_INVALID_ARG, "num_levels %d not in 1..%d", d->num_levels, TRIPS_UNET_MAX_LEVELS);
    if (d->num_input_channels < 1 || d->num_input_channels > kUnetMaxImageChannels)
        return set_error(TRIPS_ERR_UNSUPPORTED, "num_input_channels %d not in 1..%d", d->num_input_channels, kUnetMaxImageChannels);
    if (d->num_output_channels < 1 || d->num_output_channels > 4)
        return set_error(TRIPS_ERR_UNSUPPORTED, "num_output_channels %d not in 1..4", d->num_output_channels);
    if (d->batch < 1) return set_error(TRIPS_ERR_INVALID_ARG, "batch < 1");
    const int C = d->num_input_channels, L = d->num_levels;
    for (int i = 0; i < L; ++i)
    {
        if (d->level_w[i] < 1 || d->level_h[i] < 1 || d->level_w[i] > 32768 || d->level_h[i] > 32768)
            return set_error(TRIPS_ERR_INVALID_ARG, "level %d size %dx%d", i, d->level_w[i], d->level_h[i]);
        if (i > 0)
        {
            const int w = d->level_w[i - 1], h = d->level_h[i - 1];
            const bool okw = d->level_w[i] == w / 2 || d->level_w[i] == (w + 1) / 2;
            const bool okh = d->level_h[i] == h / 2 || d->level_h[i] == (h + 1) / 2;
            if (!okw || !okh || 2 * d->level_w[i] < w || 2 * d->level_h[i] < h)
                return set_error(TRIPS_ERR_UNSUPPORTED, "level %d (%dx%d) must be half of level %d (%dx%d), rounded up", i,
                                 d->level_w[i], d->level_h[i], i - 1, w, h);
        }
        const int cout = d->filters[i] - ((i == 0 && L > 1) ? C : 2 * C);
        if (cout < 1 || cout > 64)
            return set_error(TRIPS_ERR_UNSUPPORTED, "filters[%d] = %d gives %d convolution outputs (1..64 supported)", i,
                             d->filters[i], cout);
        if (i + 1 < L && d->filters[i + 1] > 64)
            return set_error(TRIPS_ERR_UNSUPPORTED, "filters[%d] = %d input channels (at most 64 supported)", i + 1,
                             d->filters[i + 1]);
    }
    return TRIPS_OK;
}

// Workgroups of the weight gradient on a CU (`tiles`: of all its levels; `channels`: of the image). Two for 32 inputs x 32
// pre-activations. Two for 32 x 64 too (LDS 75 KB, 128 registers of a lane, for which the kernel spills 3 to 7 of the 134 to 139 that
// it takes with the bias gradients, 16 to 22 without) where one's loads and barriers then pass while the other multiplies: up to
// eight channels, from three tiles for each of the 512 on. us, one of its own registers and two, kernel + sums of the partials:
// levels of 1245 x 825, three channels 99.9 + 6.2 and 86.5 + 8.4, four 97 + 6.4 and 85 + 8.5, six 93 + 4.9 and 88 + 8.0, eight 75 + 8.8 and
// 71 + 11; four crops of 512 x 512 94 + 6.3 and 83 + 8.5. The sixteen channels of a pixel's image leave the registers less room (17
// to 38 spilled): ten channels 84 + 8.7 and 100 + 10.7, at 960 x 560 52 + 7.2 and 62 + 9.6. Around three tiles: four channels, 1500
// tiles, 32.2 + 5.2 and 30.0 + 7.6, 1800 38.2 + 5.0 and 31.6 + 7.5; eight, 1200 tiles, 31.2 + 6.6 and 31.7 + 8.5, 1610 38.4 + 7.3 and 36.1 + 9.4.
// (One on a CU, but held to 128 registers all the same: 1500 tiles of four channels 32.2 -> 33.6, 1200 of eight 31.2 -> 34.0, 650 of ten
// 22.9 -> 29.5.)
inline int wgrad_resident(int cin_pad, int npad, int channels, long long tiles)
{
    return cin_pad == 32 && (npad == 32 || (npad == 64 && channels <= 8 && tiles >= 3 * 512)) ? 2 : 1;
}

// Levels whose weight gradients are the same instance of the kernel run in one launch, whose workgroups are as many as are
// resident at once (every further one would only add a set of partial sums to write and reduce) and are dealt to the levels by their tiles. With a launch per level the coarser ones were a handful of
// tiles each, begun and ended 256 workgroups at a time: all weight gradients and the sums of their partials, default net
// of five levels at 1245 x 825 155 -> 110 us, at 105 x 74 (32/64/64/64/64) 85 -> 46, 16/32/64/64 at 1920 x 1080 217 -> 205.
// `wanted` holds a bit per level whose weight gradients are asked for: the workgroups are dealt to those alone. (Dealt as if
// all were asked for, a level on its own got a fifth of the GPU. Whole backward of the default net at 1245 x 825 with the weight
// gradients of all levels but the finest 307 -> 256 us, of the second level alone 303 -> 250, of the finest alone 310 -> 291;
// the finest without its bias gradients, then a launch of its own, 387 -> 316.)
// The partial sums lie from `at` on; returns where they end, which does not depend on `wanted`: an instance has at most
// `resident` workgroups, and at most one for each tile and share of its levels, and a workgroup writes one set of sums.
inline bool same_wgrad_kernel(const LevelPlan& a, const LevelPlan& b) { return a.cin_pad == b.cin_pad && a.wgrad_tile == b.wgrad_tile; }
inline size_t plan_wgrad(NetPlan& np, int levels, int channels, unsigned wanted, size_t at)
{
    for (int i = 0; i < levels; ++i)
    {
        const LevelPlan& lv = np.lv[i];
        bool first          = true;  // of its instance
        for (int k = 0; k < i; ++k) first = first && !same_wgrad_kernel(np.lv[k], lv);
        if (!first) continue;
        long long all = 0, work = 0, shares = 0;
        for (int k = i; k < levels; ++k)
            if (same_wgrad_kernel(np.lv[k], lv))
            {
                const int s = np.lv[k].npad / lv.wgrad_tile;
                all += np.lv[k].tiles * s;
                if (!((wanted >> k) & 1u)) continue;
                work += np.lv[k].tiles * s;
                shares += s;
            }
        const int on_a_cu        = wgrad_resident(lv.cin_pad, lv.wgrad_tile, channels, all);
        const long long resident = 256 * on_a_cu;
        size_t o = at;
        for (int k = i; k < levels; ++k)
        {
            LevelPlan& l = np.lv[k];
            if (!same_wgrad_kernel(l, lv) || !((wanted >> k) & 1u)) continue;
            l.wgrad_resident = on_a_cu;
            // one workgroup for every share, the others by the tiles (rounded down: one that has to wait for another to end
            // would take as long again)
            l.groups   = (int)std::min(1 + (resident - shares) * l.tiles / work, l.tiles);
            l.part_off = o;
            o += (size_t)l.groups * 9 * l.npad * l.cin_pad * sizeof(float);
            l.bias_part_off = o;
            o += (size_t)l.groups * l.npad * sizeof(float);
        }
        at += align256((size_t)std::min(resident, all) * lv.wgrad_tile * (9 * lv.cin_pad + 1) * sizeof(float));
    }
    return at;
}

// Block i convolves cat(in[i], up2(x_{i+1})) (F[i+1] channels; C for the start block) to F[i] - 2C outputs
// (F[0] - C for the last block when it is not also the start block), Networks.h:1034-1037,1104-1118.
inline NetPlan make_plan(const TripsUnetDesc& d)
{
    NetPlan np;
    const int C = d.num_input_channels, L = d.num_levels;
    size_t o = 0;
    for (int i = 0; i < L; ++i)
    {
        LevelPlan& lv = np.lv[i];
        lv.H          = d.level_h[i];
        lv.W          = d.level_w[i];
        lv.cin_real   = (i == L - 1) ? C : d.filters[i + 1];
        lv.cin_pad    = lv.cin_real <= 32 ? 32 : 64;
        lv.cout       = d.filters[i] - ((i == 0 && L > 1) ? C : 2 * C);
        lv.npad       = 2 * round_up(lv.cout, 16);
        lv.row_stride = round_up(2 * C + lv.cout, 8);
        lv.wpack_off  = o;
        o += align256((size_t)9 * lv.npad * lv.cin_pad * sizeof(_Float16));
        lv.bias_off = o;
        o += align256((size_t)lv.npad * sizeof(float));
    }
    np.fin_off = o;
    o += align256((size_t)(np.lv[0].npad / 32 + 1) * 64 * sizeof(_Float16));
    for (int i = 0; i < L; ++i)
    {
        // (the rows of the finest level do not leave their kernel)
        np.lv[i].rows_off = o;
        if (i > 0) o += align256((size_t)d.batch * np.lv[i].H * np.lv[i].W * np.lv[i].row_stride * sizeof(_Float16));
    }
    np.bytes = o;
    size_t sv = 0, bw = 0;
    for (int i = 0; i < L; ++i)
    {
        LevelPlan& lv       = np.lv[i];
        const size_t pixels = (size_t)d.batch * lv.H * lv.W;
        lv.saved_rows_off   = sv;
        if (i > 0) sv += align256(pixels * lv.row_stride * sizeof(_Float16));
        lv.saved_pre_off = sv;
        sv += align256(pixels * lv.npad * sizeof(_Float16));
        lv.wt_off = bw;
        bw += align256((size_t)9 * lv.cin_pad * lv.npad * sizeof(_Float16));
        lv.dpre_off = bw;
        bw += align256(pixels * lv.npad * sizeof(_Float16));
        lv.din_off = bw;
        if (i < L - 1 && !bwd_data_up_fits(lv.npad, lv.cin_pad, true)) bw += align256(pixels * lv.cin_pad * sizeof(_Float16));
        const long long tiles = (long long)d.batch * ((lv.W + kConvTileW - 1) / kConvTileW) * ((lv.H + kConvTileH - 1) / kConvTileH);
        lv.wgrad_tile = wgrad_tile(lv.cin_pad, lv.npad, tiles);
        lv.tiles      = tiles;
    }
    for (int i = 0; i < L; ++i)
    {
        np.lv[i].sliced_off = bw;
        bw += align256((size_t)16 * 9 * np.lv[i].npad * np.lv[i].cin_pad * sizeof(float));
    }
    np.wgrad_off = bw;
    bw           = plan_wgrad(np, L, C, ~0u, bw);
    {
        const size_t chunks = d.batch * (((size_t)np.lv[0].H * np.lv[0].W + kFinalPixelsPerBlock - 1) / kFinalPixelsPerBlock);
        // as many workgroups as are resident at once walk the chunks (four per CU at the 100 to 118 registers of most
        // instances): a second, partly filled round of one-chunk workgroups cost a third of the kernel's time. Three per CU
        // with chunks of 512 pixels 95 us at 1245 x 825, four 90, four with chunks of 256 (less difference between the
        // workgroup with the most and the one with the fewest) 84; five, at 96 registers, no faster.
        np.final_groups     = chunks < 1024 ? (int)chunks : 1024;
        np.final_part_off   = bw;
        bw += align256((size_t)np.final_groups * kFinalPartFloats * sizeof(float));
    }
    np.saved_bytes    = sv;
    np.backward_bytes = bw;
    return np;
}


}  // namespace trips
