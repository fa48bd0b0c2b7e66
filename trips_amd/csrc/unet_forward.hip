// Forward of the decoder-only gated-convolution U-Net on the gfx950 matrix cores.
//
//   gated_conv3x3_kernel <- SmallDecStartBlockImpl::forward / UpsampleDecOnlySmallBlockFixedImpl::forward
//                           src/lib/models/Networks.h:751-787, 999-1098
//                           and, in the finest block's epilogue, the `final` 1x1 Sequential of
//                           MultiScaleUnet2dDecOnlySmallFixedImpl, Networks.h:1129-1131
//
// The reference runs, per level, upsample -> cat -> two 3x3 convolutions -> elu / sigmoid -> multiply -> cat as
// separate libtorch ops on NCHW tensors, materialising every intermediate. Here one kernel per level does all of
// it as an implicit GEMM: M = 256 output pixels of an 8 x 32 patch, N = feature and mask outputs side by side,
// K = 9 taps x input channels. The input patch (with its one-pixel halo) is assembled in LDS, channels innermost:
// channels [0, C) come straight from this level's splat image, the others are the bilinear 2x upsampling of the
// level below (its splat image, then its convolution outputs), computed on the way in, so neither the upsampled
// tensor nor the concatenations ever exist in memory. Activations between levels are fp16, channels innermost, and
// carry the level's image with them (the row format is described at LevelPlan).
// MFMA: v_mfma_f32_16x16x32_f16; lane l holds, of A, row l % 16 and the 8 consecutive K values (l / 16) * 8 ..,
// of B the same for column l % 16, and of the 16 x 16 result rows (l / 16) * 4 .. + 3 of column l % 16.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>

#include "unet_common.h"

namespace trips
{
struct ConvParams
{
    int H, W;            // this level
    int Hb, Wb;          // level below (0 x 0 for the start block)
    int c_feat;          // channels of the splat images (C)
    int cout;            // real outputs of each of the two convolutions
    int npad;            // halves per pixel of `pre`
    int tiles_x, tiles, batch;  // tiles of a row and of one image, images
    const float* feat;   // this level's image: element (pixel, channel) at pixel * feat_ps + channel * feat_cs
    int feat_ps;
    size_t feat_cs;
    const _Float16* below;    // rows of the level below, [Hb][Wb][below_stride], or nullptr
    int below_stride;
    const _Float16* wfrag;    // weights as MFMA fragments: [pair][tap][CIN / 32][feature, mask][lane][8]
    const float* bias;        // [pair][feature, mask][16]
    _Float16* out;            // this level's rows, [H][W][out_stride], or nullptr when only the fused 1x1 reads them
    int out_stride;
    _Float16* pre;            // [H][W][npad] pre-activations for the backward (see LevelPlan), or nullptr
    // the net's 1x1 output convolution on x_0 = cat(image, block output), fused into the finest block, or nullptr
    const _Float16* fin_frag;  // [pair, then the image][lane % 4 = output][lane / 16][4]: see pack_conv_weights_kernel
    const float* final_b;      // [final_cout]
    float* final_out;          // [final_cout][H][W]
    int final_cout;
};

// One workgroup walks tiles of 8 x 32 pixels and computes PAIRS pairs of (16 feature, 16 mask) outputs of each. Its
// wavefronts split the pairs and the tile: a wavefront owns one pair for STRIPS strips of 16 pixels x MB rows, so that its A
// operands (LDS) are shared by the three vertical taps and a lane ends up with four features and the masks of the same
// four channels of a pixel: the gate, the stores and the 1x1 of the finest level need no LDS and no further exchange.
// What bounds it: vector instructions (loads, upsampling, the gate's two exponentials), then the latency of the phases
// between two barriers; the matrix cores are busy for a fifth of the time. Hence: what a tile's threads share is worked
// out once per workgroup or on the scalar unit, the loads of the next tile travel during this one's products, and the
// upsampling makes 2 x 2 pixels from one set of four neighbours (385 instead of 710 vector instructions per wavefront
// and 256-pixel tile at the finest level of the 16/32/64/64 net). 1920 x 1080, that net, per level, against one tile
// per workgroup with LDS-staged epilogues: 100 -> 76, 59 -> 60, 36 -> 34, 13 -> 11 us.
// KREG: the pair's weights of so many blocks of 32 inputs (9 taps: 72 registers each) stay in registers for all tiles of
// the workgroup, the others are staged in LDS once. With 32 inputs all are (held in registers they leave room for half the
// wavefronts: 121 us at the finest level, where six wavefronts per SIMD, with 4 registers spilled, take 74 and four 83);
// with 64 none, but for three pairs, where half of them in LDS let twelve wavefronts share the SIMDs evenly: 252 us for
// 64 -> 96 at 1920 x 1080, 364 with six wavefronts and all weights in registers.
// CI: image channels the kernel has room for (4, 8 or 16); FOUR: C is exactly 4, the splat's usual descriptor width
template <int CIN, int PAIRS, int CI, bool FOUR, int THREADS, int KREG, int WAVES_PER_EU>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(WAVES_PER_EU))) void gated_conv3x3_kernel(const ConvParams p)
{
    constexpr int KB      = CIN / 32;
    constexpr int ROW     = CIN + kLdsChanPad;  // halves per patch pixel in LDS
    constexpr int GROUPS  = CIN / 8;
    constexpr int WAVES   = THREADS / 64;
    constexpr int MB      = std::min(16 * PAIRS / WAVES, 4);  // rows of a strip (the 1x1 keeps them in one accumulator)
    constexpr int STRIPS  = 16 * PAIRS / WAVES / MB;          // strips of a wavefront, one after the other
    static_assert(WAVES % PAIRS == 0 && WAVES * MB * STRIPS == 16 * PAIRS, "the strips of a tile");
    static_assert(PAIRS > 2 || STRIPS == 1, "the sums of the 1x1 are handed over once per tile");
    constexpr int kPatch  = kConvPatchH * kConvPatchW;
    constexpr int kQuads  = (kConvPatchH / 2) * (kConvPatchW / 2);
    constexpr int QITEMS  = (kQuads * GROUPS + THREADS - 1) / THREADS;
    // (8 and 16 image channels, and 64 inputs with three and more pairs, leave no registers for the loads of the next tile:
    // 64 -> 96 at 1920 x 1080, 273 us with them and 18 registers spilled, 252 without)
    constexpr bool kPrefetch = (CI == 4 && (CIN == 32 || PAIRS <= 2)) || (CIN == 32 && CI == 8);
    // ... and beside weights in registers none for them over the end of a tile either
    constexpr bool kAhead = kPrefetch || KREG == 0;
    constexpr int FITEMS     = (kPatch + THREADS - 1) / THREADS;
    constexpr int KLDS       = KB - KREG;  // 32-input blocks whose weights sit in LDS
    __shared__ __align__(16) _Float16 s_patch[kPatch * ROW];
    __shared__ __align__(16) _Float16 s_w[KLDS == 0 ? 8 : PAIRS * 9 * KLDS * 2 * 512];
    __shared__ float4 s_fin[PAIRS == 1 ? 1 : (PAIRS == 2 ? 1 : PAIRS) * 4 * 64];

    const int lane = (int)threadIdx.x & 63;
    // (a wavefront's number is the same for its lanes: kept on the scalar unit)
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int lrow = lane & 15, lq = lane >> 4;
    const int C    = FOUR ? 4 : p.c_feat;
    const int pair = PAIRS == 1 ? 0 : PAIRS == 2 ? wave & 1 : wave % PAIRS;
    const int gp   = blockIdx.y * PAIRS + pair;  // this wavefront's pair of the level
    const int first_strip = PAIRS == 1 ? wave : wave / PAIRS;
    const int tiles = p.tiles * p.batch;

    const int below_groups = p.below_stride / 8;
    // ---- this thread's share of the loads of a tile ----
    struct Loads
    {
        float f[FITEMS][CI];   // pixels of the image patch
        uint4 q[QITEMS][4];    // eight channels of 2 x 2 pixels of the level below: they make 2 x 2 pixels of the patch
    };
    struct Tile
    {
        int image, x0, y0;
    };
    auto decode = [&](int t)
    {
        Tile r;
        r.image      = t / p.tiles;
        const int i  = t - r.image * p.tiles;
        const int ty = i / p.tiles_x;
        r.x0         = (i - ty * p.tiles_x) * kConvTileW;
        r.y0         = ty * kConvTileH;
        return r;
    };
    auto issue = [&](const Tile& t, int tid, Loads& r)
    {
        // (addresses: what a tile shares is added up on the scalar unit, a thread's own part fits 32 bits)
        const float* img = p.feat + (size_t)t.image * p.H * p.W * C + ((size_t)t.y0 * p.W + t.x0) * p.feat_ps;
#pragma unroll
        for (int k = 0; k < FITEMS; ++k)
        {
            const int item = min(tid + THREADS * k, kPatch - 1);
            const int y = t.y0 + item / kConvPatchW - 1, x = t.x0 + item % kConvPatchW - 1;
            const int off = ((min(max(y, 0), p.H - 1) - t.y0) * p.W + min(max(x, 0), p.W - 1) - t.x0) * p.feat_ps;
#pragma unroll
            for (int c = 0; c < CI; ++c) r.f[k][c] = (img + (c < C ? c : 0) * p.feat_cs)[off];
        }
        if (below_groups > 0)
        {
            const int y00 = max(t.y0 / 2 - 1, 0);
            const _Float16* src = p.below + ((size_t)t.image * p.Hb + y00) * p.Wb * p.below_stride;
#pragma unroll
            for (int k = 0; k < QITEMS; ++k)
            {
                const int item = tid + THREADS * k;
                const int g = item % GROUPS, quad = min(item / GROUPS, kQuads - 1);
                const int j = quad / (kConvPatchW / 2), i = quad - j * (kConvPatchW / 2);
                const int ya = min(max(t.y0 / 2 - 1 + j, 0), p.Hb - 1) - y00, yb = min(t.y0 / 2 + j, p.Hb - 1) - y00;
                const int xa = min(max(t.x0 / 2 - 1 + i, 0), p.Wb - 1), xb = min(t.x0 / 2 + i, p.Wb - 1);
                const _Float16* s = src + 8 * min(g, below_groups - 1);
                const int ra = ya * p.Wb, rb = yb * p.Wb;
                r.q[k][0] = *reinterpret_cast<const uint4*>(s + (ra + xa) * p.below_stride);
                r.q[k][1] = *reinterpret_cast<const uint4*>(s + (ra + xb) * p.below_stride);
                r.q[k][2] = *reinterpret_cast<const uint4*>(s + (rb + xa) * p.below_stride);
                r.q[k][3] = *reinterpret_cast<const uint4*>(s + (rb + xb) * p.below_stride);
            }
        }
    };
    // Consecutive tiles share their halos: they go to one XCD (workgroups are dealt to the eight of them in turn). The XCDs'
    // shares differ by one tile at most, the first ones' being the larger as are their numbers of workgroups: with as many
    // workgroups as tiles each has one. (With shares rounded up, a workgroup of some XCD took a second tile: 75 tiles of
    // 32 -> 32, 11.0 instead of 8.2 us, of 64 -> 64 at 160 x 120, 19.5 instead of 13.1.)
    const int xcd  = (int)blockIdx.x & 7, in_xcd = ((int)gridDim.x - xcd + 7) >> 3;
    const int last = (xcd + 1) * (tiles >> 3) + min(xcd + 1, tiles & 7);
    int at         = xcd * (tiles >> 3) + min(xcd, tiles & 7) + ((int)blockIdx.x >> 3);

    // The first tile's loads travel while weights are staged and the patch is cleared, and the weights on their way to LDS
    // are all requested together: a level of few tiles lasts as long as this and one tile (finest level of 160 x 120,
    // 32 -> 64: 10.7 -> 9.8 us, start block of eight image channels: 9.5 -> 8.8).
    Loads cur;
    if (kAhead && KREG == 0 && at < last) issue(decode(at), (int)threadIdx.x, cur);

    // ---- what stays for all tiles: weights, biases, the 1x1's weights ----
    const half8* wsrc = reinterpret_cast<const half8*>(p.wfrag) + (size_t)gp * (9 * KB * 2 * 64) + lane;
    half8 w[KREG > 0 ? 9 : 1][KREG > 0 ? KREG : 1][2];
    if (KREG > 0)
    {
#pragma unroll
        for (int t = 0; t < (KREG > 0 ? 9 : 1); ++t)
#pragma unroll
            for (int kb = 0; kb < KREG; ++kb)
#pragma unroll
                for (int h = 0; h < 2; ++h) w[t][kb][h] = wsrc[((t * KB + kb) * 2 + h) * 64];
    }
    constexpr int kRun = KLDS > 0 ? KLDS * 2 * 64 : 1;  // 16-byte words of a tap
    constexpr int kStaged = PAIRS * 9 * KLDS * 2 * 64, WITEMS = (kStaged + THREADS - 1) / THREADS;
    half8 staged[WITEMS > 0 ? WITEMS : 1];
    {
        const half8* src = reinterpret_cast<const half8*>(p.wfrag) + (size_t)blockIdx.y * PAIRS * (9 * KB * 2 * 64);
#pragma unroll
        for (int k = 0; k < WITEMS; ++k)
        {
            const int i = min((int)threadIdx.x + THREADS * k, kStaged - 1);
            staged[k]   = src[KREG == 0 ? i : i / kRun * (KB * 2 * 64) + KREG * 2 * 64 + i % kRun];
        }
    }
    const float4 bias_f = *reinterpret_cast<const float4*>(p.bias + gp * 32 + lq * 4);
    const float4 bias_m = *reinterpret_cast<const float4*>(p.bias + gp * 32 + 16 + lq * 4);
    // A operand of the 1x1: every lane group's rows hold the four outputs, of which group m keeps those of the strip's row m
    // (the same number of selects as zero weights for the other rows, through which an infinite operand of one row would
    // make all of them not a number)
    half4 fw = half4{}, fimg = half4{};
    if (p.final_out)
    {
        fw   = *reinterpret_cast<const half4*>(p.fin_frag + (gp * 16 + (lrow & 3) * 4 + lq) * 4);
        fimg = *reinterpret_cast<const half4*>(p.fin_frag + ((p.npad / 32) * 16 + (lrow & 3) * 4 + lq) * 4);
    }
    if (kAhead && KREG > 0 && at < last) issue(decode(at), (int)threadIdx.x, cur);
    // channels that nothing ever writes: of the start block all but the image's, of the others the groups that the
    // rows of the level below do not have; and the padding of the patch's rows
    for (int i = threadIdx.x; i < kPatch * (GROUPS + 1); i += THREADS)
        if (i % (GROUPS + 1) >= below_groups) *reinterpret_cast<half8*>(s_patch + (i / (GROUPS + 1)) * ROW + 8 * (i % (GROUPS + 1))) = half8{};

#pragma unroll
    for (int k = 0; k < WITEMS; ++k)
        if (kStaged % THREADS == 0 || (int)threadIdx.x + THREADS * k < kStaged) reinterpret_cast<half8*>(s_w)[threadIdx.x + THREADS * k] = staged[k];

    // ... and from the registers into the patch: the 2x upsampling on the way
    auto commit = [&](const Tile& t, int tid, Loads& r)
    {
        const bool interior = t.y0 > 0 && t.x0 > 0 && t.y0 + kConvTileH < p.H && t.x0 + kConvTileW < p.W;
        auto put_image = [&]()
        {
#pragma unroll
            for (int k = 0; k < FITEMS; ++k)
            {
                const int item = tid + THREADS * k;
                if (item < kPatch)
                {
                    const int y = t.y0 + item / kConvPatchW - 1, x = t.x0 + item % kConvPatchW - 1;
                    const bool in = interior || ((unsigned)y < (unsigned)p.H && (unsigned)x < (unsigned)p.W);
                    _Float16* row = s_patch + item * ROW;
                    if (FOUR)
                        *reinterpret_cast<half4*>(row) =
                            in ? half4{_Float16(r.f[k][0]), _Float16(r.f[k][1]), _Float16(r.f[k][2]), _Float16(r.f[k][3])} : half4{};
                    else
                    {
                        // (run-time bounds would put the register array into scratch memory)
#pragma unroll
                        for (int g = 0; g < CI / 4; ++g)
                        {
                            half4 v;
#pragma unroll
                            for (int i = 0; i < 4; ++i) v[i] = in ? _Float16(r.f[k][4 * g + i]) : _Float16(0.f);
                            if (4 * g + 4 <= C)
                                *reinterpret_cast<half4*>(row + 4 * g) = v;
                            else
                            {
#pragma unroll
                                for (int i = 0; i < 3; ++i)
                                    if (4 * g + i < C) row[4 * g + i] = v[i];
                            }
                        }
                    }
                }
            }
        };
        if (FOUR) put_image();
        if (below_groups > 0)
        {
#pragma unroll
            for (int k = 0; k < QITEMS; ++k)
            {
                const int item = tid + THREADS * k;
                const int g = item % GROUPS, quad = item / GROUPS;
                if (quad >= kQuads || g >= below_groups || 8 * g + 8 <= C) continue;
                const int j = quad / (kConvPatchW / 2), i = quad - j * (kConvPatchW / 2);
                half8 v[4];
                upsample_quad(__builtin_bit_cast(half8, r.q[k][0]), __builtin_bit_cast(half8, r.q[k][1]), __builtin_bit_cast(half8, r.q[k][2]),
                              __builtin_bit_cast(half8, r.q[k][3]), t.y0 + j == 0, t.x0 + i == 0, v);
#pragma unroll
                for (int n = 0; n < 4; ++n)
                {
                    const int py = 2 * j + (n >> 1), px = 2 * i + (n & 1);
                    if (!interior && !((unsigned)(t.y0 + py - 1) < (unsigned)p.H && (unsigned)(t.x0 + px - 1) < (unsigned)p.W)) v[n] = half8{};
                    _Float16* dst = s_patch + (py * kConvPatchW + px) * ROW + 8 * g;
                    if (FOUR && g == 0)
                        *reinterpret_cast<half4*>(dst + 4) = half4{v[n][4], v[n][5], v[n][6], v[n][7]};
                    else
                        *reinterpret_cast<half8*>(dst) = v[n];  // (zero where the image goes)
                }
            }
        }
        // A group of eight that holds both is written whole, then the image in 8-byte words and what remains of one: a test
        // and two bytes at a time, on either side, cost a quarter of the level (16 image channels, 64 -> 32 at 960 x 540:
        // 71 -> 49 us, 3 channels, 64 -> 64 at 1920 x 1080: 266 -> 220).
        if (!FOUR && below_groups > 0 && (C & 7)) __syncthreads();
        if (!FOUR) put_image();
    };

    for (; at < last; at += in_xcd)
    {
        const Tile t = decode(at);
        // The thread's number is made anew for every tile: what follows from it (addresses of loads, of the patch, of the
        // staged weights and the weights themselves) would otherwise be kept in registers across the loop, which has
        // none to spare.
        int tid = (int)threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int lane = tid & 63, lrow = lane & 15, lq = lane >> 4;
        if (!kAhead) issue(t, tid, cur);
        __syncthreads();  // the previous tile's patch has been read (and the fills above are done)
        commit(t, tid, cur);
        __syncthreads();
        if (kPrefetch && at + in_xcd < last) issue(decode(at + in_xcd), tid, cur);  // travels during the taps and the epilogue

        int strip = first_strip;
        do  // (a loop with STRIPS = 1 cost the kernel of the finest level 12 spilled registers and a fifth of its time)
        {
            const int r0 = (strip >> 1) * MB, c0 = (strip & 1) * 16;  // the strip's first row and column of the tile
            floatx4 acc[MB][2];
#pragma unroll
            for (int m = 0; m < MB; ++m)
            {
                acc[m][0] = floatx4{bias_f.x, bias_f.y, bias_f.z, bias_f.w};
                acc[m][1] = floatx4{bias_m.x, bias_m.y, bias_m.z, bias_m.w};
            }
            const half8* wlds  = reinterpret_cast<const half8*>(s_w) + pair * (9 * KLDS * 2 * 64) + lane;
            const _Float16* a0 = s_patch + (r0 * kConvPatchW + c0 + lrow) * ROW + lq * 8;
#pragma unroll
            for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                for (int dx = 0; dx < 3; ++dx)
                {
                    half8 b[3][2];
#pragma unroll
                    for (int dy = 0; dy < 3; ++dy)
#pragma unroll
                        for (int h = 0; h < 2; ++h) b[dy][h] = kb < KREG ? w[KREG > 0 ? 3 * dy + dx : 0][kb < KREG ? kb : 0][h] : wlds[(((3 * dy + dx) * KLDS + kb - KREG) * 2 + h) * 64];
#pragma unroll
                    for (int r = 0; r < MB + 2; ++r)
                    {
                        const half8 a = *reinterpret_cast<const half8*>(a0 + (r * kConvPatchW + dx) * ROW + kb * 32);
#pragma unroll
                        for (int dy = 0; dy < 3; ++dy)
                        {
                            const int m = r - dy;
                            if (m < 0 || m >= MB) continue;
                            acc[m][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[dy][0], a, acc[m][0], 0, 0, 0);
                            acc[m][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[dy][1], a, acc[m][1], 0, 0, 0);
                        }
                    }
                }

            // ---- epilogue: elu(feature) * sigmoid(mask); a lane: four channels of one pixel per row of the strip ----
            const int x = t.x0 + c0 + lrow, ch0 = gp * 16 + lq * 4;
            const size_t tile_pix = (size_t)t.image * p.H * p.W + (size_t)t.y0 * p.W + t.x0;
            _Float16* pre_tile    = p.pre ? p.pre + tile_pix * p.npad : nullptr;
            _Float16* out_tile    = p.out ? p.out + tile_pix * p.out_stride : nullptr;
            floatx4 fin = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int m = 0; m < MB; ++m)
            {
                const int y       = t.y0 + r0 + m;
                const bool inside = y < p.H && x < p.W;
                const int pix     = (r0 + m) * p.W + c0 + lrow;  // from the tile's first
                const floatx4 f = acc[m][0], g = acc[m][1];
                if (p.pre && inside)
                {
                    const half8 v = half8{_Float16(f[0]), _Float16(f[1]), _Float16(f[2]), _Float16(f[3]),
                                          _Float16(g[0]), _Float16(g[1]), _Float16(g[2]), _Float16(g[3])};
                    __builtin_nontemporal_store(v, reinterpret_cast<half8*>(pre_tile + pix * p.npad + 2 * ch0));
                }
                half4 o;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                {
                    const float e = f[i] > 0.f ? f[i] : (__expf(f[i]) - 1.f);
                    // v_rcp_f32 is good to 1 ulp of fp32 and the product is rounded to fp16 next: no IEEE division needed
                    const float sg = __builtin_amdgcn_rcpf(1.f + __expf(-g[i]));
                    o[i]           = _Float16(e * sg);
                }
                // padding channels: of an infinite operand their zero weights make not a number, not zero
                if (p.cout & 15)
                {
                    if (p.cout & 3)
                    {
#pragma unroll
                        for (int i = 1; i < 4; ++i) o[i] = ch0 + i < p.cout ? o[i] : _Float16(0.f);
                    }
                    if (ch0 >= p.cout) o = half4{};
                }
                // the image of the pixel, as the convolution saw it: channels lq * 4 .. + 3
                const _Float16* mine = s_patch + ((r0 + m + 1) * kConvPatchW + c0 + lrow + 1) * ROW;
                if (p.out && inside)
                {
                    _Float16* row = out_tile + pix * p.out_stride;
                    const int pos = 2 * C + ch0;
                    if (pos + 4 <= p.out_stride)
                    {
                        if (FOUR || (C & 1) == 0)
                            *reinterpret_cast<half4*>(row + pos) = o;
                        else
                        {
                            typedef _Float16 half2v __attribute__((ext_vector_type(2)));
                            *reinterpret_cast<half2v*>(row + pos)     = half2v{o[0], o[1]};
                            *reinterpret_cast<half2v*>(row + pos + 2) = half2v{o[2], o[3]};
                        }
                    }
                    else
                    {
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            if (pos + i < p.out_stride) row[pos + i] = o[i];
                    }
                    if (gp == 0 && FOUR)
                    {
                        if (lq == 0)
                        {
                            const half4 im                 = *reinterpret_cast<const half4*>(mine);
                            *reinterpret_cast<half8*>(row) = half8{_Float16(0.f), _Float16(0.f), _Float16(0.f), _Float16(0.f), im[0], im[1], im[2], im[3]};
                        }
                    }
                    else if (gp == 0)
                    {
                        // the row's other positions: [0, C) zero, [C, 2C) the image, what the outputs do not reach zero
                        if ((C & 3) == 0)
                        {
                            for (int c = 4 * lq; c < 2 * C; c += 16)
                                *reinterpret_cast<half4*>(row + c) = c < C ? half4{} : *reinterpret_cast<const half4*>(mine + c - C);
                        }
                        else if ((C & 1) == 0)
                        {
                            for (int c = 2 * lq; c < 2 * C; c += 8)
                                *reinterpret_cast<unsigned*>(row + c) = c < C ? 0u : *reinterpret_cast<const unsigned*>(mine + c - C);
                        }
                        else
                        {
                            for (int c = lq; c < C; c += 4) row[c] = _Float16(0.f), row[C + c] = mine[c];
                        }
                        for (int c = 2 * C + p.npad / 2 + lq; c < p.out_stride; c += 4) row[c] = _Float16(0.f);
                    }
                }
                if (p.final_out)
                {
                    // (of the 16 positions that a product takes, those past the image are zero: for four channels read from the
                    // row's padding, else cleared)
                    half4 im = *reinterpret_cast<const half4*>(mine + (FOUR ? (lq == 0 ? 0 : CIN) : CI == 4 ? 0 : lq * 4));
                    if (!FOUR)
                    {
#pragma unroll
                        for (int i = 0; i < 4; ++i) im[i] = lq * 4 + i < C ? im[i] : _Float16(0.f);
                    }
                    floatx4 row     = __builtin_amdgcn_mfma_f32_16x16x16f16(fw, o, floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                    if (pair == 0) row = __builtin_amdgcn_mfma_f32_16x16x16f16(fimg, im, row, 0, 0, 0);
                    fin = lq == m ? row : fin;
                }
            }
            if (p.final_out)
            {
                // lane group m: the outputs of row m, pixel lrow; with two pairs the wavefront of the second one hands over
                // its share of the sums, with more all of them do
                if constexpr (PAIRS > 2)
                {
                    s_fin[(pair * 4 + strip) * 64 + lane] = make_float4(fin[0], fin[1], fin[2], fin[3]);
                    continue;
                }
                if (PAIRS == 2)
                {
                    if (pair == 1) s_fin[strip * 64 + lane] = make_float4(fin[0], fin[1], fin[2], fin[3]);
                    __syncthreads();
                }
                const int y = t.y0 + r0 + lq;
                if (pair == 0 && lq < MB && y < p.H && x < p.W)
                {
                    if (PAIRS == 2)
                    {
                        const float4 o = s_fin[strip * 64 + lane];
                        fin[0] += o.x, fin[1] += o.y, fin[2] += o.z, fin[3] += o.w;
                    }
                    const size_t plane = (size_t)p.H * p.W;
                    float* dst         = p.final_out + (size_t)t.image * p.final_cout * plane + (size_t)y * p.W + x;
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (k < p.final_cout) dst[k * plane] = fin[k] + p.final_b[k];
                }
            }
        } while (STRIPS > 1 && (strip += WAVES / PAIRS) < 16 / MB);
        if (kAhead && !kPrefetch && at + in_xcd < last) issue(decode(at + in_xcd), tid, cur);
        if constexpr (PAIRS > 2)
            if (p.final_out)
            {
                __syncthreads();
                if (tid < kConvTileH * kConvTileW)
                {
                    float4 sum = s_fin[tid];
#pragma unroll
                    for (int j = 1; j < PAIRS; ++j)
                    {
                        const float4 o = s_fin[j * (4 * 64) + tid];
                        sum.x += o.x, sum.y += o.y, sum.z += o.z, sum.w += o.w;
                    }
                    const int of = tid >> 6;  // the pixel's strip: of four rows, whatever the number of pairs
                    const int y = t.y0 + (of >> 1) * 4 + lq, x = t.x0 + (of & 1) * 16 + lrow;
                    if (y < p.H && x < p.W)
                    {
                        const size_t plane = (size_t)p.H * p.W;
                        float* dst         = p.final_out + (size_t)t.image * p.final_cout * plane + (size_t)y * p.W + x;
                        const float f[4]   = {sum.x, sum.y, sum.z, sum.w};
#pragma unroll
                        for (int k = 0; k < 4; ++k)
                            if (k < p.final_cout) dst[k * plane] = f[k] + p.final_b[k];
                    }
                }
            }
    }
}

// Weights of all levels in one launch, the level is blockIdx.y (a launch per level costs more than the work itself):
// MFMA fragments in the order a wavefront reads them, [pair][tap][cin / 32][feature, mask][lane][8]: output pair * 16 +
// lane % 16, input channel 32 kb + (lane / 16) * 8 + i; zero outside the real ranges. Behind them the biases,
// [pair][feature, mask][16]. The finest level's workgroups also pack the 1x1's weights:
// [pair, then the image][output o < 4][quarter q][i]: channel 16 pair + 4 q + i of the block (of the image).
struct PackLevel
{
    const float *wf, *bf, *wm, *bm;
    int cout, cin_real, cin_pad, npad;
    _Float16* wfrag;
    float* bias;
};
struct PackTable
{
    PackLevel lv[TRIPS_UNET_MAX_LEVELS];
    const float* final_w;
    _Float16* fin_frag;
    int c_feat, final_cout;
};
__global__ __launch_bounds__(256) void pack_conv_weights_kernel(const PackTable t)
{
    const PackLevel& l = t.lv[blockIdx.y];
    const int cout = l.cout, cin_real = l.cin_real, npad = l.npad, kbs = l.cin_pad / 32;
    const int total = 9 * npad * l.cin_pad;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256)
    {
        const int e = i & 7, lane = (i >> 3) & 63, h = (i >> 9) & 1;
        const int rest = i >> 10, kb = rest % kbs, tap = (rest / kbs) % 9, pair = rest / (kbs * 9);
        const int o = pair * 16 + (lane & 15), c = kb * 32 + (lane >> 4) * 8 + e;
        float v = 0.f;
        if (o < cout && c < cin_real) v = (h ? l.wm : l.wf)[((size_t)o * cin_real + c) * 9 + tap];
        l.wfrag[i] = _Float16(v);
    }
    for (int n = blockIdx.x * 256 + threadIdx.x; n < npad; n += gridDim.x * 256)
    {
        const int o = (n >> 5) * 16 + (n & 15);
        l.bias[n]   = o < cout ? ((n & 16) ? l.bm : l.bf)[o] : 0.f;
    }
    if (blockIdx.y == 0)
    {
        const int pairs = npad / 32, cin = t.c_feat + cout;
        for (int i = blockIdx.x * 256 + threadIdx.x; i < (pairs + 1) * 64; i += gridDim.x * 256)
        {
            const int pair = i >> 6, o = (i >> 4) & 3, k = i & 15;
            const int c = pair < pairs ? (pair * 16 + k < cout ? t.c_feat + pair * 16 + k : -1) : (k < t.c_feat ? k : -1);
            t.fin_frag[i] = _Float16(o < t.final_cout && c >= 0 ? t.final_w[o * cin + c] : 0.f);
        }
    }
}

// ---------------------------------------------------------------------------------------------------------
namespace
{
template <int CIN, int PAIRS, int CI, bool FOUR, int THREADS, int KREG, int WAVES_PER_EU>
hipError_t launch_conv(const ConvParams& p, int splits, hipStream_t stream)
{
    const long long tiles = (long long)p.tiles * p.batch;
    // as many workgroups as are resident at once
    const int resident = std::max(1, 256 * (4 * WAVES_PER_EU / (THREADS / 64)) / splits);
    const dim3 grid((unsigned)std::min<long long>(tiles, resident), splits);
    hipLaunchKernelGGL((gated_conv3x3_kernel<CIN, PAIRS, CI, FOUR, THREADS, KREG, WAVES_PER_EU>), grid, dim3(THREADS), 0, stream, p);
    return hipGetLastError();
}

template <int CI, bool FOUR>
hipError_t dispatch_conv_ci(const ConvParams& p, int cin_pad, hipStream_t stream)
{
    // Two pairs of outputs per workgroup where there are enough tiles to fill the chip's 256 CUs that way (the patch is
    // then assembled half as often); an odd number of pairs and the coarse levels take one: with a few tiles the level
    // lasts as long as one tile's chain of products, which two pairs double (64 -> 128, 3 tiles: 16 -> 10 us).
    // Three and four pairs go together where every CU has tiles to walk: with 2040 tiles 125 -> 68 us (64 -> 96) and
    // 111 -> 97 us (64 -> 128), with 300 tiles 26 and 27 -> 31 us. The finest level takes all of them in any case: its 1x1
    // needs a whole pixel, and as a kernel of its own, behind rows written for it, it and the patches assembled three and
    // four times took 665 us instead of 252 (1920 x 1080, 64 -> 96) and 717 instead of 370 (64 -> 128).
    const int pairs       = p.npad / 32;
    const long long tiles = (long long)p.tiles * p.batch;
    if (pairs > 2 && (p.final_out || tiles >= 512))
    {
        if (pairs == 3) return cin_pad == 32 ? launch_conv<32, 3, CI, FOUR, 768, 0, 3>(p, 1, stream) : launch_conv<64, 3, CI, FOUR, 768, 1, 3>(p, 1, stream);
        return cin_pad == 32 ? launch_conv<32, 4, CI, FOUR, 1024, 0, 4>(p, 1, stream) : launch_conv<64, 4, CI, FOUR, 512, 2, 2>(p, 1, stream);
    }
    const bool two = pairs % 2 == 0 && (p.final_out || tiles * (pairs / 2) >= 256);
    if (cin_pad == 32) return two ? launch_conv<32, 2, CI, FOUR, 512, 0, 4>(p, pairs / 2, stream) : launch_conv<32, 1, CI, FOUR, 512, 0, (FOUR ? 6 : 4)>(p, pairs, stream);
    return two ? launch_conv<64, 2, CI, FOUR, 512, 2, 2>(p, pairs / 2, stream) : launch_conv<64, 1, CI, FOUR, 512, 2, 2>(p, pairs, stream);
}

// (the kernel is built for exactly 4 image channels and with room for 4, 8 and 16; other counts use the next size up)
hipError_t dispatch_conv(const ConvParams& p, int cin_pad, hipStream_t stream)
{
    if (p.c_feat == 4) return dispatch_conv_ci<4, true>(p, cin_pad, stream);
    if (p.c_feat < 4) return dispatch_conv_ci<4, false>(p, cin_pad, stream);
    if (p.c_feat <= 8) return dispatch_conv_ci<8, false>(p, cin_pad, stream);
    return dispatch_conv_ci<16, false>(p, cin_pad, stream);
}
}  // namespace
}  // namespace trips

using namespace trips;

extern "C" {

int trips_unet_workspace_size(const TripsUnetDesc* desc, size_t* bytes)
{
    if (int e = check_unet_desc(desc)) return e;
    if (!bytes) return set_error(TRIPS_ERR_INVALID_ARG, "bytes is NULL");
    *bytes = make_plan(*desc).bytes;
    return TRIPS_OK;
}

int trips_unet_saved_size(const TripsUnetDesc* desc, size_t* bytes)
{
    if (int e = check_unet_desc(desc)) return e;
    if (!bytes) return set_error(TRIPS_ERR_INVALID_ARG, "bytes is NULL");
    *bytes = make_plan(*desc).saved_bytes;
    return TRIPS_OK;
}

int trips_unet_flops(const TripsUnetDesc* desc, double* flops)
{
    if (int e = check_unet_desc(desc)) return e;
    if (!flops) return set_error(TRIPS_ERR_INVALID_ARG, "flops is NULL");
    const NetPlan np = make_plan(*desc);
    double f         = 0.0;
    for (int i = 0; i < desc->num_levels; ++i)
        f += 2.0 * 2.0 * 9.0 * np.lv[i].cin_real * np.lv[i].cout * (double)np.lv[i].H * np.lv[i].W;
    f += 2.0 * desc->filters[0] * desc->num_output_channels * (double)desc->level_h[0] * desc->level_w[0];
    *flops = f * desc->batch;
    return TRIPS_OK;
}

}  // extern "C"

namespace
{
// hwc: inputs[i] is [batch, level_h, level_w, C] (the splat's eval layout) instead of [batch, C, level_h, level_w]
int unet_forward(TripsCtx* ctx, const TripsUnetDesc* desc, const TripsUnetWeights* weights,
                 const float* const inputs[TRIPS_UNET_MAX_LEVELS], bool hwc, float* output, void* saved, void* workspace,
                 size_t workspace_bytes, void* stream_)
{
    if (!ctx) return set_error(TRIPS_ERR_INVALID_ARG, "ctx is NULL");
    if (int e = check_unet_desc(desc)) return e;
    if (!weights || !inputs || !output || !workspace) return set_error(TRIPS_ERR_INVALID_ARG, "NULL argument");
    const TripsUnetDesc& d = *desc;
    const int C = d.num_input_channels, L = d.num_levels;
    for (int i = 0; i < L; ++i)
    {
        if (!inputs[i]) return set_error(TRIPS_ERR_INVALID_ARG, "inputs[%d] is NULL", i);
        if (!weights->feature_weight[i] || !weights->feature_bias[i] || !weights->mask_weight[i] || !weights->mask_bias[i])
            return set_error(TRIPS_ERR_INVALID_ARG, "weights of block %d are NULL", i);
    }
    if (!weights->final_weight || !weights->final_bias) return set_error(TRIPS_ERR_INVALID_ARG, "final weights are NULL");
    if ((reinterpret_cast<uintptr_t>(workspace) & 255) || (reinterpret_cast<uintptr_t>(saved) & 255))
        return set_error(TRIPS_ERR_INVALID_ARG, "workspace / saved must be 256-byte aligned");
    const NetPlan np = make_plan(d);
    if (workspace_bytes < np.bytes)
        return set_error(TRIPS_ERR_WORKSPACE_SMALL, "workspace has %zu bytes, %zu needed", workspace_bytes, np.bytes);
    hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
    char* ws           = reinterpret_cast<char*>(workspace);
    char* sv           = reinterpret_cast<char*>(saved);
    Profiler* prof     = ctx->prof.enabled ? &ctx->prof : nullptr;
    // the rows of a level live in the saved state when there is one (the backward reads them), else in the workspace
    auto rows_ptr = [&](int level) { return reinterpret_cast<_Float16*>(sv && level > 0 ? sv + np.lv[level].saved_rows_off : ws + np.lv[level].rows_off); };

    if (!d.weights_packed)
    {
        ProfScope ps(prof, "unet_pack_weights", stream);
        PackTable pt;
        int most = 0;
        for (int i = 0; i < L; ++i)
        {
            const LevelPlan& lv = np.lv[i];
            pt.lv[i] = PackLevel{weights->feature_weight[i], weights->feature_bias[i], weights->mask_weight[i], weights->mask_bias[i],
                                 lv.cout, lv.cin_real, lv.cin_pad, lv.npad, reinterpret_cast<_Float16*>(ws + lv.wpack_off),
                                 reinterpret_cast<float*>(ws + lv.bias_off)};
            most     = std::max(most, 9 * lv.npad * lv.cin_pad);
        }
        pt.final_w    = weights->final_weight;
        pt.fin_frag   = reinterpret_cast<_Float16*>(ws + np.fin_off);
        pt.c_feat     = C;
        pt.final_cout = d.num_output_channels;
        hipLaunchKernelGGL(pack_conv_weights_kernel, dim3((most + 255) / 256, L), dim3(256), 0, stream, pt);
    }
    static const char* const kLevelNames[TRIPS_UNET_MAX_LEVELS] = {"unet_conv_l0", "unet_conv_l1", "unet_conv_l2", "unet_conv_l3",
                                                                   "unet_conv_l4", "unet_conv_l5", "unet_conv_l6", "unet_conv_l7"};
    for (int i = L - 1; i >= 0; --i)
    {
        const LevelPlan& lv = np.lv[i];
        ProfScope ps(prof, kLevelNames[i], stream);
        ConvParams p;
        std::memset(&p, 0, sizeof(p));
        p.H       = lv.H;
        p.W       = lv.W;
        p.c_feat  = C;
        p.cout    = lv.cout;
        p.npad    = lv.npad;
        p.tiles_x = (lv.W + kConvTileW - 1) / kConvTileW;
        p.tiles   = p.tiles_x * ((lv.H + kConvTileH - 1) / kConvTileH);
        p.batch   = d.batch;
        p.feat    = inputs[i];
        p.feat_ps = hwc ? C : 1;
        p.feat_cs = hwc ? 1 : (size_t)lv.H * lv.W;
        p.wfrag   = reinterpret_cast<const _Float16*>(ws + lv.wpack_off);
        p.bias    = reinterpret_cast<const float*>(ws + lv.bias_off);
        // (nobody reads the finest block's output again: its 1x1 runs in the same kernel, and the backward takes it from
        // the pre-activations)
        p.out        = i > 0 ? rows_ptr(i) : nullptr;
        p.out_stride = lv.row_stride;
        p.pre        = sv ? reinterpret_cast<_Float16*>(sv + lv.saved_pre_off) : nullptr;
        if (i < L - 1)
        {
            p.Hb           = np.lv[i + 1].H;
            p.Wb           = np.lv[i + 1].W;
            p.below        = rows_ptr(i + 1);
            p.below_stride = np.lv[i + 1].row_stride;
        }
        if (i == 0)
        {
            p.fin_frag   = reinterpret_cast<const _Float16*>(ws + np.fin_off);
            p.final_b    = weights->final_bias;
            p.final_out  = output;
            p.final_cout = d.num_output_channels;
        }
        hipError_t e = dispatch_conv(p, lv.cin_pad, stream);
        if (e != hipSuccess) return set_error(TRIPS_ERR_HIP, "gated conv launch (level %d): %s", i, hipGetErrorString(e));
    }
    return TRIPS_OK;
}
}  // namespace

extern "C" {

int trips_unet_forward(TripsCtx* ctx, const TripsUnetDesc* desc, const TripsUnetWeights* weights,
                       const float* const inputs[TRIPS_UNET_MAX_LEVELS], float* output, void* saved, void* workspace,
                       size_t workspace_bytes, void* stream)
{
    return unet_forward(ctx, desc, weights, inputs, false, output, saved, workspace, workspace_bytes, stream);
}

int trips_unet_forward_hwc(TripsCtx* ctx, const TripsUnetDesc* desc, const TripsUnetWeights* weights,
                           const float* const inputs[TRIPS_UNET_MAX_LEVELS], float* output, void* workspace, size_t workspace_bytes,
                           void* stream)
{
    return unet_forward(ctx, desc, weights, inputs, true, output, nullptr, workspace, workspace_bytes, stream);
}

}  // extern "C"
