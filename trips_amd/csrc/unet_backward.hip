// Backward of the decoder-only gated-convolution U-Net on the gfx950 matrix cores: what libtorch's autograd does
// for MultiScaleUnet2dDecOnlySmallFixedImpl::forward in the reference (src/lib/models/Networks.h:1139-1191, blocks
// at :751-787 and :999-1098), as hand-written kernels over the state the training forward saved.
//
//   final_backward_kernel     1x1 output convolution: gradient of x_0, split into dL/d in[0] and, through the gate,
//                             the gradient of the finest block's pre-activations; its weight and bias gradients
//   conv_bwd_data_kernel      gradient of a block's input: the forward's implicit GEMM with flipped, transposed
//                             weights (M = 256 pixels, N = input channels, K = 9 taps x pre-activations)
//   conv_bwd_data_up_kernel   these two in one, for blocks of few enough channels
//   up2_adjoint_gate_kernel   adjoint of the bilinear 2x upsampling (a gather over <= 4 x 4 finer pixels), then
//                             dL/d in[i+1] and the gate of the coarser block
//   conv_bwd_weight_kernel    weight gradients: GEMM with the pixels as the reduction dimension. Both operands are
//                             needed pixel-contiguous; the tiles stay pixel-major in LDS, as they are assembled, and
//                             the operands are fetched with the transposing LDS read (ds_read_b64_tr_b16);
//                             persistent workgroups keep their partial sums in registers over many tiles; the
//                             bias gradients (sums of the pre-activation gradients) are one more MFMA per tile row
//                             against a matrix of ones
//   bias_grad_kernel          bias gradients alone, when no weight gradient is asked for
//   reduce_weight_grad_kernel
//
// Intermediate gradients are fp16 and carried multiplied by grad_scale; every fp32 result is divided by it again.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "unet_common.h"

namespace trips
{

// d(elu(f) * sigmoid(m)) for an incoming gradient da
// (`act`: the gated value itself, elu(f) * sigmoid(m), with the forward's formula)
__device__ __forceinline__ void gate_backward(float da, float f, float m, float& df, float& dm, float& act)
{
    const float s  = __builtin_amdgcn_rcpf(1.f + __expf(-m));  // 1 ulp; the gradients are rounded to fp16 next
    const float ex = __expf(f);
    const float e  = f > 0.f ? f : ex - 1.f;
    const float de = f > 0.f ? 1.f : ex;
    df             = da * s * de;
    dm             = da * e * s * (1.f - s);
    act            = e * s;
}
__device__ __forceinline__ void gate_backward(float da, float f, float m, float& df, float& dm)
{
    float act;
    gate_backward(da, f, m, df, dm, act);
}

// wt[tap'][c][n] = W[n][c][8 - tap']: the data gradient is a correlation of the pre-activation gradient with the
// spatially flipped kernel, input and output channels exchanged
// (all levels in one launch, the level is blockIdx.y: a launch per level costs more than the work itself)
struct PackTLevel
{
    const float *wf, *wm;
    int cout, cin_real, cin_pad, npad;
    _Float16* wt;
};
struct PackTTable
{
    PackTLevel lv[TRIPS_UNET_MAX_LEVELS];
};
__global__ __launch_bounds__(256) void pack_conv_weights_T_kernel(const PackTTable t)
{
    const PackTLevel& l = t.lv[blockIdx.y];
    const float* __restrict__ wf = l.wf;
    const float* __restrict__ wm = l.wm;
    const int cout = l.cout, cin_real = l.cin_real, cin_pad = l.cin_pad, npad = l.npad;
    _Float16* __restrict__ wt = l.wt;
    const int total = 9 * cin_pad * npad;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256)
    {
        const int n = i % npad, c = (i / npad) % cin_pad, tap = i / (npad * cin_pad);
        const int o = preact_channel(n);
        float v     = 0.f;
        if (o < cout && c < cin_real) v = (preact_is_mask(n) ? wm : wf)[((size_t)o * cin_real + c) * 9 + (8 - tap)];
        wt[i] = _Float16(v);
    }
}

__global__ __launch_bounds__(256) void fill_f32_kernel(float* __restrict__ p, float v, int n)
{
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) p[i] = v;
}

struct FinalBwdParams
{
    int H, W, c_feat, cact, cout;
    float scale;
    const float* feat;        // [C][H][W]
    const _Float16* pre;      // [H][W][NPAD]
    const float* weight;      // [cout][c_feat + cact]
    const float* d_out;       // [cout][H][W]
    float* d_feat;            // [C][H][W], written
    _Float16* dpre;           // [H][W][NPAD], written
    float* part;              // [gridDim.x][4 * (4 + CS) + 4] sums of this launch's workgroups (WGRAD)
    int chunks;               // of one image: ceil(pixels / kFinalPixelsPerBlock)
    int batch;                // images, one after the other in every array
};

// One pass over the pixels of the finest level: dL/d in[0], the gated block's pre-activation gradients and, when
// WGRAD, the weight and bias gradients of the 1x1 convolution. Every thread keeps the cout x cin products of its
// pixels in registers, a workgroup folds them through LDS and writes its sums once (final_reduce_kernel adds the
// workgroups up: atomics of a thousand workgroups on these few addresses would serialise in one L2 channel).
// (The library is compiled without contraction of products and sums; here the sums are written as fused multiply-adds.)
// Bound by the memory: about 300 bytes a pixel at 64 gates, most of them the rows that it reads and the rows that it
// writes. The rows it reads are read for the last time, whole lines of them by a wavefront, and are loaded past the caches:
// loaded as usual they push out the rows that are written, which the data gradient reads next. 1245 x 825 pixels: 96 us, 71
// with the loads past the caches (and the data gradient of the level 113, now 106), 4.3 TB/s; four crops of 512^2: 83, now
// 64; 1717 x 783 at 32 gates: 71, now 57, all with caches that other data has been through; in a loop over the same buffers
// the loads past the caches change nothing and the workgroups and chunks (unet_common.h) save 1 % of a training step on the crops. Two or four pixels
// of a lane requested together gave nothing (86 and 93 us where one gave 84): the registers cost as many wavefronts as they
// add loads.
// CI = image channels the kernel has room for (4, 8 or 16).
template <int NPAD, bool WGRAD, int CI>
__global__ __launch_bounds__(256) void final_backward_kernel(const FinalBwdParams p)
{
    constexpr int CS   = NPAD / 2;  // block outputs, padded
    constexpr int MAXC = CI + CS;
    // LPP lanes share a pixel, one per 16 bytes of its pre-activation row (the features and the masks of four channels),
    // so that a wavefront reads and writes whole lines of the channels-innermost arrays.
    constexpr int LPP = NPAD <= 32 ? 4 : NPAD <= 64 ? 8 : 16;
    constexpr int PPW = 64 / LPP;  // pixels per wavefront and iteration
    __shared__ float s_w[4 * MAXC];
    __shared__ float s_sum[4 * MAXC + 4];
    const int cin = p.c_feat + p.cact;
    // weights as the forward used them (fp16), laid out [k][CI image channels | CS block outputs], zero where unused
    for (int i = threadIdx.x; i < 4 * MAXC; i += 256)
    {
        const int k = i / MAXC, r = i - k * MAXC;
        const int c = r < CI ? (r < p.c_feat ? r : -1) : (r - CI < p.cact ? p.c_feat + r - CI : -1);
        s_w[i]      = (k < p.cout && c >= 0) ? float(_Float16(p.weight[k * cin + c])) : 0.f;
    }
    for (int i = threadIdx.x; i < 4 * MAXC + 4; i += 256) s_sum[i] = 0.f;
    __syncthreads();
    const size_t plane = (size_t)p.H * p.W;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int g = lane % LPP, sub = lane / LPP;
    // lanes past the row (rows of 96 halves on 16 lanes) work on its first word again and store nothing
    const bool in_row = NPAD / 8 == LPP || g < NPAD / 8;
    const int row_word = in_row ? 8 * g : 0;
    const int c0      = 4 * g;         // first of this lane's four channels
    // ... and the image channels g, g + LPP, ... (one each for up to LPP image channels)
    constexpr int NI = (CI + LPP - 1) / LPP;
    bool has_img[NI];
#pragma unroll
    for (int j = 0; j < NI; ++j) has_img[j] = g + LPP * j < p.c_feat;
    float wj[4][4], wimg[4][NI];
#pragma unroll
    for (int k = 0; k < 4; ++k)
    {
#pragma unroll
        for (int j = 0; j < NI; ++j) wimg[k][j] = has_img[j] ? s_w[k * MAXC + g + LPP * j] : 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) wj[k][i] = in_row ? s_w[k * MAXC + CI + c0 + i] : 0.f;
    }
    float acc[4][4];
    float acc_img[4][NI], accb[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc_img[k][j] = 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[k][i] = 0.f;

    struct Loaded
    {
        float g[4], x[NI];
        half8 mine;
    };
    constexpr int STEP = 4 * PPW;  // pixels per iteration of the workgroup
    for (int item = blockIdx.x; item < p.chunks * p.batch; item += gridDim.x)
    {
        const int image = item / p.chunks, chunk = item - image * p.chunks;
        const size_t first = (size_t)chunk * kFinalPixelsPerBlock;
        const int n        = (int)std::min(plane - first, (size_t)kFinalPixelsPerBlock);
        // the arrays from the chunk's first pixel on: what a lane adds to them fits in 32 bits
        const float* d_out  = p.d_out + (size_t)image * p.cout * plane + first;
        const float* feat   = p.feat + (size_t)image * p.c_feat * plane + first;
        float* d_feat       = p.d_feat + (size_t)image * p.c_feat * plane + first;
        const _Float16* pre = p.pre + ((size_t)image * plane + first) * NPAD;
        _Float16* dpre      = p.dpre + ((size_t)image * plane + first) * NPAD;
        const float* x_of[NI];
        float* dx_of[NI];
#pragma unroll
        for (int j = 0; j < NI; ++j)
        {
            const size_t at = has_img[j] ? (size_t)(g + LPP * j) * plane : 0;
            x_of[j]  = feat + at;
            dx_of[j] = d_feat + at;
        }
        // (pixels past the end: the last one's values, which are not used; a load behind a condition of the lane costs more
        // than the load)
        auto load = [&](unsigned pix)
        {
            Loaded l;
            const unsigned at = min(pix, (unsigned)n - 1u);
#pragma unroll
            for (int k = 0; k < 4; ++k)
            {
                l.g[k] = 0.f;
                if (k < p.cout) l.g[k] = (d_out + k * plane)[at];
            }
#pragma unroll
            for (int j = 0; j < NI; ++j) l.x[j] = WGRAD ? x_of[j][at] : 0.f;
            l.mine = __builtin_nontemporal_load(reinterpret_cast<const half8*>(pre + (at * NPAD + row_word)));
            return l;
        };
        unsigned pix = wave * PPW + sub;
        Loaded next  = load(pix);
        for (int base = 0; base < n; base += STEP, pix += STEP)
        {
            const Loaded cur = next;
            if (base + STEP < n) next = load(pix + STEP);  // in flight while this pixel is worked on
            if (pix >= (unsigned)n) continue;
            half8 out;   // gradients of the four features, then of the four masks
            float v[4];  // the block's output as the forward's 1x1 convolution read it (fp16)
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                float da = 0.f;
#pragma unroll
                for (int k = 0; k < 4; ++k) da = __builtin_fmaf(wj[k][i], cur.g[k], da);
                float df, dm, a;
                gate_backward(da * p.scale, float(cur.mine[i]), float(cur.mine[4 + i]), df, dm, a);
                out[i]     = _Float16(df);
                out[4 + i] = _Float16(dm);
                v[i]       = float(_Float16(a));  // (sums of padding channels are not read)
            }
            if (in_row) *reinterpret_cast<half8*>(dpre + (pix * NPAD + row_word)) = out;
#pragma unroll
            for (int j = 0; j < NI; ++j)
            {
                float d = 0.f;
#pragma unroll
                for (int k = 0; k < 4; ++k) d = __builtin_fmaf(wimg[k][j], cur.g[k], d);
                if (has_img[j]) dx_of[j][pix] = d;
            }
            if (WGRAD)
            {
                float xr[NI];
#pragma unroll
                for (int j = 0; j < NI; ++j) xr[j] = float(_Float16(cur.x[j]));
#pragma unroll
                for (int k = 0; k < 4; ++k)
                {
                    accb[k] += cur.g[k];
#pragma unroll
                    for (int j = 0; j < NI; ++j) acc_img[k][j] = __builtin_fmaf(cur.g[k], xr[j], acc_img[k][j]);
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[k][i] = __builtin_fmaf(cur.g[k], v[i], acc[k][i]);
                }
            }
        }
    }
    if (!WGRAD) return;
    // fold the lanes that hold the same channels with a butterfly first: many lanes adding to one LDS address would
    // be serialised
    auto fold = [](float v)
    {
#pragma unroll
        for (int o = 32; o >= LPP; o >>= 1) v += __shfl_xor(v, o);
        return v;
    };
#pragma unroll
    for (int k = 0; k < 4; ++k)
    {
        const float b = fold(accb[k]);
        if (lane == 0) atomicAdd(&s_sum[4 * MAXC + k], b);
#pragma unroll
        for (int j = 0; j < NI; ++j)
        {
            const float im = fold(acc_img[k][j]);
            if (lane < LPP && has_img[j]) atomicAdd(&s_sum[k * MAXC + g + LPP * j], im);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
        {
            const float v = fold(acc[k][i]);
            if (lane < LPP && in_row) atomicAdd(&s_sum[k * MAXC + CI + c0 + i], v);
        }
    }
    __syncthreads();
    float* part = p.part + (size_t)blockIdx.x * (4 * MAXC + 4);
    for (int t = threadIdx.x; t < 4 * MAXC + 4; t += 256) part[t] = s_sum[t];
}

// Adds up `rows` partial-sum rows of `cols` floats: workgroup c sums column c, thread 0 holds the result.
__device__ __forceinline__ float block_column_sum(const float* __restrict__ part, int rows, int cols, int c)
{
    __shared__ float s_red[4];
    float s = 0.f;
    for (int r = threadIdx.x; r < rows; r += 256) s += part[(size_t)r * cols + c];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = s;
    __syncthreads();
    return (s_red[0] + s_red[1]) + (s_red[2] + s_red[3]);
}

// d_weight [cout][c_feat + cact] and d_bias [cout] of the 1x1 convolution from final_backward_kernel's partial sums
// (row layout [k][ci image channels | CS block outputs], then 4 biases; maxc = ci + CS); one workgroup per result
__global__ __launch_bounds__(256) void final_reduce_kernel(const float* __restrict__ part, int rows, int maxc, int ci, int c_feat, int cact,
                                                           int cout, float* __restrict__ d_weight, float* __restrict__ d_bias)
{
    const int cin = c_feat + cact;
    const int t   = blockIdx.x;  // < cout * cin + cout
    int col;
    float* dst;
    if (t < cout * cin)
    {
        const int k = t / cin, c = t - k * cin;
        col = k * maxc + (c < c_feat ? c : ci + (c - c_feat));
        dst = d_weight + t;
    }
    else
    {
        col = 4 * maxc + (t - cout * cin);
        dst = d_bias + (t - cout * cin);
    }
    if (!(t < cout * cin ? d_weight : d_bias)) return;  // the caller asked for one of the two only
    const float s = block_column_sum(part, rows, 4 * maxc + 4, col);
    if (threadIdx.x == 0) *dst = s;
}

// ---------------------------------------------------------------------------------------------------------
// The 9-tap implicit-GEMM core of the data gradient. A operands are 16-byte LDS reads from a (8+2) x (32+2) pixel patch with
// KIN channels innermost (row stride KIN + 8 halves). B operands (packed weights [tap][NOUT][KIN]) reach the matrix cores
// through LDS as well: with every wavefront loading its own fragments from memory, each of a tile's wavefronts pulled the
// level's whole weight set out of the L2 again, and that traffic, not the MFMAs, set the length of the tap loop. The rows
// have the patch's bank-conflict-free layout. A tap's MFMAs take far less time than a round trip to the L2, so as many taps
// as the LDS has room for are staged together: all nine (requested when the kernel starts; the tap loop then has neither
// loads nor barriers), or three (the next three travel in registers while these are multiplied; two barriers per three
// taps), or one (two buffers, one barrier per tap).
// Each of the workgroup's eight wavefronts owns one row of the 8 x 32 output tile = two 16-pixel row blocks; acc[m][n] is
// the 16 x 16 block of pixels m, outputs 16n .. 16n+15.
constexpr int kTapThreads  = 512;
constexpr int kTapLdsBytes = 28 * 1024;  // LDS that the staged taps of a workgroup may take
template <int KIN, int NOUT>
struct ConvTapStage
{
    static constexpr int NB    = NOUT / 16;
    static constexpr int KB    = KIN / 32;
    static constexpr int ROW   = KIN + kLdsChanPad;   // halves per output row of a tap in LDS
    static constexpr int ITEMS = NOUT * KIN / 8;      // 16-byte words per tap
    static constexpr int MB    = 16 / (kTapThreads / 64);  // 16-pixel row blocks of a wavefront
    static constexpr int BUF   = NOUT * ROW;           // halves per tap in LDS
    // taps staged together
    static constexpr int T = 9 * BUF * 2 <= kTapLdsBytes ? 9 : 3 * BUF * 2 <= kTapLdsBytes ? 3 : 1;
    static constexpr int STAGE_ITEMS = T * ITEMS;      // 16-byte words per stage
    static constexpr int PER   = (STAGE_ITEMS + kTapThreads - 1) / kTapThreads;  // per thread
    static constexpr int LDS_HALVES = (T == 1 ? 2 : T) * BUF;  // what the kernel provides at s_taps
    half8 r[PER];
};

// this thread's share of taps `tap` .. `tap` + T - 1 from memory into registers (the packed weights are dense:
// [tap][NOUT][KIN])
template <int KIN, int NOUT>
__device__ __forceinline__ void conv_tap_fetch(ConvTapStage<KIN, NOUT>& st, const _Float16* __restrict__ wpack, int tap)
{
    using S = ConvTapStage<KIN, NOUT>;
    const half8* src = reinterpret_cast<const half8*>(wpack + (size_t)tap * NOUT * KIN);
#pragma unroll
    for (int j = 0; j < S::PER; ++j)
    {
        const int item = threadIdx.x + kTapThreads * j;
        if (S::STAGE_ITEMS % kTapThreads == 0 || item < S::STAGE_ITEMS) st.r[j] = src[item];
    }
}

// ... and from the registers into the tap buffers at s_tap (T of them, one after the other)
template <int KIN, int NOUT>
__device__ __forceinline__ void conv_tap_stage(const ConvTapStage<KIN, NOUT>& st, _Float16* s_tap)
{
    using S = ConvTapStage<KIN, NOUT>;
#pragma unroll
    for (int j = 0; j < S::PER; ++j)
    {
        const int item = threadIdx.x + kTapThreads * j;
        if (S::STAGE_ITEMS % kTapThreads == 0 || item < S::STAGE_ITEMS)
        {
            const int t = item / S::ITEMS, w = item - t * S::ITEMS;
            *reinterpret_cast<half8*>(s_tap + t * S::BUF + (w / (KIN / 8)) * S::ROW + (w % (KIN / 8)) * 8) = st.r[j];
        }
    }
}

// Precondition: the first T taps sit at s_taps (conv_tap_fetch(.., 0) + conv_tap_stage) and a barrier has passed since.
// Every thread of the workgroup must call this (it contains barriers unless all nine taps are staged).
// Result layout: lane l holds, of the 16 x 16 block acc[m][n], outputs 16n + (l / 16) * 4 .. + 3 of pixel l % 16, four
// neighbouring channels of one pixel, which an epilogue can store as one 8-byte word (the weights are the MFMA's A operand).
template <int KIN, int NOUT>
__device__ __forceinline__ void conv_taps_mfma(const _Float16* s_patch, _Float16* s_taps, const _Float16* __restrict__ wpack,
                                               ConvTapStage<KIN, NOUT>& st,
                                               floatx4 (&acc)[ConvTapStage<KIN, NOUT>::MB][NOUT / 16])
{
    using S = ConvTapStage<KIN, NOUT>;
    constexpr int MB = S::MB;
    constexpr int ROW = KIN + kLdsChanPad;
    constexpr int NB  = S::NB;
    constexpr int KB  = S::KB;
    constexpr int T   = S::T;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lrow = lane & 15, lk = (lane >> 4) * 8;
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int n = 0; n < NB; ++n) acc[m][n] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int tap = 0; tap < 9; ++tap)
    {
        const int dy = tap / 3, dx = tap - dy * 3;  // patch coordinates already include the halo
        // the next stage's weights: requested before this stage's first tap is multiplied
        if (T < 9 && tap % T == 0 && tap + T < 9) conv_tap_fetch(st, wpack, tap + T);
        const _Float16* sb = s_taps + (T == 1 ? tap & 1 : tap % T) * S::BUF;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
        {
            half8 bfrag[NB];
#pragma unroll
            for (int n = 0; n < NB; ++n) bfrag[n] = *reinterpret_cast<const half8*>(sb + (n * 16 + lrow) * S::ROW + kb * 32 + lk);
#pragma unroll
            for (int m = 0; m < MB; ++m)
            {
                const int r = wave, cb = m * 16;
                const half8 a = *reinterpret_cast<const half8*>(s_patch + ((r + dy) * kConvPatchW + cb + lrow + dx) * ROW + kb * 32 + lk);
#pragma unroll
                for (int n = 0; n < NB; ++n)
                    acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bfrag[n], a, acc[m][n], 0, 0, 0);
            }
        }
        if (T == 1)
        {
            if (tap + 1 < 9) conv_tap_stage(st, s_taps + ((tap + 1) & 1) * S::BUF);
            __syncthreads();  // the next tap is in place; nobody reads this tap's buffer any more
        }
        else if (T < 9 && tap % T == T - 1 && tap + 1 < 9)
        {
            __syncthreads();  // nobody reads this stage's taps any more
            conv_tap_stage(st, s_taps);
            __syncthreads();  // the next stage is in place
        }
    }
    if (T != 1) __syncthreads();  // (as after the last tap of the one-tap form: patch and taps may be overwritten now)
}

// Copies `groups` x 8 halves per pixel of an 8 x 32 tile staged in LDS ([256][lds_stride]) to a channels-innermost
// image ([H][W][dst_stride]) with 16-byte stores: consecutive lanes write consecutive 16 bytes, so a tile row leaves
// as whole lines (2-byte stores straight from the MFMA result layout cost twice the memory requests).
__device__ __forceinline__ void store_tile_nhwc(const _Float16* s_tile, int lds_stride, int groups, _Float16* dst,
                                                int dst_stride, int x0, int y0, int W, int H)
{
    for (int item = threadIdx.x; item < kConvTileH * kConvTileW * groups; item += kTapThreads)
    {
        const int g = item % groups, tp = item / groups;
        const int y = y0 + tp / kConvTileW, x = x0 + tp % kConvTileW;
        if (y < H && x < W)
            *reinterpret_cast<half8*>(dst + ((size_t)y * W + x) * dst_stride + 8 * g) =
                *reinterpret_cast<const half8*>(s_tile + (size_t)tp * lds_stride + 8 * g);
    }
}

struct BwdDataParams
{
    int H, W, c_feat;
    float scale_inv;
    const _Float16* dpre;  // [H][W][KC]
    const _Float16* wt;    // [9][NN][KC]
    float* d_feat;         // [C][H][W], accumulated
    _Float16* d_in;        // [H][W][NN] or nullptr (start block: nothing below)
    int first_image;       // images of a batch: the grid's z dimension, one after the other in every array
};

// CI = image channels the kernel has room for (4, 8 or 16): positions [0, C) of the block input are the level's image.
template <int KC, int NN, int CI>
__global__ __launch_bounds__(kTapThreads) void conv_bwd_data_kernel(BwdDataParams p)
{
    {
        const size_t pixels = (size_t)(p.first_image + blockIdx.z) * p.H * p.W;
        p.dpre += pixels * KC;
        p.d_feat += pixels * p.c_feat;
        p.d_in = p.d_in ? p.d_in + pixels * NN : nullptr;
    }
    constexpr int THREADS = kTapThreads, MB = ConvTapStage<KC, NN>::MB;
    constexpr int ROW    = KC + kLdsChanPad;
    constexpr int GROUPS = KC / 8;
    constexpr int NB     = NN / 16;
    extern __shared__ _Float16 smem[];
    _Float16* s_patch = smem;
    const int x0 = blockIdx.x * kConvTileW, y0 = blockIdx.y * kConvTileH;
    ConvTapStage<KC, NN> taps;
    conv_tap_fetch(taps, p.wt, 0);  // in flight while the patch is loaded
    _Float16* s_taps = s_patch + kConvPatchH * kConvPatchW * ROW;  // the staged taps of the weights
    // the patch of pre-activation gradients, four 16-byte loads of a thread in flight together
    constexpr int kItems = kConvPatchH * kConvPatchW * GROUPS;
    for (int item0 = threadIdx.x; item0 < kItems; item0 += 4 * THREADS)
    {
        // (every load unconditional, at a position clamped into the image, and all four requested before the first is
        // used: a load under a condition is waited for where the condition ends)
        uint4 raw[4];
        bool in[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            const int item = min(item0 + THREADS * j, kItems - 1);
            const int g = item % GROUPS, pp = item / GROUPS;
            const int py = pp / kConvPatchW, px = pp - py * kConvPatchW;
            const int y = y0 + py - 1, x = x0 + px - 1;
            in[j]  = y >= 0 && y < p.H && x >= 0 && x < p.W;
            raw[j] = *reinterpret_cast<const uint4*>(p.dpre + ((size_t)min(max(y, 0), p.H - 1) * p.W + min(max(x, 0), p.W - 1)) * KC + 8 * g);
        }
        half8 v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            asm volatile("" : "+v"(raw[j].x), "+v"(raw[j].y), "+v"(raw[j].z), "+v"(raw[j].w));
            if (!in[j]) raw[j] = make_uint4(0u, 0u, 0u, 0u);
            v[j] = __builtin_bit_cast(half8, raw[j]);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            const int item = item0 + THREADS * j;
            if (item < kItems) *reinterpret_cast<half8*>(s_patch + (size_t)(item / GROUPS) * ROW + 8 * (item % GROUPS)) = v[j];
        }
    }
    conv_tap_stage(taps, s_taps);
    __syncthreads();
    floatx4 acc[MB][NB];
    conv_taps_mfma<KC, NN>(s_patch, s_taps, p.wt, taps, acc);  // a lane: four channels of one pixel
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lrow = lane & 15;
    // ---- epilogue: the tile staged in LDS (the patch is no longer needed) and written channels innermost with
    // 16-byte stores, whole lines at a time; the image channels' share kept in fp32 beside it ----
    constexpr int OS   = NN + kLdsChanPad;
    _Float16* s_out    = smem;                                                                   // [256][OS]
    float* s_img       = reinterpret_cast<float*>(smem + kConvTileH * kConvTileW * OS);          // [CI][256]
    __syncthreads();  // every wavefront is done reading the patch
#pragma unroll
    for (int m = 0; m < MB; ++m)
    {
        const int tp = wave * kConvTileW + m * 16 + lrow;  // this lane's pixel of the block
#pragma unroll
        for (int n = 0; n < NB; ++n)
        {
            const int c0 = 16 * n + (lane >> 4) * 4;  // this lane's four channels
            *reinterpret_cast<half4*>(s_out + tp * OS + c0) =
                half4{_Float16(acc[m][n][0]), _Float16(acc[m][n][1]), _Float16(acc[m][n][2]), _Float16(acc[m][n][3])};
            if (n == 0 && c0 < CI)
            {
#pragma unroll
                for (int i = 0; i < 4; ++i) s_img[(c0 + i) * (kConvTileH * kConvTileW) + tp] = acc[m][0][i];
            }
        }
    }
    __syncthreads();
    if (p.d_in) store_tile_nhwc(s_out, OS, NN / 8, p.d_in, NN, x0, y0, p.W, p.H);
    {
        const size_t plane = (size_t)p.H * p.W;
        const int y = y0 + threadIdx.x / kConvTileW, x = x0 + threadIdx.x % kConvTileW;
        if ((int)threadIdx.x < kConvTileH * kConvTileW && y < p.H && x < p.W)
        {
            float old[CI];
#pragma unroll
            for (int c = 0; c < CI; ++c) old[c] = c < p.c_feat ? p.d_feat[c * plane + (size_t)y * p.W + x] : 0.f;
#pragma unroll
            for (int c = 0; c < CI; ++c)
                if (c < p.c_feat) p.d_feat[c * plane + (size_t)y * p.W + x] = old[c] + s_img[c * (kConvTileH * kConvTileW) + threadIdx.x] * p.scale_inv;
        }
    }
}

// ---------------------------------------------------------------------------------------------------------
struct UpAdjointParams
{
    int H, W;      // finer level, whose block input gradient is given
    int Hb, Wb;    // this (coarser) level
    int cin_fine;  // halves per pixel of d_in
    int c_feat, cout, npad;
    float scale_inv;
    const _Float16* d_in;  // [H][W][cin_fine]: position k = channel k of cat(in, up2(x))
    const _Float16* pre;   // [Hb][Wb][npad]
    float* d_feat;         // [C][Hb][Wb], written
    _Float16* dpre;        // [Hb][Wb][npad], written
    int first_image;       // images of a batch: the grid's y dimension
};

// weight with which finer row / column `dst` reads coarser row / column `src`
__device__ __forceinline__ float up2_weight(int dst, int fine_size, int src, int coarse_size)
{
    if (dst < 0 || dst >= fine_size) return 0.f;
    int i0, i1;
    float l;
    up2_source(dst, coarse_size, i0, i1, l);
    return (i0 == src ? 1.f - l : 0.f) + (i1 == src ? l : 0.f);
}

// SHIFT = (2 C) % 8: the block outputs of the coarser level start at position 2 C of the finer block's input, which is
// a multiple of 8 halves only for C = 4; otherwise a group of eight outputs straddles two aligned groups of positions.
template <int SHIFT>
__global__ __launch_bounds__(256) void up2_adjoint_gate_kernel(UpAdjointParams p)
{
    if (const size_t image = p.first_image + blockIdx.y; image > 0)
    {
        const size_t coarse = image * p.Hb * p.Wb;
        p.d_in += image * p.H * p.W * p.cin_fine;
        p.pre += coarse * p.npad;
        p.dpre += coarse * p.npad;
        p.d_feat += coarse * p.c_feat;
    }
    const int half   = p.npad / 2;
    const int C      = p.c_feat;
    // the coarser level's image sits at positions [C, 2C) of the finer block's input: the aligned groups of eight
    // positions g0 .. g0 + ig - 1 (one group up to C = 4 and for C = 8, two for 6 and 16)
    const int g0 = C / 8, ig = (2 * C - 1) / 8 - g0 + 1;
    const int groups = ig + half / 8;  // groups 0 .. ig - 1: the image below; then 8 block outputs each
    const size_t pb  = (size_t)p.Hb * p.Wb;
    const int base8  = (2 * C) & ~7;  // aligned position at or before the first block output
    for (size_t item = (size_t)blockIdx.x * 256 + threadIdx.x; item < pb * groups; item += (size_t)gridDim.x * 256)
    {
        const int q     = (int)(item % groups);
        const size_t bp = item / groups;
        const int Y = (int)(bp / p.Wb), X = (int)(bp - (size_t)Y * p.Wb);
        // the pre-activations first: in flight during the gather
        const int ch0 = 8 * (q - ig);
        half8 f8, m8;
#pragma unroll
        for (int i = 0; i < 8; ++i) f8[i] = m8[i] = _Float16(0.f);
        if (q >= ig)
        {
            const half8 lo = *reinterpret_cast<const half8*>(p.pre + bp * p.npad + 2 * ch0);
            const half8 hi = *reinterpret_cast<const half8*>(p.pre + bp * p.npad + 2 * ch0 + 8);
            f8 = half8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            m8 = half8{lo[4], lo[5], lo[6], lo[7], hi[4], hi[5], hi[6], hi[7]};
        }
        float wy[4], wx[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
        {
            wy[k] = up2_weight(2 * Y - 1 + k, p.H, Y, p.Hb);
            wx[k] = up2_weight(2 * X - 1 + k, p.W, X, p.Wb);
        }
        // the adjoint of the upsampling for the eight positions from `pos` on (a multiple of 8)
        auto gather = [&](int pos, float (&a)[8])
        {
#pragma unroll
            for (int i = 0; i < 8; ++i) a[i] = 0.f;
            if (pos >= p.cin_fine) return;
            // all 16 gathers are issued before the first one is used (a load inside a branch on its weight would be
            // waited for there: 16 memory round trips in a row); pixels outside the image have weight 0 and are read
            // at a clamped position instead
            half8 v[4][4];
            int xoff[4];  // (a row of the finer level stays below 2^31 halves)
#pragma unroll
            for (int kx = 0; kx < 4; ++kx) xoff[kx] = min(max(2 * X - 1 + kx, 0), p.W - 1) * p.cin_fine + pos;
#pragma unroll
            for (int ky = 0; ky < 4; ++ky)
            {
                const int y         = min(max(2 * Y - 1 + ky, 0), p.H - 1);
                const _Float16* row = p.d_in + (size_t)y * p.W * p.cin_fine;
#pragma unroll
                for (int kx = 0; kx < 4; ++kx) v[ky][kx] = *reinterpret_cast<const half8*>(row + xoff[kx]);
            }
#pragma unroll
            for (int ky = 0; ky < 4; ++ky)
            {
#pragma unroll
                for (int kx = 0; kx < 4; ++kx)
                {
                    const float w = wy[ky] * wx[kx];
                    if (w != 0.f)
                    {
                        // (one fused multiply-add that reads the fp16 value, instead of a conversion, a product and a sum)
#pragma unroll
                        for (int i = 0; i < 8; ++i) a[i] = __builtin_fmaf(w, float(v[ky][kx][i]), a[i]);
                    }
                }
            }
        };
        // (one gather for all lanes of a wavefront, whatever their group: lanes of both kinds sit side by side)
        float a[8];
        const int first = q < ig ? 8 * (g0 + q) : base8 + ch0;  // first of the eight positions this item gathers
        gather(first, a);
        if (q < ig)
        {
            // positions [0, C) are the finer level's own image, [C, 2C) this level's
#pragma unroll
            for (int i = 0; i < 8; ++i)
            {
                const int c = first + i - C;  // (a[] only with compile-time indices: else the array goes to scratch memory)
                if (c >= 0 && c < C) p.d_feat[(size_t)c * pb + bp] = a[i] * p.scale_inv;
            }
        }
        else
        {
            // output ch0 + i of this level sits at position 2 C + ch0 + i = base8 + ch0 + SHIFT + i
            if (SHIFT != 0)
            {
                float hi[8];
                gather(base8 + ch0 + 8, hi);
#pragma unroll
                for (int i = 0; i < 8; ++i) a[i] = SHIFT + i < 8 ? a[(SHIFT + i) & 7] : hi[(SHIFT + i) & 7];
            }
            _Float16* dp = p.dpre + bp * p.npad;
            half8 of, om;
#pragma unroll
            for (int i = 0; i < 8; ++i)
            {
                float df, dm;
                gate_backward(ch0 + i < p.cout ? a[i] : 0.f, float(f8[i]), float(m8[i]), df, dm);
                of[i] = _Float16(df);
                om[i] = _Float16(dm);
            }
            *reinterpret_cast<half8*>(dp + 2 * ch0)     = half8{of[0], of[1], of[2], of[3], om[0], om[1], om[2], om[3]};
            *reinterpret_cast<half8*>(dp + 2 * ch0 + 8) = half8{of[4], of[5], of[6], of[7], om[4], om[5], om[6], om[7]};
        }
    }
}

// ---------------------------------------------------------------------------------------------------------
// conv_bwd_data_kernel and up2_adjoint_gate_kernel in one, for blocks with a level below: the gradient of the block's
// input, 2 to 4 bytes written and read again per byte of result, never leaves the chip.
//
// A workgroup walks down a strip of 15 columns of the coarser level, eight rows of the finer one at a time. Per step: the
// data gradient of 8 x 32 pixels (30 columns of its own and one at each side, which the neighbour works out too) goes
// into a ring of ten rows in LDS, rounded to fp16 as it was in memory; four rows of the coarser level then gather their
// 4 x 4 finer pixels from it, in the order of up2_adjoint_gate_kernel, and leave gated. The patch of pre-activation
// gradients is a ring of ten rows too. The eight rows of the next step travel in registers during the products where a CU
// holds one workgroup; where it holds two they go straight to LDS during the gather, which leaves the registers for the
// second workgroup: its products then run beside the first one's gather.
// A wavefront owns 4 x 16 pixels and half of the outputs and keeps the weights of those in registers for the whole strip:
// an operand read from the patch then serves up to three taps, and the sums run in the order of conv_taps_mfma.
//
// Bound at the finest level of a large image by memory, elsewhere by the steps' latencies (two barriers each). As two kernels and as
// one: 1920 x 1080, 32 pre-activations x 32 inputs: 90 + 68 and 125 us; 960 x 540, 64 x 64: 54 + 36 and 82 us; 1245 x 825 and
// the levels below it, 64 x 32: 119 + 60 and 142 us. Of these two workgroups on a CU at 64 x 32, 168 -> 145 (four crops of 512 x 512
// 189 -> 152); neighbouring strips on one XCD, whose L2 then holds the halos that they share, 145 -> 142 and 127 -> 125. The gather as
// matrix products from a ring with the pixels innermost took 358 us where this takes 164.
struct BwdDataUpParams
{
    BwdDataParams fine;   // d_in is not used
    UpAdjointParams up;   // d_in, first_image are not used
    int steps;            // of a workgroup: 8 * steps rows of the finer level, of which it owns 8 * steps - 2
};
// The weights with which rows (columns) 2 v - 1 .. 2 v + 2 of the finer level read row v of the coarser one: up2_weight for
// all four, 0 only for rows outside the image.
__device__ __forceinline__ void up2_adjoint_weights(int v, int fine_size, int coarse_size, float (&w)[4])
{
    w[0] = v > 0 ? 0.25f : 0.f;
    w[1] = v > 0 ? 0.75f : 1.f;
    w[2] = 2 * v + 1 >= fine_size ? 0.f : v + 1 < coarse_size ? 0.75f : 1.f;
    w[3] = v + 1 < coarse_size ? 0.25f : 0.f;
}
constexpr int kStripFine   = kConvTileW - 2;  // columns of the finer level that a strip owns
constexpr int kStripCoarse = kStripFine / 2;
constexpr int kRingRows    = kConvTileH + 2;
constexpr int strip_lds_bytes(int kc, int nn, int ci)
{
    return kConvPatchH * kConvPatchW * (kc + kLdsChanPad) * 2 + kRingRows * kConvTileW * (nn + kLdsChanPad) * 2 + kConvTileH * kConvTileW * ci * 4;
}
// Workgroups of a CU: two where LDS and registers (the weights take 36 (kc / 32) (nn / 32) of a lane) hold them.
// (LDS is given out in 128 pieces of 1280 bytes. From five image channels on, whose share of the image has room for eight, 64
// pre-activations take 82752 bytes, 832 too many.)
constexpr int strip_resident(int kc, int nn, int ci) { return strip_lds_bytes(kc, nn, ci) <= 64 * 1280 && nn == 32 ? 2 : 1; }

alignas(16) __device__ const _Float16 k_zeros[8] = {};  // what lies outside the image

// 16 bytes of each active lane, from its address to LDS: at `to` (the same for all lanes), in the order of the lanes, the places of
// inactive ones left as they are. In flight until wait_for_loads.
__device__ __forceinline__ void load_to_lds16(const void* from, void* to)
{
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)from, (__attribute__((address_space(3))) void*)to, 16, 0, 0);
}
__device__ __forceinline__ void wait_for_loads() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// ALIGNED: 2 C is a multiple of 4, so that a group of four block outputs is one aligned read.
template <int KC, int NN, int CI, bool ALIGNED>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2 * strip_resident(KC, NN, CI)))) void conv_bwd_data_up_kernel(BwdDataUpParams q)
{
    constexpr int THREADS = 512;
    constexpr int ROW = KC + kLdsChanPad, OS = NN + kLdsChanPad;
    constexpr int GROUPS = KC / 8, KB = KC / 32, NBW = NN / 32;
    constexpr int kPixels = kConvTileH * kConvTileW;
    const int H = q.fine.H, W = q.fine.W, C = q.fine.c_feat, Hb = q.up.Hb, Wb = q.up.Wb, npad_b = q.up.npad;
    // Neighbouring strips share halos: they go to one XCD (workgroups are dealt to the eight of them in turn).
    const int all = gridDim.x * gridDim.y * gridDim.z, dealt = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    const int at_block = (dealt & 7) * (all >> 3) + min(dealt & 7, all & 7) + (dealt >> 3);
    const int strip_x = at_block % gridDim.x, strip_yz = at_block / gridDim.x, strip_y = strip_yz % gridDim.y;
    const size_t image  = (size_t)q.fine.first_image + strip_yz / gridDim.y;
    const size_t plane  = (size_t)H * W, plane_b = (size_t)Hb * Wb;
    const _Float16* dpre  = q.fine.dpre + image * plane * KC;
    float* d_feat         = q.fine.d_feat + image * plane * C;
    const _Float16* pre_b = q.up.pre + image * plane_b * npad_b;
    _Float16* dpre_b      = q.up.dpre + image * plane_b * npad_b;
    float* d_feat_b       = q.up.d_feat + image * plane_b * C;
    const float scale_inv = q.fine.scale_inv;

    // (arrays of their own: the loads into the patch are then known to leave what is read from the ring alone)
    __shared__ __align__(16) _Float16 s_patch[kConvPatchH * kConvPatchW * ROW];  // [10 rows][34][ROW]
    __shared__ __align__(16) _Float16 s_ring[kRingRows * kConvTileW * OS];       // [10 rows][32][OS]
    __shared__ float s_img[CI * kPixels];                                        // [CI][8 x 32]
    constexpr bool kAlone = strip_resident(KC, NN, CI) == 1;  // one workgroup on a CU

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lrow = lane & 15, lk = (lane >> 4) * 8;
    const int wr = (wave & 1) * 4, wc = ((wave >> 1) & 1) * 16, wn = (wave >> 2) * NBW;  // this wavefront's rows, columns, output blocks
    const int rows_own = 4 * q.steps - 1;                      // rows of the coarser level
    const int Y0 = strip_y * rows_own, Y1 = min(Y0 + rows_own, Hb);
    const int yf = 2 * Y0 - 1, xf = strip_x * kStripFine - 1;  // the strip's first computed pixel
    const int steps = (2 * (Y1 - Y0) + 2 + kConvTileH - 1) / kConvTileH;

    half8 b[9][KB][NBW];
#pragma unroll
    for (int tap = 0; tap < 9; ++tap)
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int n = 0; n < NBW; ++n)
                b[tap][kb][n] = *reinterpret_cast<const half8*>(q.fine.wt + ((size_t)tap * NN + (wn + n) * 16 + lrow) * KC + kb * 32 + lk);

    // This thread's number, worked out anew where it is called: what follows from it (positions, LDS addresses, weights of
    // the upsampling) would otherwise be kept in registers over the whole strip, beside the convolution's weights.
    auto thread = [&]()
    {
        int t = threadIdx.x;
        asm volatile("" : "+v"(t));
        return t;
    };
    // A row of the patch per wavefront, 16 bytes of a lane at a time; rows are those of the finer level from yf - 1 on.
    // (Unconditional loads, at positions clamped into the image: a load under a condition is waited for where the condition
    // ends.)
    constexpr int kRowItems = kConvPatchW * GROUPS;
    constexpr int kNext     = (kRowItems + 63) / 64;
    uint4 next[kNext];
    auto fetch_row = [&](int row)
    {
        const int tl = thread() & 63;
        const _Float16* src = dpre + (size_t)min(max(yf - 1 + row, 0), H - 1) * W * KC;
#pragma unroll
        for (int j = 0; j < kNext; ++j)
        {
            const int x = min(max(xf - 1 + (tl + 64 * j) / GROUPS, 0), W - 1);
            next[j]     = *reinterpret_cast<const uint4*>(src + x * KC + 8 * (tl % GROUPS));
        }
    };
    auto put_row = [&](int row, int slot)
    {
        const int tl = thread() & 63;
        const int y  = yf - 1 + row;
        _Float16* dst = s_patch + (slot * kConvPatchW + tl / GROUPS) * ROW + 8 * (tl % GROUPS);
#pragma unroll
        for (int j = 0; j < kNext; ++j)
        {
            const int px = (tl + 64 * j) / GROUPS, x = xf - 1 + px;
            const bool in = y >= 0 && y < H && x >= 0 && x < W;
            const uint4 v = make_uint4(in ? next[j].x : 0u, in ? next[j].y : 0u, in ? next[j].z : 0u, in ? next[j].w : 0u);
            if (kRowItems % 64 == 0 || px < kConvPatchW) *reinterpret_cast<uint4*>(dst + j * (64 / GROUPS) * ROW) = v;
        }
    };
    // The same without registers on the way: a wavefront's loads write LDS in the order of its lanes, so the lanes are dealt to
    // whole rows of the patch, and those of the padding sit out.
    auto load_row = [&](int row, int slot)
    {
        constexpr int kWords = GROUPS + kLdsChanPad / 8;  // of 16 bytes, of a pixel
        const int tl = thread() & 63;
        const int y  = yf - 1 + row;
#pragma unroll
        for (int j = 0; j < (kConvPatchW * kWords + 63) / 64; ++j)
        {
            const int i = tl + 64 * j, px = i / kWords, g = i - px * kWords, x = xf - 1 + px;
            const _Float16* src = y >= 0 && y < H && x >= 0 && x < W ? dpre + ((size_t)y * W + x) * KC + 8 * g : k_zeros;
            if (px < kConvPatchW && g < GROUPS) load_to_lds16(src, s_patch + slot * kConvPatchW * ROW + 64 * 8 * j);
        }
    };
    auto first_row = [&](int row)
    {
        if (kAlone)
        {
            fetch_row(row);
            put_row(row, row);
        }
        else
            load_row(row, row);
    };
    if (wave < 2) first_row(wave);
    first_row(wave + 2);

    // the items of the adjoint: a pixel of the coarser level and four positions (see up2_adjoint_gate_kernel), the gated
    // ones before those of the image. (Eight positions to an item are 300 items of a step at 64 pre-activations: five of the eight
    // wavefronts work, and one SIMD does the work of two: 960 x 540, 64 x 64, 88 -> 82 us, 1920 x 1080, 32 x 32, 132 -> 127.)
    const int gates = npad_b / 8;
    const int g0 = C / 4, ig = (2 * C - 1) / 4 - g0 + 1;
    const int gate_items = 4 * kStripCoarse * gates;
    const int items      = gate_items + 4 * kStripCoarse * ig;
    struct Item
    {
        int q, c, cx;
    };
    auto item_of = [&](int item)
    {
        const int past = item - gate_items, per = past < 0 ? gates : ig, i = past < 0 ? item : past;
        const int bp   = i / per;
        return Item{i - bp * per + (past < 0 ? 0 : gates), bp / kStripCoarse, bp % kStripCoarse};
    };
    auto load_pre = [&](const Item& it, int Yk)
    {
        const int Y = min(max(Yk + it.c, 0), Hb - 1), X = min(strip_x * kStripCoarse + it.cx, Wb - 1);
        return *reinterpret_cast<const half8*>(pre_b + ((size_t)Y * Wb + X) * npad_b + 8 * min(it.q, gates - 1));
    };
    const Item first_item = item_of(threadIdx.x);
    const int packed      = first_item.q | first_item.c << 8 | first_item.cx << 16;
    auto mine             = [&]()
    {
        int t = packed;
        asm volatile("" : "+v"(t));
        return Item{t & 255, t >> 8 & 255, t >> 16};
    };
    if (!kAlone) wait_for_loads();
    __syncthreads();

    int slot = 0;  // of the step's first row, in both rings
    for (int k = 0; k < steps; ++k)
    {
        const int yk = yf + kConvTileH * k;  // the step's first row of the finer level
        const int Yk = Y0 - 1 + 4 * k;       // ... and of the coarser one (k = 0: the strip above owns that row)
        const bool more = k + 1 < steps;
        // rows 2 .. 9 of the next step, a row per wavefront, into the slots of rows 0 .. 7 of this one: in flight during the
        // products, where no other workgroup hides the latency, else during the adjoint
        const int next_row = kConvTileH * (k + 1) + 2 + wave, next_slot = slot + wave < kConvPatchH ? slot + wave : slot + wave - kConvPatchH;
        if (kAlone && more) fetch_row(next_row);
        half8 pre;  // four features, four masks
        float old[kPixels * CI / THREADS];
        auto load_rest = [&]()
        {
            pre = load_pre(mine(), Yk);
            const int tid_load = thread();
#pragma unroll
            for (int j = 0; j < kPixels * CI / THREADS; ++j)
            {
                const int v = tid_load + THREADS * j, px = v % kPixels;
                const int y = min(max(yk + px / kConvTileW, 0), H - 1), x = min(max(xf + px % kConvTileW, 0), W - 1);
                old[j] = d_feat[min(v / kPixels, C - 1) * plane + (size_t)y * W + x];
            }
        };
        // (before the products where there are registers for it)
        constexpr bool kEarly = kAlone && KC * NN <= 64 * 32;
        if (kEarly) load_rest();
        floatx4 acc[4][NBW];
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int n = 0; n < NBW; ++n) acc[r][n] = floatx4{0.f, 0.f, 0.f, 0.f};
        // step t: column dx = t % 3 of patch row pr = t / 3; its operands are requested two steps ahead (and no further:
        // the registers would not do)
        constexpr int kAhead = kAlone || KC * NN <= 32 * 32 ? 2 : 1;
        half8 a3[kAhead + 1][KB];
        auto operands = [&](int t)
        {
            const int pr  = t / 3, dx = t - 3 * pr;
            const int at  = slot + wr + pr < kConvPatchH ? slot + wr + pr : slot + wr + pr - kConvPatchH;
            const _Float16* src = s_patch + (at * kConvPatchW + wc + lrow + dx) * ROW + lk;
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) a3[t % (kAhead + 1)][kb] = *reinterpret_cast<const half8*>(src + kb * 32);
        };
#pragma unroll
        for (int t = 0; t < kAhead; ++t) operands(t);
#pragma unroll
        for (int t = 0; t < 18; ++t)
        {
            const int pr = t / 3, dx = t - 3 * pr;
            if (t + kAhead < 18) operands(t + kAhead);
#pragma unroll
            for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                for (int dy = 0; dy < 3; ++dy)
                    if (pr - dy >= 0 && pr - dy < 4)
#pragma unroll
                        for (int n = 0; n < NBW; ++n)
                            acc[pr - dy][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[dy * 3 + dx][kb][n], a3[t % (kAhead + 1)][kb], acc[pr - dy][n], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (!kEarly)
        {
            __builtin_amdgcn_sched_barrier(0);  // (not before the products: their registers are all taken)
            load_rest();
        }
        // a lane: outputs 16 n + 4 (lane / 16) .. + 3 of the pixel in column lane % 16
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            const int at = slot + wr + r < kRingRows ? slot + wr + r : slot + wr + r - kRingRows;
            const int y = yk + wr + r, x = xf + wc + lrow;
            const bool in = y >= 0 && y < H && x >= 0 && x < W;
#pragma unroll
            for (int n = 0; n < NBW; ++n)
            {
                const int c0 = (wn + n) * 16 + (lane >> 4) * 4;
                if (!in) acc[r][n] = floatx4{0.f, 0.f, 0.f, 0.f};
                *reinterpret_cast<half4*>(s_ring + (at * kConvTileW + wc + lrow) * OS + c0) =
                    half4{_Float16(acc[r][n][0]), _Float16(acc[r][n][1]), _Float16(acc[r][n][2]), _Float16(acc[r][n][3])};
                if (n == 0 && c0 < CI)
                {
#pragma unroll
                    for (int i = 0; i < 4; ++i) s_img[(c0 + i) * kPixels + (wr + r) * kConvTileW + wc + lrow] = acc[r][0][i];
                }
            }
        }
        __syncthreads();  // the step's rows are in the ring; nobody reads the patch any more
        if (more)
        {
            if (kAlone)
                put_row(next_row, next_slot);
            else
                load_row(next_row, next_slot);
        }

        // the finer level's own image
        const int tid_store = thread();
#pragma unroll
        for (int j = 0; j < kPixels * CI / THREADS; ++j)
        {
            const int v = tid_store + THREADS * j, px = v % kPixels, c = v / kPixels;
            const int y = yk + px / kConvTileW, col = px % kConvTileW, x = xf + col;
            if (c < C && y >= 2 * Y0 && y < min(2 * Y1, H) && col >= 1 && col <= kStripFine && x < W)
                d_feat[c * plane + (size_t)y * W + x] = old[j] + s_img[v] * scale_inv;
        }

        for (int item = threadIdx.x; item < items; item += THREADS)
        {
            const Item it = item < THREADS ? mine() : item_of(item);
            const int Y = Yk + it.c, X = strip_x * kStripCoarse + it.cx;
            if (Y < Y0 || Y >= Y1 || X >= Wb) continue;
            if (item >= THREADS && it.q < gates) pre = load_pre(it, Yk);
            const int pos = it.q < gates ? 2 * C + 4 * it.q : 4 * (g0 + it.q - gates);  // first of the four positions
            float wy[4], wx[4], a[4];
            up2_adjoint_weights(Y, H, Hb, wy);
            up2_adjoint_weights(X, W, Wb, wx);
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = 0.f;
            if (pos < NN)  // (a row ends with eight unused halves: the last group may reach into them, past the block's outputs)
            {
#pragma unroll
                for (int ky = 0; ky < 4; ++ky)
                {
                    // rows 2 c - 2 + ky of the step, those before it from the step before
                    int at = slot + 8 + 2 * it.c + ky;
                    at -= at >= 2 * kRingRows ? 2 * kRingRows : at >= kRingRows ? kRingRows : 0;
                    const _Float16* src = s_ring + (at * kConvTileW + 2 * it.cx) * OS + pos;
                    if (!kAlone) __builtin_amdgcn_sched_barrier(0);  // one row's reads at a time: more would take the weights' registers
#pragma unroll
                    for (int kx = 0; kx < 4; ++kx)
                    {
                        half4 v;
                        if (ALIGNED)
                            v = *reinterpret_cast<const half4*>(src + kx * OS);
                        else
                        {
                            // (2 C is even: words of four bytes)
                            const unsigned* w2 = reinterpret_cast<const unsigned*>(src + kx * OS);
                            v = __builtin_bit_cast(half4, make_uint2(w2[0], w2[1]));
                        }
                        const float w = wy[ky] * wx[kx];  // (0 for pixels outside the image only: the ring holds zeros there)
#pragma unroll
                        for (int i = 0; i < 4; ++i) a[i] = __builtin_fmaf(w, float(v[i]), a[i]);
                    }
                }
            }
            const size_t bp = (size_t)Y * Wb + X;
            if (it.q >= gates)
            {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                {
                    const int c = pos + i - C;
                    if (c >= 0 && c < C) d_feat_b[(size_t)c * plane_b + bp] = a[i] * scale_inv;
                }
            }
            else
            {
                half8 out;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                {
                    float df, dm;
                    gate_backward(4 * it.q + i < q.up.cout ? a[i] : 0.f, float(pre[i]), float(pre[4 + i]), df, dm);
                    out[i]     = _Float16(df);
                    out[4 + i] = _Float16(dm);
                }
                *reinterpret_cast<half8*>(dpre_b + bp * npad_b + 8 * it.q) = out;
            }
        }
        if (!kAlone) wait_for_loads();
        slot = slot + kConvTileH < kRingRows ? slot + kConvTileH : slot + kConvTileH - kRingRows;
        __syncthreads();  // the next step's patch is in place; nobody reads the ring any more
    }
}

// ---------------------------------------------------------------------------------------------------------
struct BiasGradParams
{
    size_t pixels;
    int npad, cout;
    float scale_inv;
    const _Float16* dpre;  // [pixels][npad]
    float* d_bias_f;       // [cout], accumulated (zeroed by the caller)
    float* d_bias_m;
};

constexpr int kBiasChunk = 1024;
__global__ __launch_bounds__(256) void bias_grad_kernel(const BiasGradParams p)
{
    __shared__ float s_sum[128];
    if (threadIdx.x < 128) s_sum[threadIdx.x] = 0.f;
    __syncthreads();
    const int groups = p.npad / 8;
    const int lanes  = 256 / groups;  // pixels in flight per block
    const int g = threadIdx.x % groups, sub = threadIdx.x / groups;
    if (sub < lanes)
    {
        float a[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) a[i] = 0.f;
        const size_t p0 = (size_t)blockIdx.x * kBiasChunk, p1 = std::min(p.pixels, p0 + kBiasChunk);
        for (size_t pix = p0 + sub; pix < p1; pix += lanes)
        {
            const half8 v = *reinterpret_cast<const half8*>(p.dpre + pix * p.npad + 8 * g);
#pragma unroll
            for (int i = 0; i < 8; ++i) a[i] += float(v[i]);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) atomicAdd(&s_sum[8 * g + i], a[i]);
    }
    __syncthreads();
    if ((int)threadIdx.x < p.npad)
    {
        const int n = threadIdx.x, o = preact_channel(n);
        if (o < p.cout)
        {
            float* dst = preact_is_mask(n) ? p.d_bias_m : p.d_bias_f;
            if (dst) atomicAdd(dst + o, s_sum[n] * p.scale_inv);
        }
    }
}

// ---------------------------------------------------------------------------------------------------------
struct BwdWeightParams
{
    int H, W, Hb, Wb;
    int c_feat, below_stride;
    int tiles_x, tiles;  // tiles of one image
    int batch;           // images, one after the other in every array
    const float* feat;
    const _Float16* below;  // rows of the level below, [Hb][Wb][below_stride]
    int npad;               // pre-activations of a pixel, of which a workgroup takes NPAD
    const _Float16* dpre;   // [H][W][npad]
    int groups;            // workgroups of each share of NPAD pre-activations
    float* part;           // [groups][9][npad][CIN]
    // bias gradients = sums of dpre over the pixels, taken from the transposed tile while it is in LDS
    float* bias_part;      // [groups][npad]
};
// The levels of a launch, one after the other in its workgroups: level, share, group.
struct BwdWeightTable
{
    BwdWeightParams lv[TRIPS_UNET_MAX_LEVELS];
    int first[TRIPS_UNET_MAX_LEVELS];  // first workgroup of every level
    int n;
};

// Pixel-major tiles and the transposing LDS read. Both operands of the weight-gradient GEMM are needed with eight
// consecutive pixels per lane, while the tiles are assembled (and arrive from memory) with the channels of a pixel side
// by side. ds_read_b64_tr_b16 closes the gap: the 16 lanes of a group read a 4 x 16 block of halves row by row (lane
// i: row i / 4, columns 4 (i % 4) .. + 3) and each receives one column (lane n: rows 0 .. 3 of column n). Two such
// reads give a lane the eight pixels of its channel; the tiles stay as the forward kernel builds them, written with
// 16-byte stores (written transposed, 2 bytes at a time, the staging took most of the kernel's time).
typedef short short4v __attribute__((ext_vector_type(4)));
// rows `pix` .. `pix + 7` of column `col0 + lane % 16` of a tile [pixel][stride halves]; `col0` a multiple of 16
__device__ __forceinline__ half8 lds_read_pixels_of_channel(const _Float16* tile, int stride, int pix, int col0)
{
    const int i = threadIdx.x & 15;
    const _Float16* src = tile + (size_t)(pix + (i >> 2)) * stride + col0 + (i & 3) * 4;
    using lds_ptr = __attribute__((address_space(3))) short4v*;
    const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)src);
    const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(src + 4 * stride));
    union
    {
        short s[8];
        half8 h;
    } u;
#pragma unroll
    for (int k = 0; k < 4; ++k)
    {
        u.s[k]     = lo[k];
        u.s[4 + k] = hi[k];
    }
    return u.h;
}

// The same for the three horizontal taps at once: pixels `pix + dx` .. `pix + dx + 7`, dx = 0, 1, 2, of column
// `col0 + lane % 16`, from three reads of four pixels (ten of the twelve are used; the last two may lie past the
// tile, inside the workgroup's LDS) instead of six: the window of dx = 2 is a whole register further, the window of
// dx = 1 is stitched together with four funnel shifts.
__device__ __forceinline__ void lds_read_pixel_windows(const _Float16* tile, int stride, int pix, int col0, half8 (&w)[3])
{
    const int i = threadIdx.x & 15;
    const _Float16* src = tile + (size_t)(pix + (i >> 2)) * stride + col0 + (i & 3) * 4;
    using lds_ptr = __attribute__((address_space(3))) short4v*;
    union
    {
        short4v v[3];
        unsigned d[6];
    } in;
    in.v[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)src);
    in.v[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(src + 4 * stride));
    in.v[2] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(src + 8 * stride));
    union
    {
        unsigned d[4];
        half8 h;
    } out;
#pragma unroll
    for (int k = 0; k < 4; ++k) out.d[k] = in.d[k];
    w[0] = out.h;
#pragma unroll
    for (int k = 0; k < 4; ++k) out.d[k] = __builtin_amdgcn_alignbit(in.d[k + 1], in.d[k], 16);
    w[1] = out.h;
#pragma unroll
    for (int k = 0; k < 4; ++k) out.d[k] = in.d[k + 1];
    w[2] = out.h;
}

// Eight upsampled channels (group g of a patch row) into the row, whose positions [0, C) are the level's own image.
// FOUR: C is exactly 4.
template <bool FOUR>
__device__ __forceinline__ void put_upsampled(_Float16* row, int g, int C, half8 v)
{
    _Float16* dst = row + 8 * g;
    if (FOUR ? g > 0 : 8 * g >= C)
        *reinterpret_cast<half8*>(dst) = v;
    else if (FOUR)
        *reinterpret_cast<half4*>(dst + 4) = half4{v[4], v[5], v[6], v[7]};
    else
    {
        // (the words of the image are there already)
        const uint4 have = *reinterpret_cast<const uint4*>(dst), up = __builtin_bit_cast(uint4, v);
        auto word = [C](int k, unsigned a, unsigned b)
        {
            const int n         = (C & 7) - 2 * k;  // halves of the word that are the image's
            const unsigned mask = n >= 2 ? 0xffffffffu : n == 1 ? 0xffffu : 0u;
            return (a & mask) | (b & ~mask);
        };
        *reinterpret_cast<uint4*>(dst) = make_uint4(word(0, have.x, up.x), word(1, have.y, up.y), word(2, have.z, up.z), word(3, have.w, up.w));
    }
}

// CI: image channels the kernel has room for (4, 8 or 16; C <= CI); FOUR: C is exactly 4; RESIDENT: workgroups on a CU (wgrad_resident)
template <int CIN, int NPAD, bool BIAS, int CI, bool FOUR, int RESIDENT>
__global__ __launch_bounds__(kWgradThreads) __attribute__((amdgpu_waves_per_eu(RESIDENT == 2 ? 4 : 1))) void conv_bwd_weight_kernel(const BwdWeightTable tab)
{
    int level = 0;
    while (level + 1 < tab.n && (int)blockIdx.x >= tab.first[level + 1]) ++level;
    const BwdWeightParams p = tab.lv[level];
    const int in_level = (int)blockIdx.x - tab.first[level];
    constexpr int ROW    = CIN + kLdsChanPad;   // halves per pixel of the input patch
    constexpr int DS     = NPAD + kLdsChanPad;  // halves per pixel of the gradient tile
    constexpr int GROUPS = CIN / 8;
    constexpr int NB     = NPAD / 16;
    constexpr int CB     = CIN / 16;
    // The wavefronts split the NPAD x CIN result: CBW ways over the 16-channel input blocks, NBW ways over the
    // 16-channel pre-activation blocks; each keeps all 9 taps of its blocks. Per tile row a wavefront reads its A
    // fragments (pre-activation gradients, the same for every tap) once and one B fragment per tap and input block.
    constexpr int CBW    = CB < 4 ? CB : 4;
    // (More wavefronts than 16 x 16 blocks to deal out: the wavefronts also split the rows of a tile, RW ways; the
    // shares are added up through LDS at the end.)
    constexpr int THREADS = kWgradThreads;
    constexpr int WAVES  = THREADS / 64;
    constexpr int NBW    = wgrad_nbw(CIN, NPAD);
    constexpr int RW     = wgrad_row_split(CIN, NPAD);
    static_assert(CBW == wgrad_cbw(CIN), "work split");
    constexpr int MYCB   = CB / CBW;
    constexpr int MYNB   = NB / NBW;
    constexpr int MYROWS = kConvTileH / RW;
    static_assert(CB % CBW == 0 && NB % NBW == 0 && CBW * NBW * RW == WAVES && kConvTileH % RW == 0, "block split");
    extern __shared__ _Float16 smem[];
    _Float16* s_patch = smem;                                           // [kConvPatchH * kConvPatchW][ROW]
    _Float16* s_below = s_patch + kConvPatchH * kConvPatchW * ROW;      // [kBelowH * kBelowW][ROW]
    _Float16* s_d     = s_below + kBelowH * kBelowW * ROW;              // [kConvTileH * kConvTileW][DS]
    const bool has_below = p.Hb > 0;
    const int C          = FOUR ? 4 : p.c_feat;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lk = (lane >> 4) * 8;

    const int cb0 = (wave % CBW) * MYCB, nb0 = (RW == 1 ? wave / CBW : (wave / CBW) % NBW) * MYNB;
    const int share = RW == 1 ? 0 : wave / (CBW * NBW);
    const int row0  = share * MYROWS;           // this wavefront's rows of a tile
    const int set   = in_level % p.groups;      // the workgroup's set of partial sums
    floatx4 acc[9][MYNB][MYCB];
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int n = 0; n < MYNB; ++n)
#pragma unroll
            for (int c = 0; c < MYCB; ++c) acc[t][n][c] = floatx4{0.f, 0.f, 0.f, 0.f};
    // Bias gradients = sums of the pre-activation gradients over the pixels: one more MFMA per tile row and block with
    // a matrix of ones as the other operand (every column of the result is the row sum), by the wavefronts that own
    // the first input blocks.
    floatx4 bias_acc[MYNB];
#pragma unroll
    for (int n = 0; n < MYNB; ++n) bias_acc[n] = floatx4{0.f, 0.f, 0.f, 0.f};
    half8 ones;
#pragma unroll
    for (int i = 0; i < 8; ++i) ones[i] = _Float16(1.f);

    // ---- stage 1 in two halves: every global load of a tile is issued into registers (a thread's loads are all in
    // flight together), and written to LDS one tile later, so that the loads of tile t + 1 travel while tile t is
    // upsampled and multiplied ----
    constexpr int kFeatItems  = (kConvPatchH * kConvPatchW + THREADS - 1) / THREADS;
    constexpr int kBelowItems = (kBelowH * kBelowW * GROUPS + THREADS - 1) / THREADS;
    constexpr int kDpreGroups = NPAD / 8;  // 16-byte groups of a pixel's gradient row
    constexpr int kDpreItems  = (kConvTileH * kConvTileW * kDpreGroups + THREADS - 1) / THREADS;
    struct TileLoads
    {
        float feat[kFeatItems][CI];
        uint4 below[kBelowItems];
        half8 dpre[kDpreItems];
    };
    const int below_groups = p.below_stride / 8;  // groups of eight that a row of the level below has
    // the images of the batch are walked as one run of tiles: a workgroup keeps its sums from one image to the next
    // (image after image, every image paid for a set of partial sums of its own and for a last round of its own)
    const int n0      = in_level / p.groups * NPAD;  // this workgroup's first pre-activation
    const float* feat = p.feat;
    const _Float16 *below = p.below, *dpre = p.dpre + n0;
    auto of_image = [&](int& tile)
    {
        const int image = p.batch > 1 ? tile / p.tiles : 0;
        tile -= image * p.tiles;
        feat = p.feat + (size_t)image * C * p.H * p.W;
        dpre = p.dpre + (size_t)image * p.H * p.W * p.npad + n0;
        if (has_below) below = p.below + (size_t)image * p.Hb * p.Wb * p.below_stride;
    };
    auto issue_loads = [&](int tile, TileLoads& r)
    {
        of_image(tile);
        const int ty = tile / p.tiles_x, tx = tile - ty * p.tiles_x;
        const int x0 = tx * kConvTileW, y0 = ty * kConvTileH;
        const int by0 = y0 / 2 - 1, bx0 = x0 / 2 - 1;
        const size_t plane = (size_t)p.H * p.W;
#pragma unroll
        for (int k = 0; k < kFeatItems; ++k)
        {
            const int item = threadIdx.x + THREADS * k;
            const int py = item / kConvPatchW, px = item - py * kConvPatchW;
            const int y = y0 + py - 1, x = x0 + px - 1;
            const bool in = item < kConvPatchH * kConvPatchW && y >= 0 && y < p.H && x >= 0 && x < p.W;
#pragma unroll
            for (int c = 0; c < CI; ++c) r.feat[k][c] = (in && c < C) ? feat[c * plane + (size_t)y * p.W + x] : 0.f;
        }
        if (has_below)
        {
#pragma unroll
            for (int k = 0; k < kBelowItems; ++k)
            {
                const int item = threadIdx.x + THREADS * k;
                const int g = item % GROUPS, bp = item / GROUPS;
                const int rr = bp / kBelowW, c0 = bp - rr * kBelowW;
                r.below[k] = make_uint4(0u, 0u, 0u, 0u);
                if (bp < kBelowH * kBelowW && g < below_groups)
                {
                    const int yy = min(max(by0 + rr, 0), p.Hb - 1), xx = min(max(bx0 + c0, 0), p.Wb - 1);
                    r.below[k]   = *reinterpret_cast<const uint4*>(below + ((size_t)yy * p.Wb + xx) * p.below_stride + 8 * g);
                }
            }
        }
#pragma unroll
        for (int k = 0; k < kDpreItems; ++k)
        {
            const int item = threadIdx.x + THREADS * k;
            const int g = item % kDpreGroups, tp = item / kDpreGroups;
            const int y = y0 + tp / kConvTileW, x = x0 + tp % kConvTileW;
#pragma unroll
            for (int i = 0; i < 8; ++i) r.dpre[k][i] = _Float16(0.f);
            if (tp < kConvTileH * kConvTileW && y < p.H && x < p.W)
                r.dpre[k] = *reinterpret_cast<const half8*>(dpre + ((size_t)y * p.W + x) * p.npad + 8 * g);
        }
    };
    // this level's image into channels [0, C) of a patch pixel (the channels [C, 8) follow from the upsampling, or are
    // zero for the start block, whose other channels are cleared once, below)
    auto put_image = [&](int item, const float (&v)[CI])
    {
        _Float16* row = s_patch + (size_t)item * ROW;
        if (FOUR && has_below)
            *reinterpret_cast<half4*>(row) = half4{_Float16(v[0]), _Float16(v[1]), _Float16(v[2]), _Float16(v[3])};
        else if (has_below)
        {
#pragma unroll
            for (int g4 = 0; g4 < CI / 4; ++g4)  // (run-time bounds would put the register array into scratch memory)
            {
                if (4 * g4 + 4 <= C)
                    *reinterpret_cast<half4*>(row + 4 * g4) =
                        half4{_Float16(v[4 * g4]), _Float16(v[4 * g4 + 1]), _Float16(v[4 * g4 + 2]), _Float16(v[4 * g4 + 3])};
                else
                {
#pragma unroll
                    for (int i = 0; i < 3; ++i)
                        if (4 * g4 + i < C) row[4 * g4 + i] = _Float16(v[4 * g4 + i]);
                }
            }
        }
        else
        {
            // start block: the image is the whole input; the first groups of eight written whole (v is zero past C)
#pragma unroll
            for (int g8 = 0; g8 < (CI + 7) / 8; ++g8)
            {
                half8 h;
#pragma unroll
                for (int i = 0; i < 8; ++i) h[i] = 8 * g8 + i < CI ? _Float16(v[8 * g8 + i < CI ? 8 * g8 + i : 0]) : _Float16(0.f);
                *reinterpret_cast<half8*>(row + 8 * g8) = h;
            }
        }
    };
    auto commit_loads = [&](const TileLoads& r)
    {
#pragma unroll
        for (int k = 0; k < kFeatItems; ++k)
        {
            const int item = threadIdx.x + THREADS * k;
            if (item < kConvPatchH * kConvPatchW) put_image(item, r.feat[k]);
        }
        if (has_below)
        {
#pragma unroll
            for (int k = 0; k < kBelowItems; ++k)
            {
                const int item = threadIdx.x + THREADS * k;
                if (item < kBelowH * kBelowW * GROUPS) *reinterpret_cast<uint4*>(s_below + (item / GROUPS) * ROW + 8 * (item % GROUPS)) = r.below[k];
            }
        }
#pragma unroll
        for (int k = 0; k < kDpreItems; ++k)
        {
            const int item = threadIdx.x + THREADS * k;
            if (item < kConvTileH * kConvTileW * kDpreGroups)
                *reinterpret_cast<half8*>(s_d + (size_t)(item / kDpreGroups) * DS + 8 * (item % kDpreGroups)) = r.dpre[k];
        }
    };

    // start block: the channels beyond the image's groups of eight of a patch pixel are never written and stay zero
    constexpr int kImageGroups = (CI + 7) / 8;
    if (!has_below)
        for (int i = threadIdx.x; i < kConvPatchH * kConvPatchW * (GROUPS - kImageGroups); i += THREADS)
        {
            half8 z;
#pragma unroll
            for (int k = 0; k < 8; ++k) z[k] = _Float16(0.f);
            *reinterpret_cast<half8*>(s_patch + (size_t)(i / (GROUPS - kImageGroups)) * ROW + 8 * (kImageGroups + i % (GROUPS - kImageGroups))) = z;
        }

    TileLoads cur;
    const int tiles = p.tiles * p.batch, groups = p.groups;
    if (set < tiles) issue_loads(set, cur);
    for (int tile0 = set; tile0 < tiles; tile0 += groups)
    {
        int tile = tile0;
        of_image(tile);
        const int ty = tile / p.tiles_x, tx = tile - ty * p.tiles_x;
        const int x0 = tx * kConvTileW, y0 = ty * kConvTileH;
        __syncthreads();  // the previous tile's operands have been consumed (and the zero fill is done)
        commit_loads(cur);
        if (tile0 + groups < tiles) issue_loads(tile0 + groups, cur);  // travels during stage 2 and the taps
        if (has_below)
        {
            __syncthreads();
            // ---- stage 2: bilinear 2x upsampling from the below patch into channels [C, CIN) of the patch, exactly as the
            // forward kernel does it: 2 x 2 pixels between four neighbours at a time ----
            const bool interior = x0 > 0 && y0 > 0 && x0 + kConvTileW < p.W && y0 + kConvTileH < p.H;
            constexpr int kQuadsX = kConvPatchW / 2, kQuads = kQuadsX * (kConvPatchH / 2);
            for (int item = threadIdx.x; item < kQuads * GROUPS; item += THREADS)
            {
                const int g = item % GROUPS, quad = item / GROUPS;
                if (8 * g + 8 <= C) continue;
                const int j = quad / kQuadsX, i = quad - j * kQuadsX;
                const _Float16* src = s_below + (j * kBelowW + i) * ROW + 8 * g;
                half8 v[4];
                upsample_quad(*reinterpret_cast<const half8*>(src), *reinterpret_cast<const half8*>(src + ROW),
                              *reinterpret_cast<const half8*>(src + kBelowW * ROW), *reinterpret_cast<const half8*>(src + (kBelowW + 1) * ROW),
                              y0 + j == 0, x0 + i == 0, v);
#pragma unroll
                for (int n = 0; n < 4; ++n)
                {
                    const int py = 2 * j + (n >> 1), px = 2 * i + (n & 1);
                    if (!interior && !((unsigned)(y0 + py - 1) < (unsigned)p.H && (unsigned)(x0 + px - 1) < (unsigned)p.W)) v[n] = half8{};
                    put_upsampled<FOUR>(s_patch + (py * kConvPatchW + px) * ROW, g, C, v[n]);
                }
            }
        }
        __syncthreads();
        // ---- dW[tap][n][c] += sum over the tile's pixels of dpre[pixel][n] * x[pixel + tap][c] ----
#pragma unroll
        for (int r = row0; r < row0 + MYROWS; ++r)
        {
            half8 a[MYNB];
#pragma unroll
            for (int n = 0; n < MYNB; ++n)
            {
                a[n] = lds_read_pixels_of_channel(s_d, DS, r * kConvTileW + lk, (nb0 + n) * 16);
                if (BIAS && cb0 == 0) bias_acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[n], ones, bias_acc[n], 0, 0, 0);
            }
#pragma unroll
            for (int dy = 0; dy < 3; ++dy)
            {
#pragma unroll
                for (int c = 0; c < MYCB; ++c)
                {
                    half8 b[3];
                    lds_read_pixel_windows(s_patch, ROW, (r + dy) * kConvPatchW + lk, (cb0 + c) * 16, b);
#pragma unroll
                    for (int dx = 0; dx < 3; ++dx)
#pragma unroll
                        for (int n = 0; n < MYNB; ++n)
                            acc[3 * dy + dx][n][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[dx], a[n], acc[3 * dy + dx][n][c], 0, 0, 0);
                }
            }
        }
    }

    if (RW > 1)
    {
        // the row shares of a workgroup add their sums up through LDS (the tiles are consumed), so that the workgroup
        // writes one set: share s > 0 leaves its registers there, share 0 adds them
        static_assert(RW <= 2, "row shares");
        __syncthreads();
        floatx4* s_sum = reinterpret_cast<floatx4*>(smem);  // [wavefront of the share][tap and bias][block][lane]
        constexpr int PER_WAVE = (9 * MYNB * MYCB + MYNB) * 64;
        floatx4* mine = s_sum + (size_t)(wave % (CBW * NBW)) * PER_WAVE + lane;
        if (share > 0)
        {
#pragma unroll
            for (int t = 0; t < 9; ++t)
#pragma unroll
                for (int n = 0; n < MYNB; ++n)
#pragma unroll
                    for (int c = 0; c < MYCB; ++c) mine[((t * MYNB + n) * MYCB + c) * 64] = acc[t][n][c];
#pragma unroll
            for (int n = 0; n < MYNB; ++n) mine[(9 * MYNB * MYCB + n) * 64] = bias_acc[n];
        }
        __syncthreads();
        if (share > 0) return;
#pragma unroll
        for (int t = 0; t < 9; ++t)
#pragma unroll
            for (int n = 0; n < MYNB; ++n)
#pragma unroll
                for (int c = 0; c < MYCB; ++c) acc[t][n][c] += mine[((t * MYNB + n) * MYCB + c) * 64];
#pragma unroll
        for (int n = 0; n < MYNB; ++n) bias_acc[n] += mine[(9 * MYNB * MYCB + n) * 64];
    }
    if (BIAS && cb0 == 0 && (lane & 15) == 0)
    {
        // column 0 of the row sums: this lane holds rows (lane / 16) * 4 .. + 3 of every block
        float* dst = p.bias_part + (size_t)set * p.npad + n0;
#pragma unroll
        for (int n = 0; n < MYNB; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i) dst[(nb0 + n) * 16 + (lane >> 4) * 4 + i] = bias_acc[n][i];
    }
    float* part = p.part + ((size_t)set * 9 * p.npad + n0) * CIN;
    const int lrow = lane & 15;
    // (the input channels are the rows of the MFMA result: a lane holds four neighbouring ones of output lrow)
#pragma unroll
    for (int tap = 0; tap < 9; ++tap)
#pragma unroll
        for (int n = 0; n < MYNB; ++n)
#pragma unroll
            for (int c = 0; c < MYCB; ++c)
                *reinterpret_cast<float4*>(part + ((size_t)tap * p.npad + (nb0 + n) * 16 + lrow) * CIN + (cb0 + c) * 16 + (lane >> 4) * 4) =
                    make_float4(acc[tap][n][c][0], acc[tap][n][c][1], acc[tap][n][c][2], acc[tap][n][c][3]);
}

// Sum of the partial weight gradients of all workgroups (and images), in two steps so that many loads are in
// flight and every load is a full line: slice y of kReduceSlices sums its share of the partials element by element
// (consecutive threads = consecutive elements), then the slices are summed into the reference's [Cout][Cin][3][3].
// All levels in one launch each (the level is blockIdx.z): a launch per level and step costs more than the sums.
constexpr int kReduceSlices = 16;
struct ReduceLevel
{
    const float* part;  // [groups][total]
    float* sliced;      // [kReduceSlices][total]
    int groups, total;
    int cout, cin_real, cin_pad, npad;
    float *d_wf, *d_wm;
    const float* bias_part;  // [groups][npad] or nullptr
    float *d_bf, *d_bm;
};
struct ReduceTable
{
    ReduceLevel lv[TRIPS_UNET_MAX_LEVELS];
    float scale_inv;
};
__global__ __launch_bounds__(256) void reduce_weight_grad_slices_kernel(const ReduceTable t)
{
    const ReduceLevel& l = t.lv[blockIdx.z];
    const float* __restrict__ part = l.part;
    float* __restrict__ sliced     = l.sliced;
    const int groups = l.groups, total = l.total;
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    const int per = (groups + kReduceSlices - 1) / kReduceSlices;
    const int g0 = blockIdx.y * per, g1 = min(groups, g0 + per);
    float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
    int g = g0;
    for (; g + 4 <= g1; g += 4)
    {
        s0 += part[(size_t)g * total + i];
        s1 += part[(size_t)(g + 1) * total + i];
        s2 += part[(size_t)(g + 2) * total + i];
        s3 += part[(size_t)(g + 3) * total + i];
    }
    for (; g < g1; ++g) s0 += part[(size_t)g * total + i];
    sliced[(size_t)blockIdx.y * total + i] = (s0 + s1) + (s2 + s3);
}

// ... and, in the workgroups behind those of the weights, the bias gradients from the per-workgroup sums
__global__ __launch_bounds__(256) void reduce_weight_grad_kernel(const ReduceTable t)
{
    const ReduceLevel& l = t.lv[blockIdx.z];
    const float* __restrict__ sliced = l.sliced;
    const int cout = l.cout, cin_real = l.cin_real, cin_pad = l.cin_pad, npad = l.npad;
    const float scale_inv = t.scale_inv;
    float* __restrict__ d_wf = l.d_wf;
    float* __restrict__ d_wm = l.d_wm;
    const int total = 9 * npad * cin_pad;
    const int wblocks = (total + 255) / 256;
    if ((int)blockIdx.x >= wblocks)
    {
        // one workgroup per pre-activation channel
        const int n = blockIdx.x - wblocks;
        if (n >= npad || !l.bias_part) return;
        const int o = preact_channel(n);
        float* dst  = preact_is_mask(n) ? l.d_bm : l.d_bf;
        if (o >= cout || !dst) return;
        const float s = block_column_sum(l.bias_part, l.groups, npad, n);
        if (threadIdx.x == 0) dst[o] = s * scale_inv;
        return;
    }
    const int i     = blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    const int c = i % cin_pad, n = (i / cin_pad) % npad, tap = i / (cin_pad * npad);
    const int o = preact_channel(n);
    if (o >= cout || c >= cin_real) return;
    float* dst = preact_is_mask(n) ? d_wm : d_wf;
    if (!dst) return;
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < kReduceSlices; ++k) s += sliced[(size_t)k * total + i];
    dst[((size_t)o * cin_real + c) * 9 + tap] = s * scale_inv;
}

// ---------------------------------------------------------------------------------------------------------
namespace
{
template <int KC, int NN, int CI>
hipError_t launch_bwd_data(const BwdDataParams& p, int batch, hipStream_t stream)
{
    // the patch and the staged taps of the weights
    const size_t lds_in  = ((size_t)kConvPatchH * kConvPatchW * (KC + kLdsChanPad) + ConvTapStage<KC, NN>::LDS_HALVES) * sizeof(_Float16);
    const size_t lds_out = (size_t)kConvTileH * kConvTileW * ((NN + kLdsChanPad) * sizeof(_Float16) + CI * sizeof(float));
    const size_t lds     = std::max(lds_in, lds_out);
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&conv_bwd_data_kernel<KC, NN, CI>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    for (int b = 0; b < batch; b += kMaxGridImages)
    {
        BwdDataParams q = p;
        q.first_image   = b;
        dim3 grid((p.W + kConvTileW - 1) / kConvTileW, (p.H + kConvTileH - 1) / kConvTileH, std::min(batch - b, kMaxGridImages));
        hipLaunchKernelGGL((conv_bwd_data_kernel<KC, NN, CI>), grid, dim3(kTapThreads), lds, stream, q);
    }
    return hipGetLastError();
}

hipError_t dispatch_bwd_data(const BwdDataParams& p, int batch, int npad, int cin_pad, hipStream_t stream)
{
#define TRIPS_BD(KC_, NN_)                                                                   \
    if (npad == KC_ && cin_pad == NN_)                                                       \
        return p.c_feat <= 4 ? launch_bwd_data<KC_, NN_, 4>(p, batch, stream)                       \
                             : p.c_feat <= 8 ? launch_bwd_data<KC_, NN_, 8>(p, batch, stream) : launch_bwd_data<KC_, NN_, 16>(p, batch, stream);
    // (start blocks have at most 16 inputs; up to 64 pre-activations the others are conv_bwd_data_up_kernel's)
    TRIPS_BD(32, 32) TRIPS_BD(64, 32) TRIPS_BD(96, 32) TRIPS_BD(128, 32) TRIPS_BD(96, 64) TRIPS_BD(128, 64)
#undef TRIPS_BD
    return hipErrorInvalidValue;
}

template <int KC, int NN, int CI, bool ALIGNED>
hipError_t launch_bwd_data_up(const BwdDataUpParams& p, int batch, hipStream_t stream)
{
    static_assert(strip_lds_bytes(KC, NN, CI) <= 160 * 1024, "the rings do not fit");
    const int strips = (p.up.Wb + kStripCoarse - 1) / kStripCoarse;
    for (int b = 0; b < batch; b += kMaxGridImages)
    {
        BwdDataUpParams q      = p;
        q.fine.first_image     = b;
        const int images       = std::min(batch - b, kMaxGridImages);
        // the shortest strips whose workgroups are all resident at once (a step more costs each a row that it shares with
        // the strip above; a second round of workgroups costs a whole strip)
        const long long resident = 256 * strip_resident(KC, NN, CI);
        const int most           = (p.up.Hb + 1 + 3) / 4;  // steps of a strip of the whole height
        auto segments            = [&](int steps) { return (p.up.Hb + 4 * steps - 2) / (4 * steps - 1); };
        q.steps                  = 1;
        while (q.steps < most && (long long)strips * images * segments(q.steps) > resident) ++q.steps;
        hipLaunchKernelGGL((conv_bwd_data_up_kernel<KC, NN, CI, ALIGNED>), dim3(strips, segments(q.steps), images), dim3(512), 0, stream, q);
    }
    return hipGetLastError();
}

hipError_t dispatch_bwd_data_up(const BwdDataUpParams& p, int batch, int npad, int cin_pad, hipStream_t stream)
{
    const bool aligned = p.fine.c_feat % 2 == 0;
#define TRIPS_BDU_CI(KC_, NN_, CI_) \
    return aligned ? launch_bwd_data_up<KC_, NN_, CI_, true>(p, batch, stream) : launch_bwd_data_up<KC_, NN_, CI_, false>(p, batch, stream)
#define TRIPS_BDU(KC_, NN_)                                     \
    if (npad == KC_ && cin_pad == NN_)                          \
    {                                                           \
        if (p.fine.c_feat <= 4) TRIPS_BDU_CI(KC_, NN_, 4);      \
        if (p.fine.c_feat <= 8) TRIPS_BDU_CI(KC_, NN_, 8);      \
        TRIPS_BDU_CI(KC_, NN_, 16);                             \
    }
    TRIPS_BDU(32, 32) TRIPS_BDU(64, 32) TRIPS_BDU(32, 64) TRIPS_BDU(64, 64)
#undef TRIPS_BDU
#undef TRIPS_BDU_CI
    return hipErrorInvalidValue;
}

template <int CIN, int NPAD, bool BIAS, int CI, bool FOUR, int RESIDENT>
hipError_t launch_bwd_weight(const BwdWeightTable& t, int blocks, hipStream_t stream)
{
    const size_t lds = ((size_t)(kConvPatchH * kConvPatchW + kBelowH * kBelowW) * (CIN + kLdsChanPad) +
                        (size_t)kConvTileH * kConvTileW * (NPAD + kLdsChanPad)) *
                       sizeof(_Float16);  // up to 101 KB
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&conv_bwd_weight_kernel<CIN, NPAD, BIAS, CI, FOUR, RESIDENT>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((conv_bwd_weight_kernel<CIN, NPAD, BIAS, CI, FOUR, RESIDENT>), dim3(blocks), dim3(kWgradThreads), lds, stream, t);
    return hipGetLastError();
}

template <int CI, bool FOUR>
hipError_t dispatch_bwd_weight_ci(const BwdWeightTable& t, int blocks, const LevelPlan& lv, bool bias, hipStream_t stream)
{
#define TRIPS_BW(CIN_, NT_, RES_)                                                           \
    if (lv.cin_pad == CIN_ && lv.wgrad_tile == NT_ && lv.wgrad_resident == RES_)            \
        return bias ? launch_bwd_weight<CIN_, NT_, true, CI, FOUR, RES_>(t, blocks, stream) \
                    : launch_bwd_weight<CIN_, NT_, false, CI, FOUR, RES_>(t, blocks, stream);
    TRIPS_BW(32, 32, 2) TRIPS_BW(32, 64, 1) TRIPS_BW(32, 128, 1) TRIPS_BW(64, 32, 1) TRIPS_BW(64, 64, 1)
    if constexpr (CI <= 8) TRIPS_BW(32, 64, 2)
#undef TRIPS_BW
    return hipErrorInvalidValue;
}

// `lv`: any level of the launch (all are the same instance of the kernel)
hipError_t dispatch_bwd_weight(const BwdWeightTable& t, int blocks, const LevelPlan& lv, bool bias, hipStream_t stream)
{
    const int C = t.lv[0].c_feat;
    if (C == 4) return dispatch_bwd_weight_ci<4, true>(t, blocks, lv, bias, stream);
    if (C < 4) return dispatch_bwd_weight_ci<4, false>(t, blocks, lv, bias, stream);
    if (C <= 8) return dispatch_bwd_weight_ci<8, false>(t, blocks, lv, bias, stream);
    return dispatch_bwd_weight_ci<16, false>(t, blocks, lv, bias, stream);
}
}  // namespace
}  // namespace trips

using namespace trips;

extern "C" {

int trips_unet_backward_workspace_size(const TripsUnetDesc* desc, size_t* bytes)
{
    if (int e = check_unet_desc(desc)) return e;
    if (!bytes) return set_error(TRIPS_ERR_INVALID_ARG, "bytes is NULL");
    *bytes = make_plan(*desc).backward_bytes;
    return TRIPS_OK;
}

int trips_unet_backward(TripsCtx* ctx, const TripsUnetDesc* desc, const TripsUnetWeights* weights,
                        const float* const inputs[TRIPS_UNET_MAX_LEVELS], const void* saved, const float* d_output,
                        float grad_scale, const TripsUnetGrads* grads, void* workspace, size_t workspace_bytes,
                        void* stream_)
{
    if (!ctx) return set_error(TRIPS_ERR_INVALID_ARG, "ctx is NULL");
    if (int e = check_unet_desc(desc)) return e;
    if (!weights || !inputs || !saved || !d_output || !grads || !workspace) return set_error(TRIPS_ERR_INVALID_ARG, "NULL argument");
    const TripsUnetDesc& d = *desc;
    const int C = d.num_input_channels, L = d.num_levels;
    if (!(grad_scale > 0.f) || !std::isfinite(grad_scale)) return set_error(TRIPS_ERR_INVALID_ARG, "grad_scale must be positive");
    for (int i = 0; i < L; ++i)
    {
        if (!inputs[i]) return set_error(TRIPS_ERR_INVALID_ARG, "inputs[%d] is NULL", i);
        if (!grads->inputs[i]) return set_error(TRIPS_ERR_INVALID_ARG, "grads->inputs[%d] is NULL", i);
        if (!weights->feature_weight[i] || !weights->mask_weight[i])
            return set_error(TRIPS_ERR_INVALID_ARG, "weights of block %d are NULL", i);
    }
    if (!weights->final_weight) return set_error(TRIPS_ERR_INVALID_ARG, "final weights are NULL");
    if ((reinterpret_cast<uintptr_t>(workspace) & 255) || (reinterpret_cast<uintptr_t>(saved) & 255))
        return set_error(TRIPS_ERR_INVALID_ARG, "workspace / saved must be 256-byte aligned");
    NetPlan np = make_plan(d);
    if (workspace_bytes < np.backward_bytes)
        return set_error(TRIPS_ERR_WORKSPACE_SMALL, "workspace has %zu bytes, %zu needed", workspace_bytes, np.backward_bytes);
    unsigned wanted = 0;  // levels whose weight gradients are asked for
    for (int i = 0; i < L; ++i)
        if (grads->feature_weight[i] || grads->mask_weight[i]) wanted |= 1u << i;
    plan_wgrad(np, L, C, wanted, np.wgrad_off);
    hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
    char* ws           = reinterpret_cast<char*>(workspace);
    const char* sv     = reinterpret_cast<const char*>(saved);
    Profiler* prof     = ctx->prof.enabled ? &ctx->prof : nullptr;
    const float scale_inv = 1.f / grad_scale;
    const int K           = d.num_output_channels;
    const int ci          = C <= 4 ? 4 : C <= 8 ? 8 : 16;  // image channels the kernels are built with room for

    auto rows_ptr = [&](int level)
    {
        const LevelPlan& l = np.lv[level];
        return reinterpret_cast<const _Float16*>(sv + l.saved_rows_off);
    };
    auto pre_ptr = [&](int level)
    {
        const LevelPlan& l = np.lv[level];
        return reinterpret_cast<const _Float16*>(sv + l.saved_pre_off);
    };
    auto dpre_ptr = [&](int level)
    {
        const LevelPlan& l = np.lv[level];
        return reinterpret_cast<_Float16*>(ws + l.dpre_off);
    };
    auto din_ptr = [&](int level)
    {
        const LevelPlan& l = np.lv[level];
        return reinterpret_cast<_Float16*>(ws + l.din_off);
    };
    auto fill = [&](float* p, int n)
    {
        if (p && n > 0) hipLaunchKernelGGL(fill_f32_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, p, 0.f, n);
    };

    {
        ProfScope ps(prof, "unet_bwd_prepare", stream);
        PackTTable pt;
        int most = 0;
        for (int i = 0; i < L; ++i)
        {
            const LevelPlan& lv = np.lv[i];
            pt.lv[i] = PackTLevel{weights->feature_weight[i], weights->mask_weight[i], lv.cout, lv.cin_real, lv.cin_pad, lv.npad,
                                  reinterpret_cast<_Float16*>(ws + lv.wt_off)};
            most     = std::max(most, 9 * lv.npad * lv.cin_pad);
        }
        hipLaunchKernelGGL(pack_conv_weights_T_kernel, dim3((most + 255) / 256, L), dim3(256), 0, stream, pt);
        for (int i = 0; i < L; ++i)
        {
            const LevelPlan& lv = np.lv[i];
            if (!((wanted >> i) & 1u))  // bias_grad_kernel accumulates; otherwise they are written
            {
                fill(grads->feature_bias[i], lv.cout);
                fill(grads->mask_bias[i], lv.cout);
            }
        }
    }
    {
        ProfScope ps(prof, "unet_bwd_final", stream);
        const LevelPlan& lv = np.lv[0];
        const size_t plane  = (size_t)lv.H * lv.W;
        FinalBwdParams p;
        std::memset(&p, 0, sizeof(p));
        p.H = lv.H, p.W = lv.W, p.c_feat = C, p.cact = lv.cout, p.cout = K;
        p.scale    = grad_scale;
        p.feat     = inputs[0];
        p.pre      = pre_ptr(0);
        p.weight   = weights->final_weight;
        p.d_out    = d_output;
        p.d_feat   = grads->inputs[0];
        p.dpre     = dpre_ptr(0);
        p.chunks   = (int)((plane + kFinalPixelsPerBlock - 1) / kFinalPixelsPerBlock);
        p.batch    = d.batch;
        p.part     = reinterpret_cast<float*>(ws + np.final_part_off);
        const bool wgrad = grads->final_weight || grads->final_bias;
        const int chunks = wgrad ? np.final_groups : p.chunks * p.batch;
        switch (lv.npad)
        {
#define TRIPS_FW_CI(NPAD_, CI_)                                                                               \
    if (wgrad)                                                                                                \
        hipLaunchKernelGGL((final_backward_kernel<NPAD_, true, CI_>), dim3(chunks), dim3(256), 0, stream, p); \
    else                                                                                                      \
        hipLaunchKernelGGL((final_backward_kernel<NPAD_, false, CI_>), dim3(chunks), dim3(256), 0, stream, p);
#define TRIPS_FW(NPAD_)              \
    case NPAD_:                      \
        if (ci == 4)                 \
        {                            \
            TRIPS_FW_CI(NPAD_, 4)    \
        }                            \
        else if (ci == 8)            \
        {                            \
            TRIPS_FW_CI(NPAD_, 8)    \
        }                            \
        else                         \
        {                            \
            TRIPS_FW_CI(NPAD_, 16)   \
        }                            \
        break;
            TRIPS_FW(32) TRIPS_FW(64) TRIPS_FW(96) TRIPS_FW(128)
#undef TRIPS_FW
#undef TRIPS_FW_CI
            default: return set_error(TRIPS_ERR_UNSUPPORTED, "%d pre-activations", lv.npad);
        }
        if (grads->final_weight || grads->final_bias)
        {
            hipLaunchKernelGGL(final_reduce_kernel, dim3(K * (C + lv.cout) + K), dim3(256), 0, stream,
                               reinterpret_cast<const float*>(ws + np.final_part_off), np.final_groups, ci + lv.npad / 2, ci, C,
                               lv.cout, K, grads->final_weight, grads->final_bias);
        }
    }
    static const char* const kDataNames[TRIPS_UNET_MAX_LEVELS]   = {"unet_bwd_data_l0", "unet_bwd_data_l1", "unet_bwd_data_l2", "unet_bwd_data_l3",
                                                                    "unet_bwd_data_l4", "unet_bwd_data_l5", "unet_bwd_data_l6", "unet_bwd_data_l7"};
    static const char* const kWeightNames[TRIPS_UNET_MAX_LEVELS] = {"unet_bwd_weight_l0", "unet_bwd_weight_l1", "unet_bwd_weight_l2", "unet_bwd_weight_l3",
                                                                    "unet_bwd_weight_l4", "unet_bwd_weight_l5", "unet_bwd_weight_l6", "unet_bwd_weight_l7"};
    for (int i = 0; i < L; ++i)
    {
        const LevelPlan& lv = np.lv[i];
        const bool below    = i < L - 1;
        {
            ProfScope ps(prof, kDataNames[i], stream);
            BwdDataParams dp;
            dp.H = lv.H, dp.W = lv.W, dp.c_feat = C;
            dp.scale_inv = scale_inv;
            dp.dpre      = dpre_ptr(i);
            dp.wt        = reinterpret_cast<const _Float16*>(ws + lv.wt_off);
            dp.d_feat    = grads->inputs[i];
            dp.d_in      = below ? din_ptr(i) : nullptr;
            const bool fused = bwd_data_up_fits(lv.npad, lv.cin_pad, below);
            if (!fused)
            {
                hipError_t e = dispatch_bwd_data(dp, d.batch, lv.npad, lv.cin_pad, stream);
                if (e != hipSuccess) return set_error(TRIPS_ERR_HIP, "data gradient launch (level %d): %s", i, hipGetErrorString(e));
            }
            if (below)
            {
                const LevelPlan& lb = np.lv[i + 1];
                UpAdjointParams up;
                up.H = lv.H, up.W = lv.W, up.Hb = lb.H, up.Wb = lb.W;
                up.cin_fine  = lv.cin_pad;
                up.c_feat    = C;
                up.cout      = lb.cout;
                up.npad      = lb.npad;
                up.scale_inv = scale_inv;
                up.d_in      = din_ptr(i);
                up.pre       = pre_ptr(i + 1);
                up.d_feat    = grads->inputs[i + 1];
                up.dpre      = dpre_ptr(i + 1);
                if (fused)
                {
                    BwdDataUpParams du;
                    du.fine      = dp;
                    du.up        = up;
                    hipError_t e = dispatch_bwd_data_up(du, d.batch, lv.npad, lv.cin_pad, stream);
                    if (e != hipSuccess) return set_error(TRIPS_ERR_HIP, "data gradient launch (level %d): %s", i, hipGetErrorString(e));
                }
                else
                {
                    const size_t items = (size_t)lb.H * lb.W * ((2 * C - 1) / 8 - C / 8 + 1 + lb.npad / 16);
                    for (up.first_image = 0; up.first_image < d.batch; up.first_image += kMaxGridImages)
                    {
                        const dim3 blocks((unsigned)std::min<size_t>((items + 255) / 256, 1u << 20), std::min(d.batch - up.first_image, kMaxGridImages));
                        switch ((2 * C) & 7)
                        {
                            case 0: hipLaunchKernelGGL(up2_adjoint_gate_kernel<0>, blocks, dim3(256), 0, stream, up); break;
                            case 2: hipLaunchKernelGGL(up2_adjoint_gate_kernel<2>, blocks, dim3(256), 0, stream, up); break;
                            case 4: hipLaunchKernelGGL(up2_adjoint_gate_kernel<4>, blocks, dim3(256), 0, stream, up); break;
                            default: hipLaunchKernelGGL(up2_adjoint_gate_kernel<6>, blocks, dim3(256), 0, stream, up); break;
                        }
                    }
                }
            }
        }
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return set_error(TRIPS_ERR_HIP, "backward launch (level %d): %s", i, hipGetErrorString(e));
    }
    // The weight gradients need the pre-activation gradients alone: all behind the data gradients, levels that are the same
    // instance of the kernel in one launch, which the profiler names after the finest of them. It sums the pre-activation
    // gradients as well if a bias gradient of any of its levels is asked for.
    unsigned launched = 0;
    for (int i = 0; i < L; ++i)
    {
        const LevelPlan& lv = np.lv[i];
        if (!((wanted >> i) & 1u))
        {
            if (!grads->feature_bias[i] && !grads->mask_bias[i]) continue;
            ProfScope ps(prof, kWeightNames[i], stream);
            BiasGradParams bp;
            bp.pixels    = (size_t)lv.H * lv.W * d.batch;
            bp.npad      = lv.npad;
            bp.cout      = lv.cout;
            bp.scale_inv = scale_inv;
            bp.dpre      = dpre_ptr(i);
            bp.d_bias_f  = grads->feature_bias[i];
            bp.d_bias_m  = grads->mask_bias[i];
            hipLaunchKernelGGL(bias_grad_kernel, dim3((unsigned)((bp.pixels + kBiasChunk - 1) / kBiasChunk)), dim3(256), 0, stream, bp);
            continue;
        }
        if ((launched >> i) & 1u) continue;
        ProfScope ps(prof, kWeightNames[i], stream);
        BwdWeightTable t;
        std::memset(&t, 0, sizeof(t));
        int blocks = 0;
        bool bias  = false;
        for (int k = i; k < L; ++k)
        {
            const LevelPlan& lk = np.lv[k];
            if (!((wanted >> k) & 1u) || !same_wgrad_kernel(lk, lv)) continue;
            launched |= 1u << k;
            bias                = bias || grads->feature_bias[k] || grads->mask_bias[k];
            t.first[t.n]        = blocks;
            BwdWeightParams& wp = t.lv[t.n++];
            wp.H = lk.H, wp.W = lk.W, wp.c_feat = C;
            wp.tiles_x   = (lk.W + kConvTileW - 1) / kConvTileW;
            wp.tiles     = wp.tiles_x * ((lk.H + kConvTileH - 1) / kConvTileH);
            wp.batch     = d.batch;
            wp.feat      = inputs[k];
            wp.npad      = lk.npad;
            wp.groups    = lk.groups;
            wp.dpre      = dpre_ptr(k);
            wp.part      = reinterpret_cast<float*>(ws + lk.part_off);
            wp.bias_part = reinterpret_cast<float*>(ws + lk.bias_part_off);
            if (k < L - 1)
            {
                const LevelPlan& lb = np.lv[k + 1];
                wp.Hb = lb.H, wp.Wb = lb.W, wp.below_stride = lb.row_stride;
                wp.below = rows_ptr(k + 1);
            }
            blocks += lk.groups * (lk.npad / lk.wgrad_tile);
        }
        hipError_t e = dispatch_bwd_weight(t, blocks, lv, bias, stream);
        if (e != hipSuccess) return set_error(TRIPS_ERR_HIP, "weight gradient launch (level %d): %s", i, hipGetErrorString(e));
    }
    // the partial weight and bias gradients of all levels are summed at the end, one launch per step of the sum
    {
        ProfScope ps(prof, "unet_bwd_reduce", stream);
        ReduceTable rt;
        rt.scale_inv = scale_inv;
        int n = 0, most = 0, most_npad = 0;
        for (int i = 0; i < L; ++i)
        {
            const LevelPlan& lv = np.lv[i];
            if (!((wanted >> i) & 1u)) continue;
            ReduceLevel& r = rt.lv[n++];
            r.part      = reinterpret_cast<const float*>(ws + lv.part_off);
            r.sliced    = reinterpret_cast<float*>(ws + lv.sliced_off);
            r.groups    = lv.groups;
            r.total     = 9 * lv.npad * lv.cin_pad;
            r.cout = lv.cout, r.cin_real = lv.cin_real, r.cin_pad = lv.cin_pad, r.npad = lv.npad;
            r.d_wf = grads->feature_weight[i], r.d_wm = grads->mask_weight[i];
            const bool bias = grads->feature_bias[i] || grads->mask_bias[i];
            r.bias_part = bias ? reinterpret_cast<const float*>(ws + lv.bias_part_off) : nullptr;
            r.d_bf = grads->feature_bias[i], r.d_bm = grads->mask_bias[i];
            most      = std::max(most, r.total);
            most_npad = std::max(most_npad, lv.npad);
        }
        if (n > 0)
        {
            hipLaunchKernelGGL(reduce_weight_grad_slices_kernel, dim3((most + 255) / 256, kReduceSlices, n), dim3(256), 0, stream, rt);
            hipLaunchKernelGGL(reduce_weight_grad_kernel, dim3((most + 255) / 256 + most_npad, 1, n), dim3(256), 0, stream, rt);
            hipError_t e = hipGetLastError();
            if (e != hipSuccess) return set_error(TRIPS_ERR_HIP, "gradient sums launch: %s", hipGetErrorString(e));
        }
    }
    return TRIPS_OK;
}

}  // extern "C"
