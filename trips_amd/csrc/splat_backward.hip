// Backward kernels of the splat path for gfx950 (wave64).
//
//   backward_tiles_kernel + backward_points_kernel <- BlendBackwardsBilinearTiled
//                                                     src/lib/rendering/RenderBackward.cu:90-618
//
// The reference walks one pixel list per thread and scatters every entry's gradient with float atomics
// (3 position + 1 size + 1 confidence + C descriptor atomics per retained entry). Scattered atomics run at about
// 2e10 per second on this GPU, and what bounds the kernels of this path is the number of scattered memory requests,
// whatever their size. So the four pixels of a point's footprint meet in LDS, not in memory:
//   1. tiles: a workgroup walks a block of 16 x 16 pixels, one pixel per lane, and owns the 15 x 15 cells whose four
//      pixels lie inside it (a cell = the footprints that start at that pixel); blocks overlap by one row and one
//      column, which the neighbours walk again. A lane recomputes alpha and transmittance of its pixel's retained
//      entries from the per-point record exactly as the forward computed them, forms dL/dalpha (the "all later
//      entries" sum of RenderBackward.cu:284-301 is a running sum from the back of the list) and leaves
//      {dL/dalpha, T alpha} of every entry in LDS, together with the entry's list position under the (cell, place in
//      the cell's list, corner) that the forward noted for it. After a barrier every (point, layer) pair is formed
//      once, by the wavefront of the first of its corner pixels that retained it: the pairs are queued and dealt to
//      the lanes, a lane collects the four corner pixels' entries and writes ONE row per pair: sum over the corners of
//      T alpha dL/dimage and the four dL/dalpha. The rows of a point's first two layers sit at its compact number,
//      further layers in an overflow table.
//   2. points: the (point, layer) pairs of 64 points are dealt out to the lanes; a lane reads its pair's
//      row, evaluates the bilinear weights' Jacobian and the layer factor per corner (PointBlending.h:216-264,
//      RenderBackward.cu:366-438); the point's own lane sums the image-space gradient of all its entries and runs the
//      projection chain ONCE (the chain is linear in the image-space gradient, RenderBackward.cu:385-417), then stores
//      or adds its gradients. Pose / intrinsics partials stay in registers over a grid-stride loop before one
//      block-level reduction; a workgroup leaves a row of sums (the reference keeps them in shared double arrays,
//      :160-187,546-617).
//   3. sums: adds up those rows, and the ones that the first pass's workgroups leave for the background.
// A prologue kernel clears the rows (or, for a view in which few pairs are retained, one flag byte per row) beforehand.
// The per-point gradients are summed in a fixed order and are bit-reproducible from run to run; so are the block sums
// (background, pose, intrinsics) but for the order in which several views, or images of more than kSumRows blocks, add to one.
#include "row16.h"
#include "splat_internal.h"
#include "trips_math.h"

#include <algorithm>
#include <type_traits>

#pragma clang fp contract(off)

namespace trips
{
__device__ __forceinline__ Camera load_camera_bw(const double* pose, const float* intr, const TripsView& v,
                                                 float dist_cutoff)
{
    Camera c;
    c.V  = load_pose(pose);
    c.fx = intr[0];
    c.fy = intr[1];
    c.cx = intr[2];
    c.cy = intr[3];
    c.s  = intr[4];
    c.no_distortion = true;
    for (int i = 0; i < 8; ++i)
    {
        c.dist[i] = intr[5 + i];
        c.no_distortion = c.no_distortion && c.dist[i] == 0.f;
    }
    c.cfx         = v.crop_transform[0];
    c.cfy         = v.crop_transform[1];
    c.ccx         = v.crop_transform[2];
    c.ccy         = v.crop_transform[3];
    c.cs          = v.crop_transform[4];
    c.r00         = v.crop_rotation[0];
    c.r01         = v.crop_rotation[1];
    c.r10         = v.crop_rotation[2];
    c.r11         = v.crop_rotation[3];
    c.centre_x    = float(v.w / 2);
    c.centre_y    = float(v.h / 2);
    c.dist_cutoff = dist_cutoff;
    return c;
}

typedef float vf4 __attribute__((ext_vector_type(4)));
typedef int vi4 __attribute__((ext_vector_type(4)));
typedef unsigned vu4 __attribute__((ext_vector_type(4)));

// largest value of v (0 .. LIMIT) over the wavefront's lanes, as a scalar
template <int LIMIT>
__device__ __forceinline__ int wave_max_small(int v)
{
    int m = 0;
#pragma unroll
    for (int t = 1; t <= LIMIT; ++t)
        if (__ballot(v >= t)) m = t;
    return m;
}

// ---------------------------------------------------------------------------------------------------------
// Pass 1: per block of 16 x 16 cells.
constexpr int kBlockSide   = 16;                       // pixels per side of a workgroup's block: one pixel per lane
constexpr int kBlockCells  = kBlockSide - 1;           // cells per side whose footprints lie inside those pixels
constexpr int kBlockPixels = kBlockSide * kBlockSide;  // 256

// LDS of a block for lists of up to K entries: {dL/dalpha, T alpha} per (list position, pixel); dL/dimage per pixel, four
// channels at a time; per (place in the cell's sorted list, cell) the list positions of that point's entry in its four
// corner pixels (0xFF: none; an entry at list position j has a place of at most j). The pixel or the cell is the fastest
// index everywhere: neighbouring lanes, neighbouring banks.
__host__ __device__ constexpr size_t tiles_lds_bytes(int cpad, int K)
{
    return (size_t)kBlockPixels * K * 8 + (size_t)kBlockPixels * cpad * 4 + (size_t)kBlockCells * kBlockCells * K * 4;
}

// The chunk of the binning kernels that a compact number (below 256 chunks) belongs to: the factor exceeds the quotient's by less
// than 2^-49 of it, the product by less than 2^-40, and no quotient is closer than 2^-23 below a whole number.
__device__ __forceinline__ int chunk_of_point(const BackwardParams& p, int cid) { return (int)((double)cid * p.chunk_per_point); }
// The point's first row in the overflow table, `word` being the second of its point record.
__device__ __forceinline__ int first_overflow_row(const BackwardParams& p, int cid, unsigned word)
{
    return (int)(word >> kLayersBits) + p.chunk_valid[kBinGroups + kRetainedParts + chunk_of_point(p, cid)];
}

template <int C, int kListMax>
__global__ __launch_bounds__(256) void backward_tiles_kernel(const BackwardParams p)
{
    constexpr int CPAD  = (C + 3) & ~3;
    constexpr int RF    = 4 + CPAD;  // floats per blend record
    constexpr int NQ    = CPAD / 4;
    constexpr int PRF   = pair_row_floats(CPAD);
    // list positions whose records are requested together (the LDS of a block bounds the wavefronts per SIMD before the
    // registers do)
    constexpr int BATCH = CPAD <= 4 ? 8 : 4;
    extern __shared__ __align__(16) unsigned char s_mem[];
    float2* const s_ex     = reinterpret_cast<float2*>(s_mem);
    vf4* const s_g         = reinterpret_cast<vf4*>(s_mem + (size_t)kBlockPixels * kListMax * 8);
    unsigned* const s_rank = reinterpret_cast<unsigned*>(s_mem + (size_t)kBlockPixels * kListMax * 8 + (size_t)kBlockPixels * CPAD * 4);
    __shared__ double s_acc[4][CPAD];
    // (point, layer) pairs that wait for a lane of their wavefront: slot = place * 225 + cell, and the point's compact
    // number. The queue is emptied down to fewer than kQueueSlack pairs before a list position adds up to 64.
    constexpr int kQueueSlack = 32, kQueue = kQueueSlack + 64;
    __shared__ unsigned short s_qslot[4][kQueue];
    __shared__ int s_qcid[4][kQueue];

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // Blocks of 16 x 16 pixels that overlap by one row and one column (so that every cell's four pixels lie in one
    // block): block (i, j) of a layer starts at pixel (15 i, 15 j). Runs of eight blocks of a block row share an XCD.
    // The coarsest layer, whose lists are the longest, begins, so that no few blocks are left over at the end; not in views in
    // which few pairs are retained (the forward's plan has the same rule for its reasons). us, finest layer first and coarsest: 6M
    // points in no order 317 and 305, 9M in Morton order 208 and 194, 500k at 700 x 500 72 and 63, four views of tight clusters
    // 308 and 323.
    const bool sparse = *p.mode != 0;  // only flagged rows exist (the same for the whole view)
    long long lblock  = xcd_tile_block(blockIdx.x, 8);
    if (lblock >= p.blocks_off[p.num_layers]) return;
    if (!sparse) lblock = p.blocks_off[p.num_layers] - 1 - lblock;
    int layer = 0;
#pragma unroll
    for (int l = 1; l < TRIPS_MAX_LAYERS; ++l)
        if (l < p.num_layers && lblock >= p.blocks_off[l]) layer = l;
    const int in_layer = (int)lblock - p.blocks_off[layer];
    const int byi = in_layer / p.blocks_x[layer], bxi = in_layer - byi * p.blocks_x[layer];
    const int lw = p.geom.w[layer], lh = p.geom.h[layer];
    const int x0 = bxi * kBlockCells, y0 = byi * kBlockCells;  // the block's first pixel
    const float* const gi = p.grad_image[layer];

    float acc_bg[C];  // a lane sees a few pixels: its own sums stay in single precision, everything across lanes is double
#pragma unroll
    for (int c = 0; c < C; ++c) acc_bg[c] = 0.f;

    // ---- the block's pixels, one per lane, a wavefront taking 8 x 8 of them (the four pixels of a footprint then
    // mostly sit in one wavefront and share their gathers) ----
    {
        const int px = ((wave & 1) << 3) + (lane & 7), py = ((wave >> 1) << 3) + (lane >> 3);
        const int t  = py * kBlockSide + px;
        const int gx = x0 + px, gy = y0 + py;
        const bool inside = gx < lw && gy < lh;
        // (the last row and column are the first of the neighbours' blocks)
        const bool owned   = inside && px < kBlockCells && py < kBlockCells;
        const unsigned pix = inside ? (unsigned)pix_index_mul24(p.geom, layer, gx, gy) : 0u;
        // the pixel's retained count, its list (compact numbers and where each entry came from) and dL/dimage are all
        // requested before the first is looked at; list positions past the retained ones hold anything and are not used
        int word = 0;
        int id[kListMax];
        const vi4* mine = nullptr;  // the pixel's list: positions 4q .. 4q + 3 at mine[64 q]
        unsigned tagw[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int j = 0; j < kListMax; ++j) id[j] = 0;
        if (inside)
        {
            word = p.retained[pix];
            mine = reinterpret_cast<const vi4*>(p.lists + list_word(pix, 0, p.list_depth));
            {
                const vi4 v = __builtin_nontemporal_load(mine);
                id[0] = v.x, id[1] = v.y, id[2] = v.z, id[3] = v.w;
            }
            const vu4 v = __builtin_nontemporal_load(reinterpret_cast<const vu4*>(p.tags) + pix);
            tagw[0] = v.x, tagw[1] = v.y, tagw[2] = v.z, tagw[3] = v.w;
        }

        float g[C];
#pragma unroll
        for (int c = 0; c < C; ++c) g[c] = 0.f;
        if (inside)
        {
            // offsets inside one view's image stay far below 2^32 (the pyramid has at most kMaxBins tiles)
            if (p.layout == TRIPS_LAYOUT_CHW)
            {
                const size_t plane = (size_t)lw * lh;
                const float* o     = gi + ((size_t)p.view_index * C) * plane;
                const unsigned at  = __umul24((unsigned)gy, (unsigned)lw) + (unsigned)gx;
#pragma unroll
                for (int c = 0; c < C; ++c) g[c] = (o + c * plane)[at];
            }
            else
            {
                const float* o    = gi + ((size_t)p.view_index * lh * lw) * C;
                const unsigned at = (__umul24((unsigned)gy, (unsigned)lw) + (unsigned)gx) * C;
#pragma unroll
                for (int c = 0; c < C; ++c) g[c] = o[at + c];
            }
        }
        // no entry yet under any (cell, place): cleared while the loads above travel
        for (int i = threadIdx.x; i < kBlockCells * kBlockCells * kListMax / 4; i += 256)
            reinterpret_cast<uint4*>(s_rank)[i] = make_uint4(~0u, ~0u, ~0u, ~0u);
        __syncthreads();
        const int m    = word & kRetainedMask;
        const int mmax = wave_max_small<kListMax>(m);
        // (two thirds of the pixels of a typical view retain at most four entries: the rest of a list only where needed)
#pragma unroll
        for (int q = 1; q < kListMax / 4; ++q)
        {
            if (4 * q < mmax && 4 * q < m)
            {
                const vi4 v = __builtin_nontemporal_load(mine + (q << 6));
                id[4 * q] = v.x, id[4 * q + 1] = v.y, id[4 * q + 2] = v.z, id[4 * q + 3] = v.w;
            }
        }
#pragma unroll
        for (int q = 0; q < NQ; ++q)
        {
            vf4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (4 * q + i < C) v[i] = g[4 * q + i];
            s_g[q * kBlockPixels + t] = v;
        }
        float sbg = 0.f;
#pragma unroll
        for (int c = 0; c < C; ++c) sbg += p.background[c] * g[c];

        // front to back: alpha, transmittance (the forward's chain), descriptor . dL/dimage
        float A[kListMax], Tr[kListMax], S[kListMax];
#pragma unroll
        for (int j = 0; j < kListMax; ++j) A[j] = 0.f, Tr[j] = 0.f, S[j] = 0.f;
        float T = 1.f;
        float4 r0[BATCH], rd[BATCH][NQ];
        auto position = [&](auto jc)
        {
            constexpr int j = decltype(jc)::value;
            constexpr int b = j % BATCH;
            const bool has  = j < m;
            float a         = 0.f;
            if (has) a = entry_alpha(r0[b], layer, p.num_layers, gx, gy);
            float s = 0.f;
#pragma unroll
            for (int c = 0; c < C; ++c)
            {
                const float4 t4 = rd[b][c / 4];
                const float d   = (c & 3) == 0 ? t4.x : (c & 3) == 1 ? t4.y : (c & 3) == 2 ? t4.z : t4.w;
                s += d * g[c];
            }
            A[j]  = a;
            Tr[j] = T;
            S[j]  = has ? s : 0.f;
            T     = T * (1.f - a);
        };
        auto batch = [&](auto first)
        {
            constexpr int j0 = decltype(first)::value;
#pragma unroll
            for (int b = 0; b < BATCH; ++b)
            {
                if (j0 + b < mmax && j0 + b < m)
                {
                    const float4* rec = reinterpret_cast<const float4*>(p.rec + (size_t)(unsigned)id[j0 + b] * RF);
                    r0[b]             = rec[0];
#pragma unroll
                    for (int q = 0; q < NQ; ++q) rd[b][q] = rec[1 + q];
                }
            }
            if (j0 + 0 < mmax) position(std::integral_constant<int, j0 + 0>{});
            if (j0 + 1 < mmax) position(std::integral_constant<int, j0 + 1>{});
            if (j0 + 2 < mmax) position(std::integral_constant<int, j0 + 2>{});
            if (j0 + 3 < mmax) position(std::integral_constant<int, j0 + 3>{});
            if constexpr (BATCH > 4)
            {
                if (j0 + 4 < mmax) position(std::integral_constant<int, j0 + 4>{});
                if (j0 + 5 < mmax) position(std::integral_constant<int, j0 + 5>{});
                if (j0 + 6 < mmax) position(std::integral_constant<int, j0 + 6>{});
                if (j0 + 7 < mmax) position(std::integral_constant<int, j0 + 7>{});
            }
        };
        if (mmax > 0) batch(std::integral_constant<int, 0>{});
        if constexpr (BATCH == 4)
        {
            if (mmax > 4) batch(std::integral_constant<int, 4>{});
            if constexpr (kListMax > 8)
            {
                if (mmax > 8) batch(std::integral_constant<int, 8>{});
                if (mmax > 12) batch(std::integral_constant<int, 12>{});
            }
        }
        else if constexpr (kListMax > 8)
        {
            if (mmax > 8) batch(std::integral_constant<int, 8>{});
        }

        // transmittance after the m retained entries decides whether the background is reached
        // (RenderBackward.cu:205-210,302-308); T is that product (1 for an empty list)
        const float T_after   = T;
        const bool bg_reached = inside && (T_after >= 0.001f);
        if (bg_reached && owned)
        {
#pragma unroll
            for (int c = 0; c < C; ++c) acc_bg[c] += T_after * g[c];
        }
        const float bg_term = bg_reached ? T_after * sbg : 0.f;

        // back to front: dL/dalpha_j = T_j s_j - (sum_{i>j} T_i alpha_i s_i + background term) / (1 - alpha_j + 1e-9)
        // (RenderBackward.cu:262-302); the entry goes to LDS under its pixel and under its (cell, place)
        float later = 0.f;  // sum over the entries behind this one
#pragma unroll
        for (int j = kListMax - 1; j >= 0; --j)
        {
            if (j < mmax)
            {
                const float ta = Tr[j] * A[j];
                if (j < m)
                {
                    const float dem        = 1.f / (1.f - A[j] + 1e-9f);
                    const float grad_alpha = Tr[j] * S[j] - (later + bg_term) * dem;
                    s_ex[j * kBlockPixels + t] = make_float2(grad_alpha, ta);
                    const unsigned tag     = (tagw[j / 4] >> (8 * (j & 3))) & 0xFFu;
                    const int w = (int)(tag >> 4) & 3, place = (int)(tag & 15u);
                    // the cell the entry came from: (x-1, y-1), (x, y-1), (x-1, y), (x, y) for w = 0..3; this pixel is corner
                    // 3 - w of that footprint
                    const int cxl = px - 1 + (w & 1), cyl = py - 1 + (w >> 1);
                    if ((unsigned)cxl < (unsigned)kBlockCells && (unsigned)cyl < (unsigned)kBlockCells)
                    {
                        const int slot = place * (kBlockCells * kBlockCells) + cyl * kBlockCells + cxl;
                        reinterpret_cast<unsigned char*>(s_rank)[slot * 4 + (3 - w)] = (unsigned char)j;
                    }
                }
                later += ta * S[j];
            }
        }
        __syncthreads();

        // ---- a row per (point, layer) pair that some pixel retained. Each pair is formed once: by the wavefront of
        // the first of its four corner pixels that retained it, whose lane still holds the point's compact number.
        // The pairs are unevenly spread over the pixels, so a wavefront queues {slot, compact number} of the pairs its
        // pixels are first for, position by position, and whenever enough wait, each lane forms one row. ----
        constexpr int kCells           = kBlockCells * kBlockCells;
        unsigned short* const qslot    = s_qslot[wave];
        int* const qcid                = s_qcid[wave];
        const bool inline_row          = layer < kInlineLayers;  // (the same for the whole block)
        const unsigned long long below = (1ull << lane) - 1ull;
        int waiting = 0;  // pairs in the queue (the same in every lane)
        // forms the rows of the first `n` pairs of the queue (n <= 64)
        auto form_rows = [&](int n)
        {
            if (lane < n)
            {
                const int slot  = qslot[lane];
                const int cid   = qcid[lane];
                int row_of      = cid;
                const int place = slot / kCells, c2 = slot - place * kCells;
                const int cyl = c2 / kBlockCells, cxl = c2 - cyl * kBlockCells;
                const unsigned w4 = s_rank[slot];
                // past the second layer: the number of the point's first row in the overflow table
                if (!inline_row) row_of = first_overflow_row(p, cid, __float_as_uint(p.prec[(size_t)(unsigned)cid * kPointRecordFloats + 1]));
                // the four corners' entries, all requested before the first is looked at (of a corner that did not retain the
                // point, an entry of its list that is not used)
                float2 e[4];
                vf4 g4[4][NQ];
#pragma unroll
                for (int corner = 0; corner < 4; ++corner)
                {
                    const int tp = (cyl + (corner >> 1)) * kBlockSide + cxl + (corner & 1);
                    e[corner]    = s_ex[(int)((w4 >> (8 * corner)) & (unsigned)(kListMax - 1)) * kBlockPixels + tp];
#pragma unroll
                    for (int q = 0; q < NQ; ++q) g4[corner][q] = s_g[q * kBlockPixels + tp];
                }
                float tex[CPAD], ga[4];
#pragma unroll
                for (int c = 0; c < CPAD; ++c) tex[c] = 0.f;
#pragma unroll
                for (int corner = 0; corner < 4; ++corner)
                {
                    const bool is = ((w4 >> (8 * corner)) & 0xFFu) != 0xFFu;
                    ga[corner]    = is ? e[corner].x : 0.f;
#pragma unroll
                    for (int c = 0; c < C; ++c)
                    {
                        const float more = tex[c] + e[corner].y * g4[corner][c / 4][c & 3];
                        tex[c]           = is ? more : tex[c];
                    }
                }
                const long long over = (long long)row_of + (layer - kInlineLayers);
                if (inline_row || over < p.over_capacity)
                {
                    vf4* row = reinterpret_cast<vf4*>(inline_row ? p.rows_inline + ((size_t)(unsigned)row_of * kInlineLayers + layer) * PRF
                                                                 : p.rows_over + (size_t)over * PRF);
#pragma unroll
                    for (int q = 0; q < NQ; ++q) row[q] = vf4{tex[4 * q], tex[4 * q + 1], tex[4 * q + 2], tex[4 * q + 3]};
                    row[NQ] = vf4{ga[0], ga[1], ga[2], ga[3]};
                    if (sparse) p.flags[(size_t)(unsigned)cid * TRIPS_MAX_LAYERS + layer] = 1;
                }
            }
        };
        // the first 64 pairs leave the queue, the others move up
        auto pop64 = [&]()
        {
            form_rows(min(waiting, 64));
            unsigned short mslot = 0;
            int mcid             = 0;
            if (64 + lane < waiting) mslot = qslot[64 + lane], mcid = qcid[64 + lane];
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            if (64 + lane < waiting) qslot[lane] = mslot, qcid[lane] = mcid;
            waiting = max(waiting - 64, 0);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        };
        // four list positions at a time (a loop over all sixteen, unrolled, would repeat the row code sixteen times;
        // one that is not unrolled would index the registers that hold the list)
#pragma unroll 1
        for (int q4 = 0; q4 < kListMax / 4; ++q4)
        {
            if (4 * q4 >= mmax) break;
            unsigned tw = tagw[0];
            int idq[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) idq[i] = id[i];
#pragma unroll
            for (int k = 1; k < kListMax / 4; ++k)
            {
                tw = q4 == k ? tagw[k] : tw;
#pragma unroll
                for (int i = 0; i < 4; ++i) idq[i] = q4 == k ? id[4 * k + i] : idq[i];
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                const int j = 4 * q4 + i;
                if (j >= mmax) break;
                bool own = false;
                int slot = 0;
                if (j < m)
                {
                    const unsigned tag = (tw >> (8 * i)) & 0xFFu;
                    const int w = (int)(tag >> 4) & 3, place = (int)(tag & 15u);
                    const int cxl = px - 1 + (w & 1), cyl = py - 1 + (w >> 1);
                    if ((unsigned)cxl < (unsigned)kBlockCells && (unsigned)cyl < (unsigned)kBlockCells)
                    {
                        slot              = place * kCells + cyl * kBlockCells + cxl;
                        const unsigned w4 = s_rank[slot];
                        // this pixel is corner 3 - w of the footprint: it forms the row if no corner before it retained the point
                        const int first = (w4 & 0xFFu) != 0xFFu ? 0 : ((w4 >> 8) & 0xFFu) != 0xFFu ? 1 : ((w4 >> 16) & 0xFFu) != 0xFFu ? 2 : 3;
                        own             = first == 3 - w;
                    }
                }
                const unsigned long long mask = __ballot(own);
                if (!mask) continue;
                if (own)
                {
                    const int at = waiting + (int)__popcll(mask & below);
                    qslot[at]    = (unsigned short)slot;
                    qcid[at]     = idq[i];
                }
                waiting += (int)__popcll(mask);
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                if (waiting >= kQueueSlack) pop64();
            }
        }
        while (waiting > 0) pop64();
    }

    // the block's row of the background's sums (backward_sums_kernel adds them up)
#pragma unroll
    for (int q = 0; q < NQ; ++q)
    {
        auto of = [&](int i) { return 4 * q + i < C ? (double)acc_bg[min(4 * q + i, C - 1)] : 0.0; };
        const double v = wave_sum4(of(0), of(1), of(2), of(3));
        if ((lane & 15) == 0) s_acc[wave][4 * q + (lane >> 4)] = v;
    }
    __syncthreads();
    if (threadIdx.x < CPAD)
    {
        const int i = threadIdx.x;
        p.background_sums[(size_t)lblock * CPAD + i] = (float)(s_acc[0][i] + s_acc[1][i] + s_acc[2][i] + s_acc[3][i]);
    }
}

// ---------------------------------------------------------------------------------------------------------
// Pass 2: per point. A wavefront walks 64 consecutive points at a time. Where only some of them have work (the flagged ones of
// a view with few retained pairs, or the valid ones where gradients are added to what earlier views left) they are
// queued, and worked off 64 together: all lanes work however many points a view culls or hides. What the others get in
// overwrite mode is zero, stored at once. With rows for all pairs and overwriting, the 64 points of a step are worked off
// as they are: through the queue their outputs would leave in parts of lines (6M points: 238 us instead of 175).
// The work of a point is one item per layer it was written to; points differ in the layers they reach, so the items of the
// 64 points are dealt out to the lanes through LDS, one item per lane and round: the items of a round are consecutive
// (point, layer) pairs, whose rows are consecutive in memory. An item's sums return through LDS and each point adds its
// items up in layer order. The camera's rotation is the same for all points and sits in scalar registers.
// What bounds it: vector instructions and memory together. 6M points in no order (0.85 GB) 202 -> 175 us, 9M in Morton order
// 200 -> 184, four crops of 2M 211 -> 157, four views of 4M clustered points, of which a view retains one in five, 602 ->
// 299, against a step per 64 points whatever they hold, with the camera in LDS and the weights, their derivatives and the
// layer factor worked out corner by corner. (Products and sums stay uncontracted and in this order: gradients of points that
// many pixels pull apart are small differences of large terms.)
constexpr int kItemFloats(int cpad) { return 4 + cpad; }  // {confidence, ip.x, ip.y, size} sums, then the descriptor's

struct PointPassCamera
{
    Camera cam;
    float R[9];
};

__device__ __forceinline__ float uniform(float v) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v))); }

// the camera of a view and its rotation matrix, in scalar registers
__device__ __forceinline__ PointPassCamera load_uniform_camera(const BackwardParams& p)
{
    PointPassCamera u;
    const Camera c = load_camera_bw(p.pose, p.intrinsics, p.view, p.dist_cutoff);
    rotation_matrix(c.V, u.R);
    for (int i = 0; i < 9; ++i) u.R[i] = uniform(u.R[i]);
    u.cam   = c;
    u.cam.V = Pose{uniform(c.V.qx), uniform(c.V.qy), uniform(c.V.qz), uniform(c.V.qw), uniform(c.V.tx), uniform(c.V.ty), uniform(c.V.tz)};
    return u;
}

template <int C>
__global__ __launch_bounds__(256, 4) void backward_points_kernel(const BackwardParams p)
{
    constexpr int CPAD = (C + 3) & ~3;
    constexpr int RF   = 4 + CPAD;  // floats per blend record
    constexpr int NQ   = CPAD / 4;
    constexpr int PRF  = pair_row_floats(CPAD);
    constexpr int NACC = 6 + 5 + 8;  // pose, K, distortion
    constexpr int NIT  = kItemFloats(CPAD);
    const int lane     = threadIdx.x & 63;
    const int wave     = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool want_pose = p.d_pose != nullptr;
    const bool want_intr = p.d_intrinsics != nullptr;
    const bool want_size = p.d_point_size != nullptr;
    const bool identity  = p.header->not_identity == 0;  // index[pid] == pid for every point
    const bool overwrite = p.overwrite != 0;             // outputs are written, not added to
    const bool sparse    = *p.mode != 0;  // only the flagged rows exist
    const bool direct    = overwrite && !sparse;  // every point's outputs are stored: as whole lines, without the queue
    // In overwrite mode every point stores all its outputs, zeros where it has no gradient. (Descriptor columns other than
    // the points' own, and all of them when the index is not the identity, were cleared by the prologue kernel.)

    constexpr int kQueue = 128;  // fewer than 64 that wait and up to 64 more
    __shared__ int s_pid[4][kQueue], s_cid[4][kQueue];
    __shared__ unsigned char s_mask[4][kQueue];  // the layers whose rows the point's items read
    // what an item needs of its point {ip.x, ip.y, size field, confidence, size_px, softplus' * d size_px / d size,
    // number of its first overflow row, compact number}
    __shared__ float s_point[4][64][9];
    __shared__ unsigned short s_item[4][64 * TRIPS_MAX_LAYERS];  // lane of the point | layer << 8
    __shared__ __align__(16) float s_sums[4][64][NIT];           // sums of the items of one round
    const PointPassCamera u = load_uniform_camera(p);
    auto wave_fence         = []()
    {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };

    // a thread sees a handful of points: its own sums stay in single precision, everything across threads is double
    float acc[NACC];
#pragma unroll
    for (int i = 0; i < NACC; ++i) acc[i] = 0.f;

    auto store_gradients = [&](int pid, bool any, float conf_grad, float size_grad, const float (&tex_grad)[C], const float (&g_point)[3])
    {
        if (identity && overwrite)
        {
#pragma unroll
            for (int c = 0; c < C; ++c) p.d_texture[(size_t)c * p.num_texels + pid] = tex_grad[c];
            p.d_confidence[pid] = conf_grad;
        }
        else if (identity)
        {
#pragma unroll
            for (int c = 0; c < C; ++c) p.d_texture[(size_t)c * p.num_texels + pid] += tex_grad[c];
            p.d_confidence[pid] += conf_grad;
        }
        else if (any)
        {
            const int tex = p.index[pid];  // (a column outside the table: the point was culled)
#pragma unroll
            for (int c = 0; c < C; ++c) unsafeAtomicAdd(p.d_texture + (size_t)c * p.num_texels + tex, tex_grad[c]);
            unsafeAtomicAdd(p.d_confidence + tex, conf_grad);
        }
        if (want_size)
        {
            if (overwrite)
                p.d_point_size[pid] = size_grad;
            else
                p.d_point_size[pid] += size_grad;
        }
        if (p.d_position)
        {
            float4* dp = reinterpret_cast<float4*>(p.d_position) + pid;
            float4 v   = overwrite ? make_float4(0.f, 0.f, 0.f, 0.f) : *dp;
            v.x += g_point[0];
            v.y += g_point[1];
            v.z += g_point[2];
            *dp = v;
        }
    };

    // one point per lane: number, compact number, the layers whose rows its items read (none: the point gets zeros)
    auto work_off = [&](int pid, int cid, unsigned mask)
    {
        const bool has = mask != 0u;
        int first      = 0;
        // {depth, layers written and first overflow row, softplus'(raw size), size_px}; {ip.x, ip.y, size field, confidence}
        // of the blend record
        float4 tail = make_float4(0.f, 0.f, 0.f, 0.f), r0 = tail, pos = tail;
        if (has)
        {
            tail = reinterpret_cast<const float4*>(p.prec)[cid];
            r0   = *reinterpret_cast<const float4*>(p.rec + (size_t)(unsigned)cid * RF);
            pos  = p.position[pid];
            if (p.displacement)
            {
                const float* dsp = p.displacement + (size_t)pid * 3;
                pos.x += dsp[0];
                pos.y += dsp[1];
                pos.z += dsp[2];
            }
        }
        // (rows past the capacity of the overflow table do not exist: the forward reported the overflow; a point of one or two
        // layers has none, and its number there is not looked at)
        if (mask >> kInlineLayers)
        {
            first               = first_overflow_row(p, cid, __float_as_uint(tail.y));
            const long long fit = p.over_capacity - first;
            if (fit < TRIPS_MAX_LAYERS - kInlineLayers) mask &= (1u << (kInlineLayers + (int)max(0ll, fit))) - 1u;
        }
        // ---- the point's items: the layers it was written to ----
        const int my_items = (int)__popc(mask);
        int first_item     = my_items;  // inclusive prefix over the wavefront, then made exclusive
        for (int o = 1; o < 64; o <<= 1)
        {
            const int t = __shfl_up(first_item, o);
            if (lane >= o) first_item += t;
        }
        const int num_items = __builtin_amdgcn_readlane(first_item, 63);  // <= 64 * 8
        first_item -= my_items;
        {
            int at = first_item;
            for (unsigned m = mask; m; m &= m - 1u) s_item[wave][at++] = (unsigned short)(lane | ((__ffs((int)m) - 1) << 8));
        }
        // the point in view space, exactly as the projection kernel computed it
        float view[3];
        transform_point(u.cam.V, pos.x, pos.y, pos.z, view);
        {
            const float J_softmax_proj = u.cam.fx * u.cam.cfx / fmaxf(view[2], 0.f);
            float* sp = s_point[wave][lane];
            sp[0] = r0.x, sp[1] = r0.y, sp[2] = r0.z, sp[3] = r0.w, sp[4] = tail.w, sp[5] = tail.z * J_softmax_proj;
            sp[6] = __int_as_float(first);
            sp[7] = __int_as_float(cid);
        }
        wave_fence();

        float conf_grad = 0.f, size_grad = 0.f, d0 = 0.f, d1 = 0.f;
        float tex_grad[C];
#pragma unroll
        for (int c = 0; c < C; ++c) tex_grad[c] = 0.f;
        for (int round = 0; round < num_items; round += 64)
        {
            if (round + lane < num_items)
            {
                // one layer of one point: its row holds the descriptor sums, then dL/dalpha of the four corners (zeros
                // where no pixel retained the point)
                const unsigned item = s_item[wave][round + lane];
                const int layer     = (int)(item >> 8);
                const float* sp     = s_point[wave][item & 63u];
                const float ipx = sp[0], ipy = sp[1], size_field = sp[2], conf = sp[3], size_px = sp[4], size_chain = sp[5];
                const vf4* row = reinterpret_cast<const vf4*>(
                    layer < kInlineLayers ? p.rows_inline + ((size_t)(unsigned)__float_as_int(sp[7]) * kInlineLayers + layer) * PRF
                                          : p.rows_over + ((size_t)__float_as_int(sp[6]) + (layer - kInlineLayers)) * PRF);
                vf4 tq[NQ];
#pragma unroll
                for (int q = 0; q < NQ; ++q) tq[q] = __builtin_nontemporal_load(row + q);
                const vf4 ga = __builtin_nontemporal_load(row + NQ);
                const float mfac = __uint_as_float((uint32_t)(127 - layer) << 23);
                const float ux = ipx * mfac, uy = ipy * mfac;
                const float sx = ux - floorf(ux), sy = uy - floorf(uy);
                float lfac = 1.f, J_lf = 0.f;
                if (want_size) lfac = layer_factor_encoded_grad(size_field, size_px, layer, p.num_layers, &J_lf);
                // blend_fac_index / compute_blending_fac (PointBlending.h:216-264) at the corners x = floor(ux) + 0, 1: weight 1 -
                // s and s, derivative -1 and 1; of a coordinate that is a whole number the reference takes s and 1 for both
                const bool ex = sx == 0.f, ey = sy == 0.f;
                const float wx0 = ex ? 0.f : 1.f - sx, wy0 = ey ? 0.f : 1.f - sy;
                const float gl = conf * lfac, gs = size_chain * J_lf;
                float i_conf = 0.f, i_d0 = 0.f, i_d1 = 0.f, i_size = 0.f;
#pragma unroll
                for (int corner = 0; corner < 4; ++corner)
                {
                    const bool x1 = (corner & 1) != 0, y1 = corner >= 2;
                    const float wx = x1 ? sx : wx0, wy = y1 ? sy : wy0, blend = wx * wy;
                    i_conf += blend * lfac * ga[corner];
                    const float gbs = gl * ga[corner];
                    i_d0 += (x1 ? wy : ex ? wy : -wy) * gbs;
                    i_d1 += (y1 ? wx : ey ? wx : -wx) * gbs;
                    if (want_size) i_size += blend * conf * (gs * ga[corner]);
                }
                float4* out = reinterpret_cast<float4*>(s_sums[wave][lane]);
                out[0]      = make_float4(i_conf, i_d0, i_d1, i_size);
#pragma unroll
                for (int q = 0; q < NQ; ++q) out[1 + q] = make_float4(tq[q].x, tq[q].y, tq[q].z, tq[q].w);
            }
            wave_fence();
            // the point's items of this round, in layer order
            const int j_end = min(first_item + my_items, round + 64);
            for (int j = max(first_item, round); j < j_end; ++j)
            {
                const float4* in = reinterpret_cast<const float4*>(s_sums[wave][j - round]);
                const float4 a   = in[0];
                conf_grad += a.x;
                d0 += a.y;
                d1 += a.z;
                size_grad += a.w;
#pragma unroll
                for (int q = 0; q < NQ; ++q)
                {
                    const float4 t = in[1 + q];
                    if (4 * q < C) tex_grad[4 * q] += t.x;
                    if (4 * q + 1 < C) tex_grad[4 * q + 1] += t.y;
                    if (4 * q + 2 < C) tex_grad[4 * q + 2] += t.z;
                    if (4 * q + 3 < C) tex_grad[4 * q + 3] += t.w;
                }
            }
            wave_fence();
        }
        // some gradient reached the point
        bool any = conf_grad != 0.f || d0 != 0.f || d1 != 0.f || size_grad != 0.f;
#pragma unroll
        for (int c = 0; c < C; ++c) any = any || tex_grad[c] != 0.f;
        if (pid < 0 || (!any && !overwrite)) return;

        float g_point[3] = {0.f, 0.f, 0.f}, g_pose[6], g_k[5], g_dis[8];
        if (any)
        {
            project_backward(u.cam, u.R, view[0], view[1], view[2], d0, d1, g_point, g_pose, g_k, g_dis, want_intr);
            if (want_pose)
            {
#pragma unroll
                for (int k = 0; k < 6; ++k) acc[k] += g_pose[k];
            }
            if (want_intr)
            {
#pragma unroll
                for (int k = 0; k < 5; ++k) acc[6 + k] += g_k[k];
#pragma unroll
                for (int k = 0; k < 8; ++k) acc[11 + k] += g_dis[k];
            }
        }
        store_gradients(pid, any, conf_grad, size_grad, tex_grad, g_point);
    };

    const int stride = (int)gridDim.x * 256;
    // The compact numbers of kGroup steps' points are requested two groups ahead, and the layers that they were written to (or the
    // flags of their rows) one group ahead, and looked at when the group begins. (The rest of a point's record follows in work_off, in a
    // request of its own: where every point is worked off as it comes, 634 MB read instead of 609 at 6M points in no order.) A step
    // at a time, its layers worked out where they were requested, every step waited for that: 9M points 186 -> 172 us, 6M in no order
    // 169 -> 166, four views of clusters 271 -> 256, crops 109 -> 106; four steps 164, 170, 258 and 110. One step and two of the present
    // form: four channels, 6M in no order 169 and 166, clusters 260 and 254, 9M without dropout 249 and 253, four views of 500k at
    // 512 x 512 99.6 and 101; three, 3M in a ball 115 both ways; six, 1M 59.4 and 61; eight, 300k 22.1 and 23.0; sixteen, 1.4M 96 and
    // 97.6. (A step without any work, in the form without the queue, passed over at once: 9M 170, but 6M 170 and clusters 264.)
    auto cid_at    = [&](long long pid) { return pid < p.num_points ? p.cid_of[pid] : -1; };
    auto request   = [&](int cid) -> uint2
    {
        if (cid < 0) return make_uint2(0u, 0u);
        if (sparse) return *reinterpret_cast<const uint2*>(p.flags + (size_t)(unsigned)cid * TRIPS_MAX_LAYERS);
        return make_uint2(__float_as_uint(p.prec[(size_t)(unsigned)cid * kPointRecordFloats + 1]), 0u);
    };
    auto layers_of = [&](uint2 got) -> unsigned
    {
        if (!sparse) return (1u << (got.x & kLayersMask)) - 1u;
        unsigned flagged = 0;  // (a byte of 0 or 1 per layer)
#pragma unroll
        for (int l = 0; l < 4; ++l)
        {
            flagged |= ((got.x >> (8 * l)) & 1u) << l;
            flagged |= ((got.y >> (8 * l)) & 1u) << (4 + l);
        }
        return flagged;
    };
    constexpr int kGroup = C <= 4 ? 2 : 1;
    const long long pid0 = (long long)blockIdx.x * 256 + (int)threadIdx.x;
    int cids[kGroup], cids_next[kGroup];
    unsigned masks = 0;  // a byte per step
#pragma unroll
    for (int k = 0; k < kGroup; ++k)
    {
        cids[k]      = cid_at(pid0 + (long long)k * stride);
        cids_next[k] = cid_at(pid0 + (long long)(kGroup + k) * stride);
    }
#pragma unroll
    for (int k = 0; k < kGroup; ++k) masks |= layers_of(request(cids[k])) << (8 * k);
    int waiting = 0;  // queued points (the same in every lane)
    // (the last steps, past the end, empty the queue)
    for (int base = blockIdx.x * 256; base < p.num_points || waiting > 0;)
    {
        int cids_later[kGroup];
        uint2 requested[kGroup];
#pragma unroll
        for (int k = 0; k < kGroup; ++k)
        {
            requested[k]  = request(cids_next[k]);
            cids_later[k] = cid_at((long long)base + (int)threadIdx.x + (long long)(2 * kGroup + k) * stride);
        }
#pragma unroll 1
        for (int k = 0; k < kGroup; ++k)
        {
            const int at = base;
            if (at >= p.num_points && waiting == 0) break;
            base          = min(at, p.num_points) + stride;
            int pid       = at + (int)threadIdx.x;
            int cid       = cids[0];
            unsigned mask = (masks >> (8 * k)) & 0xFFu;
#pragma unroll
            for (int j = 1; j < kGroup; ++j) cid = k == j ? cids[j] : cid;
            if (!direct)
            {
                const bool queued = mask != 0u;
                const unsigned long long qm = __ballot(queued);
                if (queued)
                {
                    const int to     = waiting + (int)__popcll(qm & ((1ull << lane) - 1ull));
                    s_pid[wave][to]  = pid;
                    s_cid[wave][to]  = cid;
                    s_mask[wave][to] = (unsigned char)mask;
                }
                waiting += (int)__popcll(qm);
                if (overwrite && !queued && pid < p.num_points)
                {
                    const float none[C] = {}, nowhere[3] = {0.f, 0.f, 0.f};
                    store_gradients(pid, false, 0.f, 0.f, none, nowhere);
                }
                if (waiting < 64 && at < p.num_points) continue;
                wave_fence();
                // 64 leave the queue, the others move up
                const int next  = 64 + lane;
                const bool here = lane < waiting, moves = next < waiting;
                pid = here ? s_pid[wave][lane] : p.num_points, cid = s_cid[wave][lane], mask = here ? s_mask[wave][lane] : 0u;
                int mpid = 0, mcid = 0;
                unsigned char mmask = 0;
                if (moves) mpid = s_pid[wave][next], mcid = s_cid[wave][next], mmask = s_mask[wave][next];
                wave_fence();
                if (moves) s_pid[wave][lane] = mpid, s_cid[wave][lane] = mcid, s_mask[wave][lane] = mmask;
                waiting = max(waiting - 64, 0);
            }
            work_off(pid < p.num_points ? pid : -1, cid, mask);
        }
        masks = 0;
#pragma unroll
        for (int k = 0; k < kGroup; ++k)
        {
            masks |= layers_of(requested[k]) << (8 * k);
            cids[k] = cids_next[k], cids_next[k] = cids_later[k];
        }
    }

    // the workgroup's row of the pose's and the intrinsics' sums (backward_sums_kernel adds them up)
    if (!want_pose && !want_intr) return;
    __shared__ double s_acc[4][kCameraSums];
#pragma unroll
    for (int q = 0; q < kCameraSums / 4; ++q)
    {
        auto of = [&](int i) { return 4 * q + i < NACC ? (double)acc[min(4 * q + i, NACC - 1)] : 0.0; };
        const double v = wave_sum4(of(0), of(1), of(2), of(3));
        if ((lane & 15) == 0) s_acc[wave][4 * q + (lane >> 4)] = v;
    }
    __syncthreads();
    if (threadIdx.x < kCameraSums)
    {
        const int i = threadIdx.x;
        p.camera_sums[(size_t)blockIdx.x * kCameraSums + i] = s_acc[0][i] + s_acc[1][i] + s_acc[2][i] + s_acc[3][i];
    }
}

// After the passes of all views of a call: the rows that the workgroups of the two passes left for the background, the poses and
// the intrinsics are added up, up to kSumRows rows to a workgroup (x: a share of the background's rows, the one after the last
// share the camera's rows; y: the view), and added to the outputs with one atomic per value. (The passes used to end on these atomics
// themselves: 12 thousand workgroups of a full-HD view add to one line of memory, which serves some 10^8 of them a second. us,
// tile pass: 6M points 331 -> 318, 9M 252 -> 210, four crops of 512 x 512 151 -> 103, four views of clusters 443 -> 308; point
// pass: 300k points 33 -> 22, crops 149 -> 111, clusters 289 -> 269; this kernel: 4 to 8 a call.) The rows are summed in a fixed
// order, so a view of up to kSumRows blocks has the same sums in every run.
constexpr int kSumThreads = 1024;  // (a chain of round trips: the more rows requested together the shorter)
__global__ __launch_bounds__(kSumThreads) void backward_sums_kernel(const SumsParams p)
{
    const int view = blockIdx.y, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    __shared__ double s_acc[kSumThreads];
    if ((int)blockIdx.x < p.background_shares)
    {
        const int quads     = p.cpad / 4;  // 1, 2 or 4: a thread stays with one quad of channels
        const long long end = min((long long)p.background_rows, ((long long)blockIdx.x + 1) * kSumRows) * quads;
        const vf4* rows     = reinterpret_cast<const vf4*>(p.background_sums + (size_t)view * p.background_stride);
        double sum[4]       = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
        for (long long i = (long long)blockIdx.x * kSumRows * quads + threadIdx.x; i < end; i += kSumThreads)
        {
            const vf4 v = rows[i];
#pragma unroll
            for (int k = 0; k < 4; ++k) sum[k] += (double)v[k];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
        {
            for (int o = 32; o >= quads; o >>= 1) sum[k] += __shfl_xor(sum[k], o);
            if (lane < quads) s_acc[wave * 16 + 4 * lane + k] = sum[k];
        }
        __syncthreads();
        if ((int)threadIdx.x < p.channels)
        {
            const int i = threadIdx.x;
            double v = 0.0;
            for (int w = 0; w < kSumThreads / 64; ++w) v += s_acc[16 * w + i];
            if (v != 0.0) unsafeAtomicAdd(p.d_background + i, (float)v);
        }
        return;
    }
    // a value per lane, the rows dealt to the groups of kCameraSums threads
    constexpr int kGroups = kSumThreads / kCameraSums;
    const int group = (int)threadIdx.x / kCameraSums, i = (int)threadIdx.x - group * kCameraSums;
    const double* rows = p.camera_sums + (size_t)view * kCameraRows * kCameraSums;
    double v           = 0.0;
    if (group < kGroups)
    {
#pragma unroll 8
        for (int r = group; r < p.camera_rows; r += kGroups) v += rows[(size_t)r * kCameraSums + i];
    }
    s_acc[threadIdx.x] = v;
    __syncthreads();
    if ((int)threadIdx.x >= kCameraSums) return;
    for (int g = 1; g < kGroups; ++g) v += s_acc[g * kCameraSums + i];
    if (v == 0.0) return;
    if (i < 6)
    {
        if (p.d_pose) unsafeAtomicAdd(p.d_pose + 6 * (size_t)p.image_index[view] + i, v);
    }
    else if (i < 6 + 13)
    {
        if (p.d_intrinsics) unsafeAtomicAdd(p.d_intrinsics + 13 * (size_t)p.camera_index[view] + (i - 6), (float)v);
    }
}

// Before the two passes of a view: the rows of the view's pairs start as zeros (the tile pass writes the rows of the
// pairs that some pixel retained, the point pass reads all rows of a point): the two inline rows of every valid point
// (compact numbers are dense within each chunk of the binning kernels) and the overflow rows that the forward counted.
// For a view in which few pairs are retained (sparse_pair_rows) the flag bytes of the rows are cleared instead; the choice
// is left in the workspace for the two passes.
// On the first view of a call also, in
// overwrite mode (`texels`): the descriptor and confidence gradients of the columns that the point pass does not write
// itself. With the identity index (the forward noted it in the header) those are the columns past the last point;
// otherwise all of them, the point pass then adds with atomics. `clear_sums`: the outputs that backward_sums_kernel adds to
// (background, every pose row, every intrinsics row).
__global__ __launch_bounds__(256) void backward_prologue_kernel(const ViewHeader* __restrict__ header, const int32_t* __restrict__ chunk_valid,
                                                                int bin_groups, int points_per_block, float* __restrict__ rows_inline,
                                                                float* __restrict__ rows_over, unsigned char* __restrict__ flags, int32_t* __restrict__ mode, int force_mode, int pair_row, long long over_capacity,
                                                                float* __restrict__ d_texture,
                                                                float* __restrict__ d_confidence, int channels, int num_texels,
                                                                int num_points, int texels, int clear_sums,
                                                                float* __restrict__ d_background, double* __restrict__ d_pose,
                                                                int num_images, float* __restrict__ d_intrinsics, int num_cameras)
{
    long long over_rows = (long long)header->overflow_rows;
    if (over_rows > over_capacity) over_rows = over_capacity;
    // the view's retained entries: every workgroup adds the blend kernel's partial sums up for itself
    __shared__ unsigned long long s_retained[4];
    {
        unsigned long long r = (unsigned long long)(unsigned)chunk_valid[bin_groups + threadIdx.x];  // (kRetainedParts = 256 threads)
        for (int o = 32; o > 0; o >>= 1) r += __shfl_xor(r, o);
        if ((threadIdx.x & 63) == 0) s_retained[threadIdx.x >> 6] = r;
        __syncthreads();
    }
    const bool sparse = force_mode == 0 ? sparse_pair_rows((s_retained[0] + s_retained[1] + s_retained[2] + s_retained[3]) * kRetainedSample, header->n_entries)
                                        : force_mode == 2;
    if (blockIdx.x == 0 && threadIdx.x == 0) *mode = sparse ? 1 : 0;
    if (sparse)
    {
        // (the table ends on a multiple of 256 bytes: whole 16-byte words are cleared)
        const long long words = ((long long)num_points * TRIPS_MAX_LAYERS + 15) / 16;
        for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < words; i += (long long)gridDim.x * 256)
            reinterpret_cast<vu4*>(flags)[i] = vu4{0u, 0u, 0u, 0u};
    }
    else
    {
        // (rows are a multiple of four floats)
        const int row_quads = kInlineLayers * pair_row / 4;
        for (int chunk = blockIdx.x; chunk < bin_groups; chunk += gridDim.x)
        {
            const int begin = min(num_points, chunk * points_per_block);
            const int quads = chunk_valid[chunk] * row_quads;
            vf4* dst        = reinterpret_cast<vf4*>(rows_inline) + (size_t)begin * row_quads;
            for (int i = threadIdx.x; i < quads; i += 256) __builtin_nontemporal_store(vf4{0.f, 0.f, 0.f, 0.f}, dst + i);
        }
        const long long quads = over_rows * pair_row / 4;
        vf4* dst              = reinterpret_cast<vf4*>(rows_over);
        for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < quads; i += (long long)gridDim.x * 256)
            __builtin_nontemporal_store(vf4{0.f, 0.f, 0.f, 0.f}, dst + i);
    }
    if (clear_sums && blockIdx.x == 0)
    {
        if (d_background)
            for (int i = threadIdx.x; i < channels; i += 256) d_background[i] = 0.f;
        if (d_pose)
            for (int i = threadIdx.x; i < num_images * 6; i += 256) d_pose[i] = 0.0;
        if (d_intrinsics)
            for (int i = threadIdx.x; i < num_cameras * 13; i += 256) d_intrinsics[i] = 0.f;
    }
    if (!texels) return;
    const int first = header->not_identity == 0 ? min(num_points, num_texels) : 0;
    const int n     = num_texels - first;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < (long long)n * (channels + 1); i += (long long)gridDim.x * 256)
    {
        const int c = (int)(i / n), t = first + (int)(i - (long long)c * n);
        if (c < channels)
            d_texture[(size_t)c * num_texels + t] = 0.f;
        else
            d_confidence[t] = 0.f;
    }
}

template <int C, int K>
hipError_t launch_tiles(const BackwardParams& p, int blocks, hipStream_t stream)
{
    const size_t lds = tiles_lds_bytes((C + 3) & ~3, K);
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&backward_tiles_kernel<C, K>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((backward_tiles_kernel<C, K>), dim3(blocks), dim3(256), lds, stream, p);
    return hipSuccess;
}
// (a list of eight takes half of the LDS and a fourth of a lane's registers less: four workgroups per CU instead of two or three)
template <int C>
hipError_t launch_tiles(const BackwardParams& p, int blocks, hipStream_t stream)
{
    return p.list_depth <= 8 ? launch_tiles<C, 8>(p, blocks, stream) : launch_tiles<C, 16>(p, blocks, stream);
}

#define TRIPS_BW_DISPATCH(KERNEL, BLOCKS)                                                                      \
    switch (channels)                                                                                          \
    {                                                                                                          \
        case 3: hipLaunchKernelGGL((KERNEL<3>), dim3(BLOCKS), dim3(256), 0, stream, p); break;                 \
        case 4: hipLaunchKernelGGL((KERNEL<4>), dim3(BLOCKS), dim3(256), 0, stream, p); break;                 \
        case 6: hipLaunchKernelGGL((KERNEL<6>), dim3(BLOCKS), dim3(256), 0, stream, p); break;                 \
        case 8: hipLaunchKernelGGL((KERNEL<8>), dim3(BLOCKS), dim3(256), 0, stream, p); break;                 \
        case 16: hipLaunchKernelGGL((KERNEL<16>), dim3(BLOCKS), dim3(256), 0, stream, p); break;               \
        default: return hipErrorInvalidValue;                                                                  \
    }

// (Four workgroups per CU, each walking its share of the points; more leave more rows of sums. us, with 1024, 2048 and 4096, the sums
// behind the plus: 6M points in no order 166 + 6.5, 170 + 10 and 173 + 16; four views of clusters 254 + 8, 253 + 11 and 292 + 18; 9M in
// Morton order 253 + 6, 257 + 10 and 253 + 16; four views of 500k at 512 x 512 101 + 6, 110 + 8 and 110 + 8; 1.4M of sixteen channels
// 96 + 8, 96 + 9 and 99 + 13.)
int point_pass_blocks(int num_points) { return std::min((num_points + 255) / 256, kCameraRows); }

hipError_t launch_backward_view(const BackwardParams& p, int channels, hipStream_t stream, Profiler* prof)
{
    const int N = p.num_points;
    {
        ProfScope ps(prof, "backward_prologue", stream);
        hipLaunchKernelGGL(backward_prologue_kernel, dim3(2048), dim3(256), 0, stream, p.header, p.chunk_valid, p.bin_groups,
                           p.points_per_block, p.rows_inline, p.rows_over, p.flags, p.mode, p.force_mode, pair_row_floats((channels + 3) & ~3),
                           p.over_capacity, p.d_texture, p.d_confidence, channels, p.num_texels,
                           N, p.overwrite, p.clear_block_sums, p.d_background, p.d_pose_all, p.num_images, p.d_intrinsics_all,
                           p.num_cameras);
    }
    {
        // (no points: only the background receives gradient)
        ProfScope ps(prof, "backward_tiles", stream);
        const long long blocks8 = (((long long)p.blocks_off[p.num_layers] + 8 * kNumXcd - 1) / (8 * kNumXcd)) * (8 * kNumXcd);  // whole runs of 8 blocks x 8 XCDs
        const int blocks        = (int)blocks8;
        hipError_t e            = hipErrorInvalidValue;
        switch (channels)
        {
            case 3: e = launch_tiles<3>(p, blocks, stream); break;
            case 4: e = launch_tiles<4>(p, blocks, stream); break;
            case 6: e = launch_tiles<6>(p, blocks, stream); break;
            case 8: e = launch_tiles<8>(p, blocks, stream); break;
            case 16: e = launch_tiles<16>(p, blocks, stream); break;
            default: break;
        }
        if (e != hipSuccess) return e;
    }
    if (N > 0)
    {
        ProfScope ps(prof, "backward_points", stream);
        const int blocks = point_pass_blocks(N);
        TRIPS_BW_DISPATCH(backward_points_kernel, blocks);
    }
    return hipGetLastError();
}

hipError_t launch_backward_sums(SumsParams& p, int num_points, hipStream_t stream, Profiler* prof)
{
    ProfScope ps(prof, "backward_sums", stream);
    const bool camera   = num_points > 0 && (p.d_pose || p.d_intrinsics);
    p.background_shares = (p.background_rows + kSumRows - 1) / kSumRows;
    p.camera_rows       = point_pass_blocks(num_points);
    hipLaunchKernelGGL(backward_sums_kernel, dim3(p.background_shares + (camera ? 1 : 0), p.num_views), dim3(kSumThreads), 0, stream, p);
    return hipGetLastError();
}

}  // namespace trips
