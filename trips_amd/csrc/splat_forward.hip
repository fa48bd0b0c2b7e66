// Forward kernels of the splat path for gfx950 (wave64).
//
//   project_bin_kernel   <- CountAndCollectTiled (projection, validity, layer selection)
//                           src/lib/rendering/RenderForward.cu:168-366
//   bin_scan / bin_scatter / tile_count / tile_scatter
//                        <- per-pixel counting (:355-361), cub ExclusiveSum section (:1155-1232) and
//                           SplattingPass (:368-436)
//   cell_sort_kernel / blend_kernel
//                        <- FastSortFusedNew    src/lib/rendering/RenderForward.cu:474-1059
//
// Differences in shape, not in result. The reference increments one global counter per (point, layer, corner),
// scans layer by layer with two blocking read-backs each, and takes one more global atomic per entry to place
// its key. Scattered global atomics run at about 2.7e10 per second on this GPU, so here a (point, layer) pair is
// first binned, once, into the 32 x 32 pixel tile of its footprint's first pixel (workgroup-private LDS histograms
// and a column scan: no global atomics); a workgroup per tile then counts, scans and places the keys of its 1024
// cells with LDS atomics, one key per pair, and the blend gathers a pixel's list from the four cells whose
// footprints cover it. The sort is done per cell (each serves four pixels); a pixel is one lane of a wavefront that
// owns 8 x 8 of them, merges its four cell lists and blends front to back, instead of two lists per 32-lane warp; the
// per-point record gathered by the blend carries position, size, confidence and descriptor together; what is kept
// for the backward is the sorted id list per pixel (64 B) and a byte per list position that says which cell the
// entry came from and where it stood in that cell's list, instead of 16 x 7 floats.
#include "row16.h"
#include "splat_internal.h"
#include "trips_math.h"

#include <type_traits>

#pragma clang fp contract(off)

namespace trips
{
typedef unsigned vu4 __attribute__((ext_vector_type(4)));
typedef float vf4 __attribute__((ext_vector_type(4)));
typedef float vf2 __attribute__((ext_vector_type(2)));
typedef int vi4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ Camera load_camera(const double* pose, const float* intr, const TripsView& v,
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

// ---------------------------------------------------------------------------------------------------------
// Projection, validity and layer selection of one point (CountAndCollectTiled, RenderForward.cu:168-366; its per-pixel
// counter updates become per-tile ones).
struct PointProjection
{
    bool valid;
    int tex;        // descriptor column
    int layers;     // layers the point is written to (0 if culled)
    float ipx, ipy, z, size_px;
    float d_softplus;  // softplus'(raw size), training mode
};

// What the projection kernel reads of a point (fetched one step ahead of its use; the descriptor column, which the
// descriptor's loads need, two steps).
template <int CPAD>
struct PointInputs
{
    int tex;  // descriptor column
    float4 pos;
    float raw_size, dropout;
    float conf, d[CPAD];
};

template <int C, bool TRAIN, int CPAD>
__device__ __forceinline__ void load_point(const ForwardParams& p, int pid, int tex, PointInputs<CPAD>& in)
{
    in.tex      = tex;
    in.pos      = p.position[pid];
    in.raw_size = p.point_size[pid];
    in.dropout  = TRAIN && p.dropout ? p.dropout[pid] : 0.f;
    in.conf     = 0.f;
#pragma unroll
    for (int c = 0; c < CPAD; ++c) in.d[c] = 0.f;
    if ((unsigned)tex < (unsigned)p.num_texels)
    {
        in.conf = p.confidence[tex];
#pragma unroll
        for (int c = 0; c < C; ++c) in.d[c] = p.texture[(size_t)c * p.num_texels + tex];
    }
}

// The last pixels, first tile and tile columns of all layers, layer l's in lane l of four registers: a loop over the layers gets
// them with v_readlane, where loads of kernel arguments are four round trips of the scalar cache per layer, one behind the
// other, which wait for the wavefront's LDS atomics as well. The whole wavefront makes them, and the whole wavefront runs the
// loops that read them: a copy or a spill of such a register where only some lanes run would leave the other layers behind.
struct LayerTable
{
    int last_x, last_y, bin_off, tiles_x;
};
__device__ __forceinline__ LayerTable layer_table(const PyramidGeom& g)
{
    const int l = min((int)(threadIdx.x & 63), TRIPS_MAX_LAYERS - 1);
    LayerTable t;
    t.last_x  = g.w[l] - 1;
    t.last_y  = g.h[l] - 1;
    t.bin_off = g.bin_off[l];
    t.tiles_x = g.tiles_x[l];
    return t;
}

// `s_hist`: LDS counters, one per tile; every layer the point is written to adds one to the tile of the footprint's
// first pixel (px, py). (The footprint (px..px+1, py..py+1) lies inside the image because px < w-1 and py < h-1.)
// Called by the whole wavefront (see LayerTable); lanes with `live` unset have no point.
template <bool TRAIN, int CPAD>
__device__ __forceinline__ PointProjection project_point(const ForwardParams& p, const Camera& cam, int pid, bool live, const PointInputs<CPAD>& in,
                                                         int* s_hist, const double2* log_table, const LayerTable& layers,
                                                         bool& not_identity, bool& bad_index)
{
    PointProjection o;
    o.valid  = false;
    o.layers = 0;
    o.ipx = o.ipy = 0.f;
    o.z       = -1.f;
    o.size_px = 0.f;
    o.d_softplus = 0.f;
    const int L = p.num_layers;
    bool skip   = !live;
    o.tex       = in.tex;
    not_identity |= live && o.tex != pid;
    if (live && (unsigned)o.tex >= (unsigned)p.num_texels)
    {
        // a column outside the descriptor table: leave the point out (reported by the status query) rather
        // than read past the tables
        bad_index    = true;
        not_identity = true;  // the backward then never uses the point's own number as a column
        skip         = true;
    }
    if (p.viewer_only && in.conf < p.stability_cutoff_value) skip = true;
    if (TRAIN && in.dropout == 1.f) skip = true;
    float4 pos = in.pos;
    if (p.displacement && live)
    {
        const float* dsp = p.displacement + (size_t)pid * 3;
        pos.x += dsp[0];
        pos.y += dsp[1];
        pos.z += dsp[2];
    }
    const Projected pr = project(cam, pos.x, pos.y, pos.z);
    float radius_px    = quotient(pr.scale * pos.w, pr.iz);  // (only its whole pixels count)
    auto small = [&](float radius) { return p.drop_out_points_by_radius && float(trunc_sat(radius)) < p.drop_out_radius_threshold; };
    o.valid = !skip && pr.z > 0.f && pr.ipx >= 0.f && pr.ipx < float(p.geom.w[0] - 1) && pr.ipy >= 0.f &&
              pr.ipy < float(p.geom.h[0] - 1) && !small(radius_px);
    int layer_higher = 0;
    if (o.valid)
    {
        o.ipx = pr.ipx;
        o.ipy = pr.ipy;
        o.z   = pr.z;
        const float size = softplus(in.raw_size, log_table, TRAIN ? &o.d_softplus : nullptr);
        o.size_px        = quotient_of_any_size(pr.scale * size, pr.z, pr.iz);
        if (o.size_px > 1.f)
        {
            int lo, hi;
            log2_floor_ceil(o.size_px, lo, hi);
            layer_higher = min(hi, L - 1);
        }
    }
    float lx = o.ipx, ly = o.ipy;
    bool more = o.valid;
    for (int layer = 0; layer < L; ++layer, lx *= 0.5f, ly *= 0.5f, radius_px *= 0.5f)
    {
        const int last_x = __builtin_amdgcn_readlane(layers.last_x, layer), last_y = __builtin_amdgcn_readlane(layers.last_y, layer);
        const int bin_off = __builtin_amdgcn_readlane(layers.bin_off, layer), tiles_x = __builtin_amdgcn_readlane(layers.tiles_x, layer);
        const int px = (int)lx, py = (int)ly;
        more = more && layer <= layer_higher && px < last_x && py < last_y && !small(radius_px);
        if (__ballot(more) == 0) break;
        o.layers += more ? 1 : 0;  // (not layer + 1: the compiler then keeps the loop's own number per lane)
        if (more) atomicAdd(s_hist + bin_off + (int)__umul24((unsigned)(py >> kTileShift), (unsigned)tiles_x) + (px >> kTileShift), 1);
    }
    return o;
}

// Calls f(px, py, counter of the tile of (px, py)) for the layers a point is written to. Called by the whole wavefront (see
// LayerTable); lanes without a point have 0 layers.
template <typename F>
__device__ __forceinline__ void for_point_tiles(const LayerTable& t, float lx, float ly, int layers, int* tile_table, F&& f)
{
    for (int layer = 0; layer < TRIPS_MAX_LAYERS; ++layer, lx *= 0.5f, ly *= 0.5f)
    {
        if (__ballot(layer < layers) == 0) break;
        const int bin_off = __builtin_amdgcn_readlane(t.bin_off, layer), tiles_x = __builtin_amdgcn_readlane(t.tiles_x, layer);
        if (layer < layers)
        {
            const int px = (int)lx, py = (int)ly;  // (not negative)
            f(px, py, tile_table + bin_off + (int)__umul24((unsigned)(py >> kTileShift), (unsigned)tiles_x) + (px >> kTileShift));
        }
    }
}

// A workgroup of the two binning kernels owns one contiguous chunk of points and walks it one point per thread at a
// time. The valid points of the chunk are numbered in point order from the chunk's first point number on ("compact numbers":
// cid = chunk begin + rank among the chunk's valid points; per step a ballot per wavefront and one exchange of the
// wavefront counts through LDS). The numbers grow with the point id, so a sort key built from them orders like one
// built from point ids; the records written at them are dense from the start of every chunk (whole lines, nothing
// for culled points).
__device__ __forceinline__ void chunk_point_range(const ForwardParams& p, int chunk, int& begin, int& end)
{
    begin = min(p.num_points, chunk * p.points_per_block);
    end   = min(p.num_points, begin + p.points_per_block);
}
// The chunk of a workgroup: consecutive chunks share an XCD (workgroups are dealt to the eight of them in turn). Worth about 1 %
// of the projection where it saves a training step's records: 6M points in no order 139.0 -> 137.7 us, 3M in a ball 83.1 ->
// 81.8, 4M clustered 112.8 -> 111.6; without the saved state, and at 9M in Morton order, nothing (128.7 and 129.0, 189.3 and 190.4).
// The scatter's time does not change (a few entries of a chunk under every tile: 108.6 and 109.4 us at 6M in no order, others
// alike), but its lines leave in more parts: 198 MB written instead of 169 there (without the saved state 184 instead of 151), as
// much as before in Morton order and of clusters.
__device__ __forceinline__ int chunk_of_workgroup()
{
    static_assert(kBinGroups % kNumXcd == 0, "equal shares");
    return (int)(blockIdx.x % kNumXcd) * (kBinGroups / kNumXcd) + (int)(blockIdx.x / kNumXcd);
}

// Projection, validity, layer selection; the records of the valid points at their compact numbers; LDS histogram of
// the tiles that this workgroup's points fall into.
template <int C, bool TRAIN>
__global__ __launch_bounds__(kBinThreads) void project_bin_kernel(const ForwardParams p)
{
    constexpr int CPAD  = (C + 3) & ~3;
    constexpr int NREC  = 1 + CPAD / 4;  // float4 per blend record
    constexpr int WAVES = kBinThreads / 64;
    extern __shared__ int s_hist[];  // bin entries of this workgroup's points, one counter per tile
    __shared__ int s_valid[2][WAVES];  // valid points of every wavefront in this step (two steps in flight)
    __shared__ double2 s_log[kLogTable];
    __shared__ vf4 s_rec[WAVES][64 * NREC];  // a wavefront's records of a step
    __shared__ int s_flags;            // bit 0: not_identity, bit 1: bad_index, of any point of the chunk
    const Camera cam  = load_camera(p.pose, p.intrinsics, p.view, p.dist_cutoff);
    const int L       = p.num_layers;
    const int NB      = p.geom.bin_off[L];
    bool not_identity = false;  // some point's descriptor column differs from its own index
    bool bad_index    = false;
    for (int i = threadIdx.x; i < NB; i += kBinThreads) s_hist[i] = 0;
    const LayerTable layers = layer_table(p.geom);
    if (threadIdx.x < kLogTable) s_log[threadIdx.x] = log_table_entry(threadIdx.x);
    if (threadIdx.x == 0) s_flags = 0;
    __syncthreads();

    int begin, end;
    const int chunk = chunk_of_workgroup();
    chunk_point_range(p, chunk, begin, end);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int next       = begin;  // workgroup-uniform: compact number of the chunk's next valid point
    int next_pair  = 0;      // workgroup-uniform: overflow rows of the chunk's points so far
    int step       = 0;
    // The loads of the next step's points, their descriptors and dropout flags among them (whether a point is visible or
    // not), are in flight while this step's are projected. (With the dropout flag and the descriptor requested in the
    // step itself, its waits were a part of every step: 9M points with dropout 225 -> 197 us.) What bounds it: without the saved
    // state the 430 MB that it moves at 6M points, 4.5 TB/s; with it the stores, 477 MB at 3.8 TB/s (that the next step waits for
    // them is not it: without branches around loads and stores, so that nothing waits for a store, it took 137 us instead of
    // 131). Before the short exp and log and the layers' table it was its vector instructions, 91 us of them: eval 6M in Morton
    // order 126 -> 99 us, train 6M 138 -> 131, 9M 191 -> 173, 4M clustered 111 -> 105 a view (then two stores less: see prec).
    // With a point's record stored by its own lane, 16 bytes of 32 (80 at 16 channels) at a time, a store touched twice (five
    // times) the lines that it filled: as runs of the wavefront 4M clustered 100 -> 91 us a view, 9M 170 -> 163, 1M without the saved
    // state 27.6 -> 26, 500k of sixteen channels 51 -> 22; 6M in no order, of which a view culls two in five, 125 both ways.
    // With culled points kept in the loop over the layers instead of leaving before it: 6M in no order 125 -> 114, 4M clustered 91 -> 85
    // a view, 9M 168 -> 160, 1M without the saved state 25.3 -> 23.8 (477 MB at 4.2 TB/s, without the saved state 430 MB at 4.4); three
    // clouds of 6M in turn, whose inputs then all come from memory, 146 to 151 before and 1 to 2 more now.
    PointInputs<CPAD> nxt{};
    int next_tex = 0;  // descriptor column of the step after `nxt`'s
    if (begin + (int)threadIdx.x < end)
    {
        const int tex = p.index[begin + (int)threadIdx.x];
        if (begin + (int)threadIdx.x + kBinThreads < end) next_tex = p.index[begin + (int)threadIdx.x + kBinThreads];
        load_point<C, TRAIN>(p, begin + (int)threadIdx.x, tex, nxt);
    }
    for (int base = begin; base < end; base += kBinThreads, step ^= 1)
    {
        const int pid              = base + threadIdx.x;
        const PointInputs<CPAD> in = nxt;
        if (pid + kBinThreads < end) load_point<C, TRAIN>(p, pid + kBinThreads, next_tex, nxt);
        if (pid + 2 * kBinThreads < end) next_tex = p.index[pid + 2 * kBinThreads];
        const PointProjection o = project_point<TRAIN>(p, cam, pid, pid < end, in, s_hist, s_log, layers, not_identity, bad_index);
        const unsigned long long vm = __ballot(o.valid);
        const unsigned long long below = (1ull << lane) - 1ull;
        // rows of the backward's overflow table (one per layer past the second) of the wavefront's points before this
        // one, and of the wavefront: 0..6 per point, one ballot per bit
        int pairs_before = 0, pairs_wave = 0;
        if (TRAIN)
        {
            const int extra = max(o.layers - kInlineLayers, 0);
#pragma unroll
            for (int b = 0; b < 3; ++b)
            {
                const unsigned long long m = __ballot((extra >> b) & 1);
                pairs_before += (int)__popcll(m & below) << b;
                pairs_wave += (int)__popcll(m) << b;
            }
        }
        // both counts of a wavefront in one word (at most 64 valid points and 384 rows per wavefront, 1024 and 6144 per
        // step: 16 bits each); every wavefront then takes the prefix over the 16 words in its 16-lane rows
        if (lane == 0) s_valid[step][wave] = (int)__popcll(vm) | (pairs_wave << 16);
        __syncthreads();
        static_assert(WAVES == 16, "the prefix below runs over one 16-lane row");
        const int word = s_valid[step][lane & (WAVES - 1)];  // the counts of wavefront w in lane w of every row
        const int inc  = row_inclusive_scan(word);
        const int upto = __builtin_amdgcn_readlane(inc, WAVES - 1);                                    // the step's totals
        const int excl = __builtin_amdgcn_readlane(inc - word, __builtin_amdgcn_readfirstlane(wave));  // the wavefronts before this one
        const int before = excl & 0xFFFF, pbefore = excl >> 16, total = upto & 0xFFFF, ptotal = upto >> 16;
        const int cid        = next + before + (int)__popcll(vm & below);
        const int first_pair = next_pair + pbefore + pairs_before;  // within the chunk
        next += total;
        next_pair += ptotal;
        if (TRAIN && pid < end) p.cid_of[pid] = o.valid ? cid : ~cid;
        // records for the blend (and the pixel pass of the backward): those of the wavefront's valid points follow each other, and
        // leave through LDS as one run of 16 bytes a lane
        vf4* const mine = s_rec[wave];
        const int rank  = (int)__popcll(vm & below), words = (int)__popcll(vm) * NREC;
        if (o.valid)
        {
            vf4* const to = mine + rank * NREC;
            to[0]         = vf4{o.ipx, o.ipy, encode_size_field(o.size_px, L), in.conf};
#pragma unroll
            for (int q = 0; q < CPAD / 4; ++q) to[1 + q] = vf4{in.d[4 * q], in.d[4 * q + 1], in.d[4 * q + 2], in.d[4 * q + 3]};
            // point record: depth and layers for the scatter pass; first overflow row, softplus' and the size for the backward (without
            // it 8 bytes: a frame of 6M points 1.5 us less here and in the scatter)
            if constexpr (TRAIN)
                __builtin_nontemporal_store(vf4{o.z, __uint_as_float((unsigned)o.layers | (unsigned)first_pair << kLayersBits), o.d_softplus, o.size_px},
                                            reinterpret_cast<vf4*>(p.prec) + cid);
            else
                __builtin_nontemporal_store(vf2{o.z, __uint_as_float((unsigned)o.layers)}, reinterpret_cast<vf2*>(p.prec) + cid);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        vf4* const rec = reinterpret_cast<vf4*>(p.rec + (size_t)(cid - rank) * p.rec_floats);
#pragma unroll
        for (int q = 0; q < NREC; ++q)
            if (64 * q + lane < words) __builtin_nontemporal_store(mine[64 * q + lane], rec + 64 * q + lane);
    }
    {
        const int flags = (__ballot(not_identity) != 0 ? 1 : 0) | (__ballot(bad_index) != 0 ? 2 : 0);
        if (flags && lane == 0) atomicOr(&s_flags, flags);
    }

    // this workgroup's row of the histogram matrix [workgroup][bin]; its valid points and flags for the scan kernel,
    // which adds the chunks up (no counter of the view is touched here: nothing has to be cleared before this kernel)
    __syncthreads();
    int32_t* row = p.bin_hist + (size_t)chunk * NB;
    for (int i = threadIdx.x; i < NB; i += kBinThreads) row[i] = s_hist[i];
    if (threadIdx.x == 0)
    {
        p.chunk_valid[chunk]                    = next - begin;
        p.chunk_valid[p.bin_groups + chunk]     = s_flags;
        p.chunk_valid[2 * p.bin_groups + chunk] = next_pair;
    }
}

// ---------------------------------------------------------------------------------------------------------
// Column-wise exclusive prefix of the histogram matrix [workgroup][bin]: afterwards hist[g][bin] = entries of
// `bin` that come from workgroups before g, and bin_count[bin] = the column total. No atomics anywhere in the
// binning, since atomics on a few thousand hot counters serialise. A workgroup owns 16 columns; its 16 row
// segments are summed side by side, prefixed through LDS, then each segment writes its rows' prefixes (one thread
// walking a whole column is a chain of G dependent-latency steps). A thread requests its 16 rows together and keeps them for the
// prefix: read twice, eight at a time, 5.5 us instead of 4.3 at 512 x 512, 9.7 instead of 8.7 at 1920 x 1080.
// A workgroup also clears the per-cell counters `counts` and `run` of those of its tiles that may be split: their slices add
// to them. Those of any other tile are written, not added to, where its keys are placed (clearing all of them is 22 MB at
// 1920 x 1080 and eight layers).
//
// The last workgroup adds up the chunks of the projection: the number of every chunk's first overflow row, and the view's
// counters, written (not added to, so that nothing has to clear them first); on the first view of a call the status block of
// the whole call as well. The scan over the tiles' totals is the scatter pass's (plan_tiles).
constexpr int kScanCols = 16, kScanSegs = 16;
static_assert(kBinGroups % kScanSegs == 0, "equal segments");
__device__ __forceinline__ int wave_inclusive_scan(int x)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1)
    {
        const int t = __shfl_up(x, o);
        if (lane >= o) x += t;
    }
    return x;
}
// sum over the wavefronts before this one, and over all of them
template <int WAVES>
__device__ __forceinline__ int waves_before(const int* waves, int& all)
{
    const int wave = threadIdx.x >> 6;
    int before     = 0;
    all            = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w)
    {
        const int x = waves[w];
        before += w < wave ? x : 0;
        all += x;
    }
    return before;
}

__device__ __forceinline__ void sum_chunks(const ForwardParams& p, bool first_view)
{
    static_assert(kBinGroups == 256 && kRetainedParts == 256, "a thread per chunk, and per part");
    constexpr int G = kBinGroups;
    __shared__ int s_over[4], s_valid[4], s_flag[4];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int valid = p.chunk_valid[t], flags = p.chunk_valid[G + t], over = p.chunk_valid[2 * G + t];
    const int inc_over = wave_inclusive_scan(over), inc_valid = wave_inclusive_scan(valid);
    const int wave_flags = (__ballot(flags & 1) ? 1 : 0) | (__ballot(flags & 2) ? 2 : 0);
    if (lane == 63) s_over[wave] = inc_over, s_valid[wave] = inc_valid, s_flag[wave] = wave_flags;
    __syncthreads();
    int total_over, total_valid;
    const int first_over = waves_before<4>(s_over, total_over) + inc_over - over;
    waves_before<4>(s_valid, total_valid);
    if (p.saved_chunk_valid)
    {
        p.saved_chunk_valid[G + kRetainedParts + t] = first_over;
        p.saved_chunk_valid[t]     = valid;
        p.saved_chunk_valid[G + t] = 0;  // (the blend adds)
    }
    if (t == 0)
    {
        const int any_flags = s_flag[0] | s_flag[1] | s_flag[2] | s_flag[3];
        *p.long_count       = 0;
        const unsigned long long bad = (unsigned long long)((any_flags >> 1) & 1);
        p.header->n_valid       = (unsigned long long)(unsigned)total_valid;
        p.header->overflow      = 0;
        p.header->retained      = 0;
        p.header->not_identity  = (unsigned long long)(any_flags & 1);
        p.header->bad_index     = 0;
        p.header->overflow_rows = (unsigned long long)(unsigned)total_over;
        if (first_view)
        {
            ViewHeader* status = p.status;
            status->n_valid = status->n_entries = status->overflow = status->retained = status->not_identity = 0;
            status->bad_index                                                       = bad;
            status->overflow_rows                                                   = 0;
        }
        else if (bad)
            p.status->bad_index = 1;  // (the views of a call run one after the other on the stream)
    }
}

__global__ __launch_bounds__(256) void bin_column_scan_kernel(const ForwardParams p, int first_view)
{
    if (blockIdx.x == gridDim.x - 1)
    {
        sum_chunks(p, first_view != 0);
        return;
    }
    __shared__ int s_seg[kScanSegs][kScanCols];
    __shared__ int s_total[kScanCols];
    const int NB = p.geom.bin_off[p.num_layers];
    const int c = threadIdx.x % kScanCols, seg = threadIdx.x / kScanCols;
    const int bin0 = blockIdx.x * kScanCols, bin = bin0 + c;
    constexpr int kRows = kBinGroups / kScanSegs;
    const bool live = bin < NB;
    int32_t* col    = p.bin_hist + (size_t)(seg * kRows) * NB + bin;
    int v[kRows], sum = 0;  // (all requested together, and kept for the prefix)
#pragma unroll
    for (int k = 0; k < kRows; ++k) v[k] = live ? col[(size_t)k * NB] : 0;
#pragma unroll
    for (int k = 0; k < kRows; ++k) sum += v[k];
    s_seg[seg][c] = sum;
    __syncthreads();
    int run = 0;
#pragma unroll
    for (int k = 0; k < kScanSegs; ++k) run += k < seg ? s_seg[k][c] : 0;
#pragma unroll
    for (int k = 0; k < kRows; ++k)
    {
        if (live) col[(size_t)k * NB] = run;
        run += v[k];
    }
    if (seg == kScanSegs - 1)
    {
        s_total[c] = run;  // (of columns past the last: 0)
        if (live) p.bin_count[bin] = run;
    }
    __syncthreads();
    // (a superset of the tiles that are split: entries past the capacity may leave a tile whole)
    static_assert(kTilePixels == 4 * 256, "four cells of a thread");
    for (int k = 0; k < kScanCols; ++k)
        if (s_total[k] > kSliceEntries)
        {
            const size_t at = (size_t)(bin0 + k) * (kTilePixels / 4) + threadIdx.x;
            reinterpret_cast<int4*>(p.counts)[at] = make_int4(0, 0, 0, 0);
            reinterpret_cast<int4*>(p.run)[at]    = make_int4(0, 0, 0, 0);
        }
}

// ---------------------------------------------------------------------------------------------------------
// A bin entry holds what the list kernels need of a (point, layer) pair: the depth bits, the compact point number and
// the cell of its tile that the footprint starts at. Depths of valid points are positive (31 bits), a cell takes 10
// bits, so clouds of up to 2^23 points have entries of 8 bytes; larger ones use 16.
template <bool PACKED>
struct BinEntry;
template <>
struct BinEntry<true>
{
    using T = u64;
    static __device__ __forceinline__ T make(unsigned zbits, unsigned cid, int px, int py)
    {
        const unsigned cell = (unsigned)((py & (kTile - 1)) << kTileShift) | (unsigned)(px & (kTile - 1));
        return ((u64)zbits << (kPackedIdBits + 2 * kTileShift)) | ((u64)cid << (2 * kTileShift)) | cell;
    }
    static __device__ __forceinline__ int cell(const T& e) { return (int)((unsigned)e & (kTilePixels - 1)); }
    static __device__ __forceinline__ u64 key(const T& e)
    {
        return ((e >> (kPackedIdBits + 2 * kTileShift)) << 32) | ((e >> (2 * kTileShift)) & ((1u << kPackedIdBits) - 1));
    }
};
template <>
struct BinEntry<false>
{
    using T = uint4;
    static __device__ __forceinline__ T make(unsigned zbits, unsigned cid, int px, int py)
    {
        const unsigned cell = (unsigned)((py & (kTile - 1)) << kTileShift) | (unsigned)(px & (kTile - 1));
        return make_uint4(zbits, cid, cell, 0u);
    }
    static __device__ __forceinline__ int cell(const T& e) { return (int)e.z; }
    static __device__ __forceinline__ u64 key(const T& e) { return ((u64)e.x << 32) | (u64)e.y; }
};
static_assert(kTilePixels == 1 << (2 * kTileShift), "a cell number takes 2 kTileShift bits");

// The plan of the view's tiles, from their totals:
//   * exclusive scan: bin_start[i] = sum_{k<i} bin_count[k], bin_start[NB] = total;
//   * slices of split tiles: a tile with more than kSliceEntries bin entries (hundreds of points per pixel, e.g.
//     tight clusters) would keep a single workgroup busy for milliseconds; it is cut into slices of kSliceEntries
//     entries, each a workgroup of its own. slice_start[t] = number of slices of split tiles before tile t;
//   * coarse_first: whether cell sort and blend begin with the coarsest layer, whose lists are the longest, so that no few
//     workgroups are left over at the end. Not where fewer than a third of the tiles hold anything: what they hold is long in
//     every layer, and side by side on a CU the heaviest slow each other down. us, cell sort and blend, finest layer first and
//     coarsest: 1M in a ball 48 + 89 and 35 + 79, 6M in no order 57 + 190 and 51 + 176, 9M in Morton order 37 + 119 and 35 + 105,
//     500k at 700 x 500 15 + 48 and 12 + 39, four views of 64 tight clusters 197 + 208 and 208 + 219. (Both spread evenly among each
//     other: between the two.)
// Every workgroup of the scatter pass makes the scan for itself (a few values of a thread, two barriers) and keeps its
// cursors in `s_cur`; the first one writes scan and slices for the kernels behind. Bound by its round trips: 1.7 us longer the
// scatter (2.6 at 2700 tiles) and a launch between column scan and scatter less, whose single workgroup took 4.5: 100k
// points at 512^2 53.9 -> 52.1 us for the whole render, 20k at 160 x 120 with the network 98.7 -> 94.7, 1M at 1920 x 1080
// 237.5 -> 234.4.
constexpr int kPlanPer = (kMaxBins + kBinThreads - 1) / kBinThreads;  // tiles of a thread
__device__ __forceinline__ void plan_tiles(const ForwardParams& p, const int32_t* __restrict__ row, int NB, int* __restrict__ s_cur)
{
    constexpr int WAVES = kBinThreads / 64;
    __shared__ int s_tiles[WAVES], s_slices[WAVES], s_filled[WAVES];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int per  = (NB + kBinThreads - 1) / kBinThreads;
    const int t0   = (int)threadIdx.x * per;
    int v[kPlanPer], before[kPlanPer], sum = 0;
#pragma unroll
    for (int j = 0; j < kPlanPer; ++j)
    {
        const bool live = j < per && t0 + j < NB;
        v[j]      = live ? p.bin_count[t0 + j] : 0;
        before[j] = live ? row[t0 + j] : 0;  // entries of the chunks before this one
    }
#pragma unroll
    for (int j = 0; j < kPlanPer; ++j) sum += v[j];
    const int inc_tiles = wave_inclusive_scan(sum);
    if (lane == 63) s_tiles[wave] = inc_tiles;
    __syncthreads();
    int total;
    const int first0 = waves_before<WAVES>(s_tiles, total) + inc_tiles - sum;  // first slot of the thread's first tile
    int first = first0;
#pragma unroll
    for (int j = 0; j < kPlanPer; ++j)
    {
        if (j < per && t0 + j < NB) s_cur[t0 + j] = first + before[j];
        first += v[j];
    }
    if (blockIdx.x == 0)
    {
        // slices of the tiles' entries that fit the capacity; tiles with any
        int sl[kPlanPer], slices = 0, filled = 0;
        first = first0;
#pragma unroll
        for (int j = 0; j < kPlanPer; ++j)
        {
            sl[j] = 0;
            if (j < per && t0 + j < NB)
            {
                p.bin_start[t0 + j]  = first;
                const long long last = min((long long)first + v[j], p.capacity);
                const long long n    = max(last - (long long)first, 0ll);
                sl[j]                = n > kSliceEntries ? (int)((n + kSliceEntries - 1) / kSliceEntries) : 0;
            }
            first += v[j];
            slices += sl[j];
            filled += (int)__popcll(__ballot(v[j] > 0));
        }
        if (lane == 0) s_filled[wave] = filled;
        const int inc_slices = wave_inclusive_scan(slices);
        if (lane == 63) s_slices[wave] = inc_slices;
        __syncthreads();
        int total_slices;
        int first_slice = waves_before<WAVES>(s_slices, total_slices) + inc_slices - slices;
#pragma unroll
        for (int j = 0; j < kPlanPer; ++j)
        {
            if (j < per && t0 + j < NB) p.slice_start[t0 + j] = first_slice;
            first_slice += sl[j];
        }
        if (threadIdx.x == 0)
        {
            p.bin_start[NB]     = total;
            p.slice_start[NB]   = total_slices;
            p.header->n_entries = (unsigned long long)(unsigned)total;
            int all_filled;
            waves_before<WAVES>(s_filled, all_filled);
            *p.coarse_first = 3 * all_filled >= NB ? 1 : 0;
        }
    }
    __syncthreads();
}

// One bin entry per (point, layer), in the tile of the footprint's first pixel. A workgroup walks
// the records that its chunk of the points left at the compact numbers; its slots inside every bin are contiguous
// and start at bin_start[bin] + hist[workgroup][bin]. (The layers' tiles come from registers, see LayerTable: 4M clustered 77 ->
// 73 us a view; walked by whole wavefronts, 9M points with entries of 16 bytes 101 -> 104, the others as before.)
template <bool PACKED>
__global__ __launch_bounds__(kBinThreads) void bin_scatter_kernel(const ForwardParams p)
{
    using E = BinEntry<PACKED>;
    typename E::T* __restrict__ entries = reinterpret_cast<typename E::T*>(p.bin_entries);
    extern __shared__ int s_cur[];
    const int NB    = p.geom.bin_off[p.num_layers];
    const int chunk = chunk_of_workgroup();
    const LayerTable layers = layer_table(p.geom);
    plan_tiles(p, p.bin_hist + (size_t)chunk * NB, NB, s_cur);
    int begin, end;
    chunk_point_range(p, chunk, begin, end);
    const int n      = p.chunk_valid[chunk];
    unsigned dropped = 0;
    // Records of a thread that are requested together. Loads and stores of a wavefront return in the order of their issue: a
    // load that follows scattered stores waits for them, so there are as few such turns as registers allow: one where no chunk
    // has more than U * kBinThreads = 16384 valid points, which clouds of up to 4.19M points never do. Two at a time / 8 / 16,
    // us: 6M points in no order 103 / 89 / 81 and with the saved state 109 / 113 / 109, 4M clustered 91 / 84 / 79, 3M in a ball
    // 61 / 58 / 55, 1M 22 / 21 / 21; 9M in Morton order 40 / 35 / 39.
    constexpr int U = 16;
    for (int first = begin; first < begin + n; first += U * kBinThreads)
    {
        const int cid0 = first + (int)threadIdx.x;
        vf2 tail[U];  // {depth, layers}
        float2 ip[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
        {
            const int cid = cid0 + u * kBinThreads;
            if (cid < begin + n)
            {
                tail[u] = __builtin_nontemporal_load(reinterpret_cast<const vf2*>(p.prec + (size_t)cid * p.prec_floats));
                ip[u]   = *reinterpret_cast<const float2*>(p.rec + (size_t)cid * p.rec_floats);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
        {
            const int cid   = cid0 + u * kBinThreads;
            const bool live = cid < begin + n;
            if (__ballot(live) == 0) break;
            const unsigned zbits = __float_as_uint(tail[u].x);
            for_point_tiles(layers, ip[u].x, ip[u].y, live ? (int)(__float_as_uint(tail[u].y) & kLayersMask) : 0, s_cur,
                            [&](int px, int py, int* bc)
                            {
                                const int slot = atomicAdd(bc, 1);
                                if ((unsigned long long)(unsigned)slot < (unsigned long long)p.capacity)
                                    entries[slot] = E::make(zbits, (unsigned)cid, px, py);
                                else
                                    dropped += 1;
                            });
        }
    }
    if (dropped) atomicAdd(&p.status->overflow, (u64)dropped);
}

// ---------------------------------------------------------------------------------------------------------
// Walks entries [0, n) with the workgroup, U loads of a thread in flight together.
template <int THREADS, int U, typename T, typename F>
__device__ __forceinline__ void for_entries(const T* __restrict__ entries, int n, F&& f)
{
    for (int i0 = threadIdx.x; i0 < n; i0 += U * THREADS)
    {
        T e[U];
#pragma unroll
        for (int j = 0; j < U; ++j)
            if (i0 + THREADS * j < n) e[j] = entries[i0 + THREADS * j];
#pragma unroll
        for (int j = 0; j < U; ++j)
            if (i0 + THREADS * j < n) f(e[j]);
    }
}

// The keys of a tile are filed by cell: the cell (px, py) holds the points whose 2 x 2 footprint starts at that pixel,
// so that a (point, layer) pair is written once and the four pixels it covers gather it from the cell. There is one key
// per bin entry: the keys of a tile start where its bin entries do.
// One workgroup per tile (blocks [0, NB)) plus one per slice of a split tile (blocks from there on; those past the
// number of slices the plan found return at once). Pass `SCATTER == false`: count the entries of the tile's 1024
// cells in LDS and write the counts (split tiles only). Pass `SCATTER == true`: the counts of a tile that is not
// split, then the exclusive scan of the 1024 counts, per-cell list starts, and the 64-bit keys (depth bits << 32 | compact point number) into their lists. A slice adds its counts to the
// tile's with atomics; when it places its keys it first counts its own entries per cell again and claims that many
// slots of each cell's list with one atomic.
// (THREADS: 256 for the counting pass, whose idle workgroups for unused slices are cheaper that way. The placement pass is a
// chain of round trips and barriers per tile, so as many tiles as possible should be under way on a CU: four workgroups of
// 512 with 39 KB of LDS each. Two of 1024 with 64 KB, and these: 6M points
// in no order 57 -> 50 us, in Morton order without the saved state 36 -> 26, 1M in a ball 37 -> 30.)
constexpr int kScatterThreads = 512;
template <bool SCATTER, int THREADS, bool PACKED>
__global__ __launch_bounds__(THREADS) void tile_lists_kernel(const ForwardParams p)
{
    using E  = BinEntry<PACKED>;
    using ET = typename E::T;
    __shared__ int s_cnt[kTilePixels];
    // per-cell entries of a slice (placement pass only; one word in the counting pass, whose code below never runs)
    __shared__ int s_mine[SCATTER ? kTilePixels : 1];
    auto mine = [&](int i) -> int& { return s_mine[SCATTER ? i : 0]; };
    __shared__ int s_wave[THREADS / 64];
    const int NB = p.geom.bin_off[p.num_layers];
    int bin      = blockIdx.x;
    int slice    = -1;  // -1: the tile's own workgroup
    if (bin >= NB)
    {
        // Runs of eight consecutive slices share an XCD (workgroups are dealt to the eight of them in turn): the slices of a
        // tile store their keys side by side all over the tile's lists, and an L2 that sees them all writes whole lines (a
        // render of 3.3M points at 1112 x 583: 64 -> 56 us).
        const int tiles8 = (NB + kNumXcd - 1) / kNumXcd * kNumXcd;
        if (bin < tiles8) return;
        const int e = (int)xcd_tile_block(bin - tiles8, 8);
        if (e >= p.slice_start[NB]) return;
        // the tile with slice_start[t] <= e < slice_start[t + 1]: a split one, tiles without slices have empty ranges
        int lo = 0, hi = NB;
        while (hi - lo > 1)
        {
            const int mid = (lo + hi) >> 1;
            if (p.slice_start[mid] <= e)
                lo = mid;
            else
                hi = mid;
        }
        bin   = lo;
        slice = e - p.slice_start[bin];
    }
    long long first = p.bin_start[bin];
    long long last  = p.bin_start[bin + 1];
    if (last > p.capacity) last = p.capacity;  // entries beyond the capacity were dropped by the scatter
    const bool split = last - first > kSliceEntries;
    if (slice >= 0)
    {
        first += (long long)slice * kSliceEntries;
        last = min(last, first + kSliceEntries);
    }
    const int n          = first < last ? (int)(last - first) : 0;
    const ET* entries    = reinterpret_cast<const ET*>(p.bin_entries) + first;
    int32_t* counts      = p.counts + (size_t)bin * kTilePixels;

    if (!SCATTER)
    {
        if (slice < 0) return;  // the slices count for a split tile; any other tile is counted where its keys are placed
        for (int i = threadIdx.x; i < kTilePixels; i += THREADS) s_cnt[i] = 0;
        __syncthreads();
        // (sixteen loads of a thread in flight: the slices of a view are few, and the kernel lasts as long as one slice's
        // round trips to memory, one after the other)
        for_entries<THREADS, 16>(entries, n, [&](const ET& e) { atomicAdd(&s_cnt[E::cell(e)], 1); });
        __syncthreads();
        for (int i = threadIdx.x; i < kTilePixels; i += THREADS)
        {
            const int c = s_cnt[i];
            if (c) atomicAdd(&counts[i], c);  // cleared before this kernel
        }
        return;
    }

    // This workgroup files at most kSliceEntries entries: a thread reads its share once, all loads in flight together,
    // and keeps it in registers from the count to the placement.
    constexpr int MAXE = (kSliceEntries + THREADS - 1) / THREADS;
    ET mine_e[MAXE];
    const int n_filed = split && slice < 0 ? 0 : n;  // (the workgroup of a split tile files nothing itself)
#pragma unroll
    for (int j = 0; j < MAXE; ++j)
        if ((int)threadIdx.x + j * THREADS < n_filed) mine_e[j] = entries[(int)threadIdx.x + j * THREADS];
    auto for_mine = [&](auto&& f)
    {
#pragma unroll
        for (int j = 0; j < MAXE; ++j)
            if ((int)threadIdx.x + j * THREADS < n_filed) f(mine_e[j]);
    };
    // exclusive scan of the tile's 1024 lengths: PER consecutive pixels per thread
    constexpr int PER = kTilePixels / THREADS;
    const int base4   = threadIdx.x * PER;
    int v[PER], sum = 0;
    if (!split)
    {
        for (int i = threadIdx.x; i < kTilePixels; i += THREADS) s_cnt[i] = 0;
        __syncthreads();
        for_mine([&](const ET& e) { atomicAdd(&s_cnt[E::cell(e)], 1); });
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < PER; ++i)
    {
        if (split)
            v[i] = counts[base4 + i];
        else
            counts[base4 + i] = v[i] = s_cnt[base4 + i];  // (the slots that this thread overwrites with the list starts below)
        sum += v[i];
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int inc = sum;
    for (int o = 1; o < 64; o <<= 1)
    {
        int t = __shfl_up(inc, o);
        if (lane >= o) inc += t;
    }
    if (lane == 63) s_wave[wave] = inc;
    if (slice >= 0)
        for (int i = threadIdx.x; i < kTilePixels; i += THREADS) mine(i) = 0;
    __syncthreads();
    int prefix = inc - sum;
    for (int w = 0; w < wave; ++w) prefix += s_wave[w];
    const int key_start = p.bin_start[bin];  // one key per bin entry: the tile's keys start where its entries do
    int32_t* cursor     = p.cursor + (size_t)bin * kTilePixels;
#pragma unroll
    for (int i = 0; i < PER; ++i)
    {
        s_cnt[base4 + i] = key_start + prefix;  // running slot of the cell
        if (slice < 0)
        {
            int where = key_start + prefix;
            if (v[i] > kLongList && (long long)key_start + prefix + v[i] <= p.capacity)
            {
                // a long list: hand its segments to the reduction pass and point the cell at their results
                const int nseg = (v[i] + kLongSegment - 1) / kLongSegment;
                const int base = atomicAdd(p.long_count, nseg);
                if (base + nseg <= p.max_long_items)
                {
                    for (int sg = 0; sg < nseg; ++sg)
                        p.long_items[base + sg] = make_int2(key_start + prefix + sg * kLongSegment, min(kLongSegment, v[i] - sg * kLongSegment));
                    where = -1 - base;
                }
            }
            cursor[base4 + i] = where;
        }
        prefix += v[i];
    }
    if (split && slice < 0) return;  // the slices place the keys
    __syncthreads();
    unsigned dropped = 0;
    if (slice >= 0)
    {
        // this slice's share of every cell's list: count, then claim the slots with one atomic per cell
        int32_t* run = p.run + (size_t)bin * kTilePixels;
        for_mine([&](const ET& e) { atomicAdd(&mine(E::cell(e)), 1); });
        __syncthreads();
        for (int i = threadIdx.x; i < kTilePixels; i += THREADS)
        {
            const int c = mine(i);
            if (c) s_cnt[i] += atomicAdd(&run[i], c);  // cleared before the counting kernel
        }
        __syncthreads();
        for_mine(
                    [&](const ET& e)
                    {
                        const u64 key  = E::key(e);
                        const int slot = atomicAdd(&s_cnt[E::cell(e)], 1);
                        if ((unsigned long long)(unsigned)slot < (unsigned long long)p.capacity)
                            p.keys[slot] = key;
                        else
                            dropped += 1;
                    });
        if (dropped) atomicAdd(&p.status->overflow, (u64)dropped);
        return;
    }
    // The tile's first kStageKeys keys are staged in LDS and copied out with full-line stores; the others of a bigger tile
    // go to their lists directly (8-byte stores scattered over the tile's region).
    extern __shared__ u64 s_keys[];
    const int tile_total = p.bin_start[bin + 1] - key_start;
    const int staged     = (int)max(0ll, min((long long)min(tile_total, kStageKeys), p.capacity - key_start));
    for_mine(
                [&](const ET& e)
                {
                    const u64 key  = E::key(e);
                    const int slot = atomicAdd(&s_cnt[E::cell(e)], 1);
                    if (slot - key_start < staged)
                        s_keys[slot - key_start] = key;
                    else if ((unsigned long long)(unsigned)slot < (unsigned long long)p.capacity)
                        p.keys[slot] = key;
                    else
                        dropped += 1;
                });
    __syncthreads();
    u64* dst = p.keys + key_start;
    for (int i = threadIdx.x; i < staged; i += THREADS) __builtin_nontemporal_store(s_keys[i], dst + i);
    if (dropped) atomicAdd(&p.status->overflow, (u64)dropped);
}

// ---------------------------------------------------------------------------------------------------------
// A pixel's list is the union of the lists of the four cells whose 2 x 2 footprints cover it: (x-1, y-1), (x, y-1),
// (x-1, y), (x, y) (CountAndCollectTiled adds every point to the four pixels of its footprint,
// RenderForward.cu:300-366; here a point is filed once, under its footprint's first pixel, and the pixels gather).
// The K nearest entries of a pixel are among the K nearest of each of its cells, and a cell serves four pixels, so the
// sort (FastSortFusedNew, RenderForward.cu:474-1059) is split:
//   cell_sort_kernel   every cell's list sorted in place, ascending, and cut to its 16 smallest keys: a list of up to
//                      8 keys by one lane (a sorting network over registers), a longer one by a 16-lane DPP row that
//                      streams it in chunks of 16.
//   blend_kernel       a wavefront owns an 8 x 8 block of pixels, one pixel per lane: a pixel merges the (sorted, cut) lists
//                      of its four cells, then the alpha blend front to back (RenderForward.cu:820-1048).
// A pixel's colour is summed in the order of a balanced binary tree over the list positions.
constexpr int kLaneSortMax = 8;   // longest list that a lane sorts with a network
constexpr int kStagedKeys  = 8;   // keys per cell that blend_kernel stages in LDS

// {first key (negative: a long list, whose candidates are in `cand`), readable keys, entries} of a cell
__device__ __forceinline__ int4 cell_info(const ForwardParams& p, int cell)
{
    const int len   = p.counts[cell];
    const int start = p.cursor[cell];  // negative: a long list, reduced to candidates by long_list_reduce_kernel
    // keys actually there: the key storage may have ended inside the list
    const int rd = start < 0 ? ((len + kLongSegment - 1) / kLongSegment) * 16 : (int)max(0ll, min((long long)len, p.capacity - start));
    return make_int4(start, rd, len, 0);
}

// the keys of a cell: in the key array, or the candidate rows that the reduction pass left for a long list
__device__ __forceinline__ u64* cell_keys(const ForwardParams& p, int start)
{
    return start >= 0 ? p.keys + (unsigned)start : p.cand + (size_t)(unsigned)(-1 - start) * 16;
}

// the same for the cell (cx, cy) of the layer of `tc`, its readable keys cut to the kCellKeep that cell_sort_kernel
// left in order (empty outside the layer and in its last row and column, where no footprint starts)
__device__ __forceinline__ int4 load_cell(const ForwardParams& p, const TileCtx& tc, int cx, int cy)
{
    int4 r = make_int4(0, 0, 0, 0);
    if (cx >= 0 && cy >= 0 && cx < tc.w - 1 && cy < tc.h - 1)
    {
        const int bin = tc.bin + ((cx - tc.x0) >> kTileShift) + ((cy - tc.y0) >> kTileShift) * tc.tiles_x;  // shifts round down
        r   = cell_info(p, (bin << (2 * kTileShift)) | ((cy & (kTile - 1)) << kTileShift) | (cx & (kTile - 1)));
        r.y = min(r.y, kCellKeep);
    }
    return r;
}

template <int C>
__device__ __forceinline__ void store_pixel(const ForwardParams& p, float* img, int lw, int lh, int gx, int gy, const float (&col)[C])
{
    // offsets inside one view's image stay far below 2^32 (the pyramid has at most kMaxBins tiles)
    if (p.layout == TRIPS_LAYOUT_CHW)
    {
        const size_t plane = (size_t)lw * lh;
        float* o           = img + ((size_t)p.view_index * C) * plane;
        const unsigned at  = __umul24((unsigned)gy, (unsigned)lw) + (unsigned)gx;
#pragma unroll
        for (int c = 0; c < C; ++c) __builtin_nontemporal_store(col[c], (o + c * plane) + at);
    }
    else
    {
        float* o          = img + ((size_t)p.view_index * lh * lw) * C;
        const unsigned at = (__umul24((unsigned)gy, (unsigned)lw) + (unsigned)gx) * C;
#pragma unroll
        for (int c = 0; c < C; ++c) __builtin_nontemporal_store(col[c], o + at + c);
    }
}

// ---- one list per lane: sorting networks over registers (Batcher's odd-even merge sort; keys are distinct or the
// all-ones filler) ----
__device__ __forceinline__ void sort_pair(u64& a, u64& b)
{
    const bool sw = b < a;
    const u64 lo = sw ? b : a, hi = sw ? a : b;
    a = lo;
    b = hi;
}
__device__ __forceinline__ void lane_sort4(u64 (&k)[kLaneSortMax])
{
    sort_pair(k[0], k[1]), sort_pair(k[2], k[3]);
    sort_pair(k[0], k[2]), sort_pair(k[1], k[3]);
    sort_pair(k[1], k[2]);
}
__device__ __forceinline__ void lane_sort8(u64 (&k)[kLaneSortMax])
{
    sort_pair(k[0], k[1]), sort_pair(k[2], k[3]), sort_pair(k[4], k[5]), sort_pair(k[6], k[7]);
    sort_pair(k[0], k[2]), sort_pair(k[1], k[3]), sort_pair(k[4], k[6]), sort_pair(k[5], k[7]);
    sort_pair(k[1], k[2]), sort_pair(k[5], k[6]);
    sort_pair(k[0], k[4]), sort_pair(k[1], k[5]), sort_pair(k[2], k[6]), sort_pair(k[3], k[7]);
    sort_pair(k[2], k[4]), sort_pair(k[3], k[5]);
    sort_pair(k[1], k[2]), sort_pair(k[3], k[4]), sort_pair(k[5], k[6]);
}
// ascending sort of the first nmax (wave-uniform) of the lane's keys
__device__ __forceinline__ void lane_sort(u64 (&k)[kLaneSortMax], int nmax)
{
    if (nmax > 4)
        lane_sort8(k);
    else if (nmax > 2)
        lane_sort4(k);
    else if (nmax > 1)
        sort_pair(k[0], k[1]);
}
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

// Sum of a sequence in the order of a balanced binary tree over the positions, (0 + 1) + (2 + 3), ...: push<J>(v) for
// J = 0, 1, ..., then total(). A skipped tail counts as zeros.
template <int C, int LEVELS>
struct TreeSum
{
    float acc[LEVELS][C];
    __device__ __forceinline__ TreeSum()
    {
#pragma unroll
        for (int l = 0; l < LEVELS; ++l)
#pragma unroll
            for (int c = 0; c < C; ++c) acc[l][c] = 0.f;
    }
    template <int J>
    __device__ __forceinline__ void push(const float (&v)[C])
    {
        float t[C];
#pragma unroll
        for (int c = 0; c < C; ++c) t[c] = v[c];
#pragma unroll
        for (int l = 0; l < LEVELS; ++l)
        {
            if ((J >> l) & 1)
            {
#pragma unroll
                for (int c = 0; c < C; ++c) t[c] = acc[l][c] + t[c], acc[l][c] = 0.f;
            }
            else
            {
#pragma unroll
                for (int c = 0; c < C; ++c) acc[l][c] = t[c];
                break;
            }
        }
    }
    __device__ __forceinline__ void total(float (&out)[C])
    {
#pragma unroll
        for (int c = 0; c < C; ++c) out[c] = acc[0][c];
#pragma unroll
        for (int l = 1; l < LEVELS; ++l)
#pragma unroll
            for (int c = 0; c < C; ++c) out[c] = acc[l][c] + out[c];
    }
};

// ---------------------------------------------------------------------------------------------------------
__device__ __forceinline__ u64 shfl16(u64 v, int src)
{
    unsigned lo = (unsigned)v, hi = (unsigned)(v >> 32);
    lo = __shfl(lo, src, 16);
    hi = __shfl(hi, src, 16);
    return ((u64)hi << 32) | lo;
}

// The 16 smallest of key_at(0 .. readable - 1) for each of the wavefront's four 16-lane rows, ascending over the row's
// lanes (all-ones where the row has fewer keys). A chunk of 16 further keys is sorted and merged only if one of them
// beats the current 16th; most chunks of a long list are passed over, so the loop runs at the latency of its loads:
// four chunks are requested together and the next four are in flight while these are looked at. The first 16 + 64
// keys can be requested ahead of the call (row_top16_first), e.g. while the rows still work on other lists.
struct RowKeys
{
    u64 k0;              // keys 0..15
    u64 f0, f1, f2, f3;  // keys 16..79
};
template <typename KeyAt>
__device__ __forceinline__ void row_load4(KeyAt&& key_at, int readable, int base, u64& f0, u64& f1, u64& f2, u64& f3)
{
    const int i = base + (int)(threadIdx.x & 15);
    const u64 kInf = ~0ull;
    f0 = i < readable ? key_at(i) : kInf;
    f1 = i + 16 < readable ? key_at(i + 16) : kInf;
    f2 = i + 32 < readable ? key_at(i + 32) : kInf;
    f3 = i + 48 < readable ? key_at(i + 48) : kInf;
}
template <typename KeyAt>
__device__ __forceinline__ RowKeys row_top16_first(KeyAt&& key_at, int readable)
{
    RowKeys r;
    const int sub = threadIdx.x & 15;
    r.k0 = sub < readable ? key_at(sub) : ~0ull;
    row_load4(key_at, readable, 16, r.f0, r.f1, r.f2, r.f3);
    return r;
}
template <typename KeyAt>
__device__ __forceinline__ u64 row_top16(KeyAt&& key_at, int readable, const RowKeys& first)
{
    const int lane = threadIdx.x & 63;
    const int grp  = lane >> 4;
    int maxlen = readable;
    maxlen     = max(maxlen, __shfl_xor(maxlen, 16));
    maxlen     = max(maxlen, __shfl_xor(maxlen, 32));
    const u64 grp_mask = 0xFFFFull << (grp * 16);
    maxlen             = __builtin_amdgcn_readfirstlane(maxlen);
    u64 best = row_sort16(first.k0);
    auto consider = [&](u64 k)
    {
        const u64 worst = shfl16(best, 15);
        const bool need = k < worst;
        if (__ballot(need) & grp_mask)
        {
            k           = row_sort16(k);
            const u64 r = row_xor_u64<15>(k);  // reversed: lane i sees the (15-i)-th smallest new key
            best        = best < r ? best : r;
            best        = row_merge16(best);
        }
    };
    if (maxlen > 16)
    {
        u64 c0 = first.f0, c1 = first.f1, c2 = first.f2, c3 = first.f3;
        u64 n0 = c0, n1 = c1, n2 = c2, n3 = c3;
        for (int base = 16; base < maxlen; base += 64)
        {
            if (base + 64 < maxlen) row_load4(key_at, readable, base + 64, n0, n1, n2, n3);
            consider(c0);
            if (base + 16 < maxlen) consider(c1);
            if (base + 32 < maxlen) consider(c2);
            if (base + 48 < maxlen) consider(c3);
            c0 = n0, c1 = n1, c2 = n2, c3 = n3;
        }
    }
    return best;
}
template <typename KeyAt>
__device__ __forceinline__ u64 row_top16(KeyAt&& key_at, int readable)
{
    return row_top16(key_at, readable, row_top16_first(key_at, readable));
}

// Reduction pass over the segments of long lists (tile_lists_kernel hands them out): a 16-lane row keeps the 16
// smallest keys of a segment. Persistent workgroups, the four rows of a wavefront take consecutive segments.
__global__ __launch_bounds__(256) void long_list_reduce_kernel(const ForwardParams p)
{
    const int n    = min(*p.long_count, p.max_long_items);
    const int lane = threadIdx.x & 63;
    const int rows = gridDim.x * 16;
    for (int first = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 4; first < n; first += rows)
    {
        const int item = first + (lane >> 4);
        int2 seg       = make_int2(0, 0);
        if (item < n) seg = p.long_items[item];
        if (seg.x < 0 || seg.y < 0 || seg.y > kLongSegment || (long long)seg.x + seg.y > p.capacity) seg = make_int2(0, 0);
        const u64* src = p.keys + seg.x;
        const u64 best = row_top16([&](int i) { return src[i]; }, seg.y);
        if (item < n) p.cand[(size_t)item * 16 + (lane & 15)] = best;
    }
}

// Every cell's list in ascending order, in place; of a list longer than kCellKeep its kCellKeep smallest keys, at its
// start. A workgroup takes 64 consecutive cells (their lists follow each other in the key array); the sixteen
// workgroups of a tile run on the XCD that blends the tile. The first wavefront sorts the lists of up to kLaneSortMax
// keys, one cell per lane, with a network; the longer lists are taken, one after the other, by whichever of the
// sixteen 16-lane rows of the workgroup's four wavefronts is free, and streamed (a wavefront that kept all 64 cells to
// itself walked up to 64 long lists one after the other, four at a time: in a crowded tile that chain of memory round
// trips was the kernel's duration). The other three wavefronts start on the long lists while the first sorts the
// short ones.
__global__ __launch_bounds__(256) void cell_sort_kernel(const ForwardParams p)
{
    __shared__ int s_start[64], s_rd[64];
    __shared__ unsigned char s_long[64];  // lanes of the cells with a longer list
    __shared__ int s_num_long, s_next;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int NB   = p.geom.bin_off[p.num_layers];
    const bool coarse_first = *p.coarse_first != 0;
    long long lblock        = xcd_tile_block(blockIdx.x, 16);
    if (lblock >= (long long)NB * 16) return;
    if (coarse_first) lblock = (long long)NB * 16 - 1 - lblock;
    int4 info = make_int4(0, 0, 0, 0);
    if (wave == 0)
    {
        const int cell = (int)lblock * 64 + lane;
        info           = cell_info(p, cell);
        const int rd   = info.y;
        const u64 longer = __ballot(rd > kLaneSortMax);
        s_start[lane] = info.x, s_rd[lane] = rd;
        if (rd > kLaneSortMax) s_long[__popcll(longer & ((1ull << lane) - 1ull))] = (unsigned char)lane;
        if (lane == 0) s_num_long = (int)__popcll(longer), s_next = 0;
    }
    __syncthreads();
    // ---- up to kLaneSortMax keys: one cell per lane of the first wavefront, while the other wavefronts start on the
    // longer lists ----
    if (wave == 0)
    {
        const int rd    = info.y;
        u64* const base = cell_keys(p, info.x);
        const int mine = rd <= kLaneSortMax ? rd : 0;
        const int nmax = wave_max_small<kLaneSortMax>(mine);
        if (nmax > 1)
        {
            u64 k[kLaneSortMax];
#pragma unroll
            for (int i = 0; i < kLaneSortMax; ++i)
            {
                k[i] = ~0ull;
                if (i < nmax && i < mine) k[i] = base[i];
            }
            lane_sort(k, nmax);
            if (mine > 1)
            {
#pragma unroll
                for (int i = 0; i < kLaneSortMax; ++i)
                    if (i < nmax && i < mine) base[i] = k[i];
            }
        }
    }
    // ---- longer lists: one cell per 16-lane row; a row takes the next list that nobody has taken yet (the first
    // wavefront's rows join when its short lists are done), and the first keys of a row's next list are requested
    // before it works on this one ----
    const int num_long = s_num_long;
    if (num_long == 0) return;
    const int sub = lane & 15;
    struct Pass
    {
        u64* base;
        int readable;
        RowKeys first;
    };
    auto take = [&]()
    {
        int index = 0;
        if (sub == 0) index = atomicAdd(&s_next, 1);
        return __shfl(index, lane & ~15);
    };
    auto pass_of = [&](int index)
    {
        Pass ps;
        const bool has = index < num_long;
        const int src  = has ? (int)s_long[index] : 0;
        ps.base        = cell_keys(p, s_start[src]);
        ps.readable    = has ? s_rd[src] : 0;
        u64* const rb  = ps.base;
        ps.first       = row_top16_first([&](int i) { return rb[i]; }, ps.readable);
        return ps;
    };
    int index = take();
    Pass cur  = pass_of(index);
    // (the rows of a wavefront walk in step: until none of them has a list)
    while (__ballot(index < num_long) != 0ull)
    {
        const int next_index = take();
        Pass nxt             = pass_of(next_index);
        u64* const rb  = cur.base;
        const u64 best = row_top16([&](int i) { return rb[i]; }, cur.readable, cur.first);
        if (sub < min(cur.readable, kCellKeep)) rb[sub] = best;
        cur   = nxt;
        index = next_index;
    }
}

// One pixel per lane, 8 x 8 pixels per wavefront, a quarter of a tile per workgroup (the four of a tile on one XCD).
// A wavefront stages the first kStagedKeys keys of its 9 x 9 sorted cell lists in LDS, each lane one cell's, and a pixel
// merges its four: the smallest of the four heads is the next list position, and the list that gave it moves on. The
// records of BATCH positions are requested as the merge finds them, then those positions are blended.
// What bounds it: vector instructions where neighbouring lanes share the records' lines, the gathers of the records where
// points are in no order. Every key is thus read once per wavefront instead of by up to four pixels, and no lane waits for
// another's way of sorting (pixels of up to eight keys used to sort them with a network, the others to merge behind a staging
// loop that waited for memory eleven times): 1920 x 1080, without / with the saved state, 6M points in Morton order 107 ->
// 91 us, 9M 134 -> 120, 1M in a ball 99 -> 89; 6M in no order 191 -> 191. A position's saved list leaves as soon as four are
// known: with all sixteen kept the kernel took 140 registers of a lane, and a fourth wavefront per SIMD is worth 4 %.
// What it costs: the requests lie a merge step apart, and a fourth wavefront shares the L1, so neighbouring pixels' requests of
// a line meet there less often than when eight positions were requested in a row: at 6M points in no order 10.1 M reads of the
// L2 instead of 7.7 M and 769 MB of memory instead of 663. All four of a group requested behind their merge: 8.6 M, 743 MB
// and 182 us; three wavefronts: 9.5 M, 733 MB, 197 us; both: 8.3 M, 717 MB, 193 us. (The former takes registers that cost the
// instances for 3 and 6 channels without the saved state and for 8 with it a wavefront, 1 to 3 % of a whole pass.)
template <int C, bool TRAIN>
__global__ __launch_bounds__(256) void blend_kernel(const ForwardParams p)
{
    constexpr int CPAD = (C + 3) & ~3;
    constexpr int RF   = 4 + CPAD;  // floats per blend record
    constexpr int NQ   = CPAD / 4;
    constexpr int BATCH = CPAD <= 8 ? 8 : 4;  // list positions whose records are requested together
    constexpr int CELLS = 81;
    __shared__ int s_start[4][CELLS];               // as cell_info's
    __shared__ unsigned s_info[4][CELLS];           // readable keys, at most kCellKeep, in bits 0..4; entries above
    __shared__ u64 s_keys[4][kStagedKeys * CELLS];  // [key][cell], all-ones past a list's end
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int NB   = p.geom.bin_off[p.num_layers];
    const bool coarse_first = *p.coarse_first != 0;
    long long lblock        = xcd_tile_block(blockIdx.x, 4);
    if (lblock >= (long long)NB * 4) return;
    if (coarse_first) lblock = (long long)NB * 4 - 1 - lblock;
    const int bin = (int)(lblock >> 2), quarter = (int)(lblock & 3);
    const TileCtx tc = tile_ctx(p.geom, bin);
    const int bx = ((quarter & 1) << 4) + ((wave & 1) << 3), by = ((quarter >> 1) << 4) + ((wave >> 1) << 3);
    const int lx = lane & 7, ly = lane >> 3;
    const int pix = (bin << (2 * kTileShift)) | ((by + ly) << kTileShift) | (bx + lx);
    const int gx = tc.x0 + bx + lx, gy = tc.y0 + by + ly;
    const bool live = gx < tc.w && gy < tc.h;  // false for the padding of partial tiles
    if (tc.x0 + bx >= tc.w || tc.y0 + by >= tc.h)
    {
        // a block of padding: its rows of the saved tables are defined as empty
        if (TRAIN) __builtin_nontemporal_store(0, p.retained + pix);
        return;
    }

    // The block gathers from the 9 x 9 cells (gx0 - 1 .. gx0 + 7) x (gy0 - 1 .. gy0 + 7): one cell per lane, then
    // the 17 that are left; a pixel takes its four from LDS.
    {
        const int i1 = lane, i2 = min(64 + lane, CELLS - 1);
        const int4 a1 = load_cell(p, tc, tc.x0 + bx - 1 + i1 % 9, tc.y0 + by - 1 + i1 / 9);
        const int4 a2 = load_cell(p, tc, tc.x0 + bx - 1 + i2 % 9, tc.y0 + by - 1 + i2 / 9);
        // (the sum of a pixel's four lengths saturates at kMaxExportedLength: so may each of them)
        s_start[wave][i1] = a1.x;
        s_info[wave][i1]  = (unsigned)a1.y | ((unsigned)min(a1.z, kMaxExportedLength) << 5);
        if (64 + lane < CELLS)
        {
            s_start[wave][i2] = a2.x;
            s_info[wave][i2]  = (unsigned)a2.y | ((unsigned)min(a2.z, kMaxExportedLength) << 5);
        }
        // Keys and, in the place after the last of a shorter list, all-ones. Every key is requested before the first is
        // stored.
        const int r1 = min(a1.y, kStagedKeys), r2 = 64 + lane < CELLS ? min(a2.y, kStagedKeys) : 0;
        const int qmax1 = wave_max_small<kStagedKeys>(r1), qmax2 = wave_max_small<kStagedKeys>(r2);
        const u64* const k1 = cell_keys(p, a1.x);
        const u64* const k2 = cell_keys(p, a2.x);
        u64 v1[kStagedKeys], v2[kStagedKeys];
#pragma unroll
        for (int q = 0; q < kStagedKeys; ++q)
        {
            v1[q] = ~0ull;
            if (q < qmax1 && q < r1) v1[q] = k1[q];
        }
#pragma unroll
        for (int q = 0; q < kStagedKeys; ++q)
        {
            v2[q] = ~0ull;
            if (q < qmax2 && q < r2) v2[q] = k2[q];
        }
#pragma unroll
        for (int q = 0; q < kStagedKeys; ++q)
            if (q <= qmax1) s_keys[wave][q * CELLS + i1] = v1[q];
#pragma unroll
        for (int q = 0; q < kStagedKeys; ++q)
            if (q <= qmax2 && 64 + lane < CELLS) s_keys[wave][q * CELLS + i2] = v2[q];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int ci0 = ly * 9 + lx;  // the pixel's cells: ci0, ci0 + 1, ci0 + 9, ci0 + 10
    int total = 0, length = 0;
    {
        const unsigned a = s_info[wave][ci0], b = s_info[wave][ci0 + 1], c = s_info[wave][ci0 + 9], d = s_info[wave][ci0 + 10];
        total  = live ? (int)((a & 31u) + (b & 31u) + (c & 31u) + (d & 31u)) : 0;  // keys to choose from
        length = (int)((a >> 5) + (b >> 5) + (c >> 5) + (d >> 5));                 // entries (0 for padding: its cells are empty)
    }
    const int n    = min(total, p.list_depth);  // list positions that hold an entry
    const int nmax = wave_max_small<16>(n);     // longest list of the block

    unsigned id[4];  // compact numbers of four entries, nearest first (positions past n hold anything)
    // where each entry came from, for the backward: which of the pixel's four cells (bits 4..5) and its place in that
    // cell's sorted list (bits 0..3); one byte per list position, four positions per word
    unsigned tagw[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int j = 0; j < 4; ++j) id[j] = ~0u;
    const u64* const keys = s_keys[wave] + ci0;
    u64 h0 = keys[0], h1 = keys[1], h2 = keys[9], h3 = keys[10];
    unsigned heads = 0x01010101u;  // a byte per list: place of the key after its head

    // ---- blend (RenderForward.cu:820-1048), front to back ----
    TreeSum<C, 5> sum;  // (five levels: up to 16 positions)
    float T       = 1.f;
    float bgw     = 1.f;  // empty list -> 1
    int ret       = 0;    // length of the leading run of kept entries
    bool run_open = true;
    float4 r0[BATCH], rd[BATCH][NQ];
    // The next list position, its number a compile-time constant (the arrays indexed by it stay in registers): the smallest
    // head, and the next key of the list that gave it. A lane whose list ends before walks on over what it finds.
    auto merge = [&](auto jc)
    {
        constexpr int j = decltype(jc)::value;
        const bool b01 = h1 < h0, b23 = h3 < h2;
        const u64 m01 = b01 ? h1 : h0, m23 = b23 ? h3 : h2;
        const bool hi = m23 < m01;
        id[j % 4]     = (unsigned)(hi ? m23 : m01);
        if (j < n)
        {
            const float4* rec = reinterpret_cast<const float4*>(p.rec + (size_t)id[j % 4] * RF);
            r0[j % BATCH]     = rec[0];
#pragma unroll
            for (int q = 0; q < NQ; ++q) rd[j % BATCH][q] = rec[1 + q];
        }
        const unsigned shift = hi ? (b23 ? 24u : 16u) : (b01 ? 8u : 0u);  // 8 x the list that gave the key
        const unsigned place = (heads >> shift) & 0xFFu;
        if (TRAIN) tagw[j / 4] |= ((shift << 1) | (place - 1u)) << (8 * (j & 3));
        heads += 1u << shift;
        if (j == 15) return;
        const unsigned cell = (0x0A090100u >> shift) & 0xFFu;  // of the list, from ci0
        u64 next            = keys[__umul24(min(place, (unsigned)kStagedKeys - 1u), (unsigned)CELLS) + cell];
        const bool further  = place >= (unsigned)kStagedKeys;
        if (__ballot(further && j + 1 < n))  // keys that are not staged (few: of one list past its eighth)
        {
            if (further)
            {
                next           = ~0ull;
                const int from = s_start[wave][ci0 + (int)cell];
                if (place < (s_info[wave][ci0 + (int)cell] & 31u)) next = cell_keys(p, from)[place];
            }
        }
        const bool w0 = !hi && !b01, w1 = !hi && b01, w2 = hi && !b23, w3 = hi && b23;
        h0 = w0 ? next : h0, h1 = w1 ? next : h1, h2 = w2 ? next : h2, h3 = w3 ? next : h3;
    };
    auto position = [&](auto jc)
    {
        constexpr int j = decltype(jc)::value;
        constexpr int b = j % BATCH;
        const bool has  = j < n;  // (otherwise the records of the position hold anything)
        float a         = 0.f;
        if (has) a = entry_alpha(r0[b], tc.layer, p.num_layers, gx, gy);
        const float Tc  = (T >= kAlphaDestCutoff) ? T : 0.f;
        const bool kept = has && Tc >= kAlphaDestCutoff;
        run_open        = run_open && kept;
        if (run_open) ret = j + 1;
        const float wgt = Tc * a;
        float pr[C];
#pragma unroll
        for (int c = 0; c < C; ++c)
        {
            const float4 t = rd[b][c / 4];
            const float d  = (c & 3) == 0 ? t.x : (c & 3) == 1 ? t.y : (c & 3) == 2 ? t.z : t.w;
            pr[c]          = has ? wgt * d : 0.f;
        }
        sum.template push<j>(pr);
        // background weight (RenderForward.cu:1002-1022): taken at the last list position
        if (j == n - 1) bgw = (p.background_mode == TRIPS_BG_REFERENCE) ? Tc : T * (1.f - a);
        T = T * (1.f - a);
    };
    // four positions found and their records requested; the saved list holds four positions of the block's 64 pixels side by
    // side (list_word)
    auto merge4 = [&](auto first)
    {
        constexpr int j0 = decltype(first)::value;
        if (j0 + 0 < nmax) merge(std::integral_constant<int, j0 + 0>{});
        if (j0 + 1 < nmax) merge(std::integral_constant<int, j0 + 1>{});
        if (j0 + 2 < nmax) merge(std::integral_constant<int, j0 + 2>{});
        if (j0 + 3 < nmax) merge(std::integral_constant<int, j0 + 3>{});
        if (TRAIN && j0 < nmax && j0 < n)
            __builtin_nontemporal_store(vi4{(int)id[0], (int)id[1], (int)id[2], (int)id[3]},
                                        reinterpret_cast<vi4*>(p.lists + list_word((unsigned)pix, j0, p.list_depth)));
    };
    // BATCH positions: found, their records requested, then blended
    auto batch = [&](auto first)
    {
        constexpr int j0 = decltype(first)::value;
        merge4(std::integral_constant<int, j0>{});
        if constexpr (BATCH > 4) merge4(std::integral_constant<int, j0 + 4>{});
        if (j0 + 0 < nmax) position(std::integral_constant<int, j0 + 0>{});
        if (j0 + 1 < nmax) position(std::integral_constant<int, j0 + 1>{});
        if (j0 + 2 < nmax) position(std::integral_constant<int, j0 + 2>{});
        if (j0 + 3 < nmax) position(std::integral_constant<int, j0 + 3>{});
        if constexpr (BATCH > 4)
        {
            if (j0 + 4 < nmax) position(std::integral_constant<int, j0 + 4>{});
            if (j0 + 5 < nmax) position(std::integral_constant<int, j0 + 5>{});
            if (j0 + 6 < nmax) position(std::integral_constant<int, j0 + 6>{});
            if (j0 + 7 < nmax) position(std::integral_constant<int, j0 + 7>{});
        }
    };
    if (nmax > 0) batch(std::integral_constant<int, 0>{});
    if constexpr (BATCH == 4)
    {
        if (nmax > 4) batch(std::integral_constant<int, 4>{});
        if (nmax > 8) batch(std::integral_constant<int, 8>{});
        if (nmax > 12) batch(std::integral_constant<int, 12>{});
    }
    else if (nmax > 8)
        batch(std::integral_constant<int, 8>{});

    float col[C];
    sum.total(col);
    if (live)
    {
        if (bgw >= kAlphaDestCutoff)
        {
#pragma unroll
            for (int c = 0; c < C; ++c) col[c] += p.background[c] * (bgw * 1.f);
        }
        store_pixel<C>(p, p.image[tc.layer], tc.w, tc.h, gx, gy, col);
    }
    // saved state, also for padding pixels (empty) so that every row of the tables is defined
    if (TRAIN)
    {
        // (bits 0..4: retained entries; bits 5..9: list positions that hold an id. Only those are stored below: the
        // backward reads the retained ones, the export fills the rest of a row with -1 itself. Bits 10..31: length of
        // the pixel's list before the cut to K, for the export; saturates.)
        __builtin_nontemporal_store(live ? (int)((unsigned)ret | ((unsigned)n << kRetainedBits) |
                                                 ((unsigned)min(length, kMaxExportedLength) << (2 * kRetainedBits)))
                                         : 0,
                                    p.retained + pix);
        if (n > 0) __builtin_nontemporal_store(vu4{tagw[0], tagw[1], tagw[2], tagw[3]}, reinterpret_cast<vu4*>(p.tags) + (unsigned)pix);
        // the view's retained entries, for the backward's choice of how it keeps its pair rows: estimated from every
        // kRetainedSample-th workgroup, one atomic per wavefront (the sum of 64 values of at most 16, a ballot per bit),
        // spread over kRetainedParts counters
        unsigned wave_ret = 0;
        if (blockIdx.x % (unsigned)kRetainedSample == 0)
        {
#pragma unroll
            for (int b = 0; b < 5; ++b) wave_ret += (unsigned)__popcll(__ballot(live && ((ret >> b) & 1))) << b;
        }
        if (lane == 0 && wave_ret)
            atomicAdd(p.saved_chunk_valid + p.bin_groups + (int)((blockIdx.x / (unsigned)kRetainedSample * 4u + (unsigned)wave) % (unsigned)kRetainedParts), (int)wave_ret);
    }
}

// ---------------------------------------------------------------------------------------------------------
// host-side launchers
#define TRIPS_DISPATCH_C(C_, ...)             \
    switch (C_)                               \
    {                                         \
        case 3: { constexpr int CC = 3; __VA_ARGS__; break; }   \
        case 4: { constexpr int CC = 4; __VA_ARGS__; break; }   \
        case 6: { constexpr int CC = 6; __VA_ARGS__; break; }   \
        case 8: { constexpr int CC = 8; __VA_ARGS__; break; }   \
        case 16: { constexpr int CC = 16; __VA_ARGS__; break; } \
        default: return hipErrorInvalidValue; \
    }

hipError_t launch_forward_view(const ForwardParams& p, int channels, bool train, bool first_view, hipStream_t stream,
                               Profiler* prof)
{
    const int NB = p.geom.bin_off[p.num_layers];

    const int G           = p.bin_groups;
    const size_t lds_hist = (size_t)NB * sizeof(int);
    // compact point numbers are below num_points: entries of 8 bytes when they fit kPackedIdBits bits
    const bool packed = p.num_points <= (1 << kPackedIdBits);
    {
        ProfScope ps(prof, "project_bin", stream);
        if (train)
        {
            TRIPS_DISPATCH_C(channels, hipLaunchKernelGGL((project_bin_kernel<CC, true>), dim3(G), dim3(kBinThreads), lds_hist, stream, p));
        }
        else
        {
            TRIPS_DISPATCH_C(channels, hipLaunchKernelGGL((project_bin_kernel<CC, false>), dim3(G), dim3(kBinThreads), lds_hist, stream, p));
        }
    }
    {
        ProfScope ps(prof, "bin_scan", stream);
        hipLaunchKernelGGL(bin_column_scan_kernel, dim3((NB + kScanCols - 1) / kScanCols + 1), dim3(256), 0, stream, p, first_view ? 1 : 0);
    }
    {
        ProfScope ps(prof, "bin_scatter", stream);
        if (packed)
            hipLaunchKernelGGL(bin_scatter_kernel<true>, dim3(G), dim3(kBinThreads), lds_hist, stream, p);
        else
            hipLaunchKernelGGL(bin_scatter_kernel<false>, dim3(G), dim3(kBinThreads), lds_hist, stream, p);
    }
    // workgroups for the slices of split tiles: at most capacity / kSliceEntries full slices plus one partial slice
    // per split tile
    const int max_slices = (int)std::min<long long>(2 * (p.capacity / kSliceEntries) + 1, 1 << 20);
    const int list_blocks = (NB + kNumXcd - 1) / kNumXcd * kNumXcd + (max_slices + 63) / 64 * 64;  // (whole runs of eight on eight XCDs)
    {
        ProfScope ps(prof, "tile_count", stream);
        if (packed)
            hipLaunchKernelGGL((tile_lists_kernel<false, 256, true>), dim3(list_blocks), dim3(256), 0, stream, p);
        else
            hipLaunchKernelGGL((tile_lists_kernel<false, 256, false>), dim3(list_blocks), dim3(256), 0, stream, p);
    }
    {
        ProfScope ps(prof, "tile_scatter", stream);
        constexpr size_t lds = kStageKeys * sizeof(u64);
        if (packed)
            hipLaunchKernelGGL((tile_lists_kernel<true, kScatterThreads, true>), dim3(list_blocks), dim3(kScatterThreads), lds, stream, p);
        else
            hipLaunchKernelGGL((tile_lists_kernel<true, kScatterThreads, false>), dim3(list_blocks), dim3(kScatterThreads), lds, stream, p);
    }
    {
        ProfScope ps(prof, "long_lists", stream);
        const int blocks = std::min((p.max_long_items + 15) / 16, 2048);
        hipLaunchKernelGGL(long_list_reduce_kernel, dim3(blocks), dim3(256), 0, stream, p);
    }
    const long long tiles8 = (((long long)NB + kNumXcd - 1) / kNumXcd) * kNumXcd;  // tiles rounded up to 8
    const int quarter_tiles = (int)(tiles8 * 4);                                   // a quarter tile per workgroup
    {
        ProfScope ps(prof, "cell_sort", stream);
        hipLaunchKernelGGL(cell_sort_kernel, dim3((unsigned)(tiles8 * 16)), dim3(256), 0, stream, p);  // 64 cells per workgroup
    }
    {
        ProfScope ps(prof, "blend", stream);
        if (train)
        {
            TRIPS_DISPATCH_C(channels, hipLaunchKernelGGL((blend_kernel<CC, true>), dim3(quarter_tiles), dim3(256), 0, stream, p));
        }
        else
        {
            TRIPS_DISPATCH_C(channels, hipLaunchKernelGGL((blend_kernel<CC, false>), dim3(quarter_tiles), dim3(256), 0, stream, p));
        }
    }
    return hipGetLastError();
}

}  // namespace trips
