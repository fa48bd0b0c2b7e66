// Fused multi-tensor Adam, pose update, and the small export / reduction kernels of the C ABI (gfx950).
//
//   adam_fused_kernel    <- adam_step      src/lib/models/MyAdam.cu:41-88 (one launch for all tensors instead of
//                                          one 128-thread launch per tensor, :226-288)
//   adam_points_kernel   <- the same step for the four tensors of a point cloud, optimiser state packed per point
//   apply_tangent_kernel <- ApplyTangent   src/lib/rendering/PointRenderer.cu:1428-1447
#include <float.h>

#include "splat_internal.h"
#include "trips_math.h"

#pragma clang fp contract(off)

namespace trips
{
constexpr int kAdamMaxTensors = 16;
constexpr int kAdamPerBlock   = 1024;  // 256 threads x 4 consecutive elements

struct AdamTable
{
    TripsAdamTensor t[kAdamMaxTensors];
    long long block_start[kAdamMaxTensors + 1];
    int32_t vec_ok[kAdamMaxTensors];
    int32_t n;
};

// What an optimiser step reads and writes passes through once: non-temporal accesses (16 bytes or a scalar each) keep it from
// displacing, and from waiting for the displacement of, what the caches hold.
typedef unsigned vu4 __attribute__((ext_vector_type(4)));
template <typename T>
__device__ __forceinline__ T nt_load(const T* a)
{
    if constexpr (sizeof(T) == 16)
        return __builtin_bit_cast(T, __builtin_nontemporal_load(reinterpret_cast<const vu4*>(a)));
    else
        return __builtin_nontemporal_load(a);
}
template <typename T>
__device__ __forceinline__ void nt_store(const T& v, T* a)
{
    if constexpr (sizeof(T) == 16)
        __builtin_nontemporal_store(__builtin_bit_cast(vu4, v), reinterpret_cast<vu4*>(a));
    else
        __builtin_nontemporal_store(v, a);
}

struct AdamScalars
{
    float lr, beta1, beta2, eps, rel_wd, abs_wd, clip, lo, hi, loss_scale;
};

// beta1^t and beta2^t for a step count t: by squaring in double precision, rounded to float once. (The library powf is some
// 400 instructions, and two of them per point were half of the packed kernel's work. The squarings' error doubles per
// squaring from 2^-53: below a float's for any t < 2^28, and beta^t of a beta < 1 is zero long before that.) The loop runs
// until the largest count of the wavefront is done: its squares are the same for every lane.
__device__ __forceinline__ void pow_steps(float beta1, float beta2, uint32_t t, float& p1, float& p2)
{
    double r1 = 1.0, r2 = 1.0, b1 = (double)beta1, b2 = (double)beta2;
    while (__ballot(t != 0u))
    {
        const double n1 = r1 * b1, n2 = r2 * b2;
        const bool bit  = (t & 1u) != 0u;
        r1 = bit ? n1 : r1;
        r2 = bit ? n2 : r2;
        b1 *= b1;
        b2 *= b2;
        t >>= 1;
    }
    p1 = (float)r1;
    p2 = (float)r2;
}

// learning rate with the bias correction of step `current_step` (MyAdam.cu:66-68)
__device__ __forceinline__ float adam_corrected_lr(const AdamScalars& h, uint32_t current_step)
{
    float p1, p2;
    pow_steps(h.beta1, h.beta2, current_step, p1, p2);
    float learning_rate = h.lr;
    learning_rate *= sqrtf(1 - p2) / (1 - p1);
    return learning_rate;
}

// What the elements of a step with one corrected learning rate share.
struct AdamRate
{
    float lr, decay, ab;
};
__device__ __forceinline__ AdamRate adam_rate(const AdamScalars& h, float learning_rate)
{
    const float rel = h.rel_wd * learning_rate;
    return AdamRate{learning_rate, 1 - rel, h.abs_wd * learning_rate};
}

// One element with a gradient (after the loss scale): moments and weight.
__device__ __forceinline__ void adam_update(const AdamScalars& h, const AdamRate& r, float gradient, float& w, float& m, float& v)
{
    const float gradient_sq   = gradient * gradient;
    const float first_moment  = h.beta1 * m + (1 - h.beta1) * gradient;
    const float second_moment = h.beta2 * v + (1 - h.beta2) * gradient_sq;
    m                         = first_moment;
    v                         = second_moment;
    const float effective_learning_rate = fminf(fmaxf(r.lr / (sqrtf(second_moment) + h.eps), h.lo), h.hi);
    const float decayed_weight          = r.decay * w - copysignf(r.ab, w);
    float nw                            = decayed_weight - effective_learning_rate * first_moment;
    if (h.clip != 0.0f)
    {
        const float lo = -h.clip, hi = h.clip;
        nw = nw < lo ? lo : (hi < nw ? hi : nw);
    }
    w = nw;
}

// The gradients divided by the loss scale. A division by 1 changes nothing: skipped, in a branch of its own (the asm keeps
// the compiler from working the divisions out in any case and choosing afterwards, a dozen instructions per element).
template <int E>
__device__ __forceinline__ void adam_unscale(float loss_scale, float (&g)[E])
{
    if (loss_scale != 1.f)
    {
        asm volatile("");
#pragma unroll
        for (int e = 0; e < E; ++e) g[e] = g[e] / loss_scale;
    }
}

// STEP = long long (the reference's state tensor) or int
template <typename STEP>
__device__ __forceinline__ void adam_block(const AdamTable& tab, int ti)
{
    const TripsAdamTensor& T = tab.t[ti];
    const AdamScalars h      = {T.lr, T.beta1, T.beta2, T.eps, T.relative_weight_decay, T.absolute_weight_decay,
                                T.weight_clipping_magnitude, T.lower_lr_bound, T.upper_lr_bound, T.loss_scale};
    const long long i0 = ((long long)blockIdx.x - tab.block_start[ti]) * kAdamPerBlock + (long long)threadIdx.x * 4;
    if (i0 >= T.n) return;
    float* mo = T.first_moment;
    float* vo = T.second_moment;
    STEP* st  = reinterpret_cast<STEP*>(T.steps);

    if (T.dtype == TRIPS_DTYPE_F32 && tab.vec_ok[ti] && i0 + 4 <= T.n)
    {
        float* w       = reinterpret_cast<float*>(T.weights);
        const float* g = reinterpret_cast<const float*>(T.grads);
        const float4 g4 = nt_load(reinterpret_cast<const float4*>(g + i0));
        float ge[4]     = {g4.x, g4.y, g4.z, g4.w};
        adam_unscale(h.loss_scale, ge);
        // (A parameter not seen in this step stays as it is, MyAdam.cu:57-61.) Four lanes share a piece of 64 bytes, the unit
        // that memory transfers, of every float array: they skip it together or write all of it, unseen elements as they were
        // read, so that nothing smaller leaves. 10M elements with 64-bit counters (1M points), us:
        //                                       other buffers between two steps      a loop over the same 240 MB
        //   share of points with a gradient         5 %   61 %    all                 5 %   61 %    all
        //   lane by lane, ordinary accesses          57    101     89                  39     75     76
        //   lines of 128 bytes, non-temporal         53     80     80                  54     81     81
        //   pieces of 64 bytes, non-temporal         46     79     80                  46     80     81
        // In a step with anything else in it the state is not in the caches when its turn comes; what fits the last-level
        // cache and is stepped over and over is better off with ordinary accesses (64-bit counters, 61 %, pieces either way:
        // 300k points 22 and 24 us, with other buffers in between 35 and 29). Whole splat steps of 20k to 300k points take the
        // same time with both, of 1M 484 us instead of 501.
        const bool some             = !(ge[0] == 0.f && ge[1] == 0.f && ge[2] == 0.f && ge[3] == 0.f);
        const unsigned long long by = __ballot(some);
        if (((by >> (threadIdx.x & 60u)) & 0xFull) == 0) return;
        const float4 w4 = nt_load(reinterpret_cast<const float4*>(w + i0));
        const float4 m4 = nt_load(reinterpret_cast<const float4*>(mo + i0));
        const float4 v4 = nt_load(reinterpret_cast<const float4*>(vo + i0));
        STEP s[4];
        if (sizeof(STEP) == 8)
        {
            *reinterpret_cast<longlong2*>(&s[0]) = nt_load(reinterpret_cast<const longlong2*>(st + i0));
            *reinterpret_cast<longlong2*>(&s[2]) = nt_load(reinterpret_cast<const longlong2*>(st + i0 + 2));
        }
        else
            *reinterpret_cast<int4*>(&s[0]) = nt_load(reinterpret_cast<const int4*>(st + i0));
        // The four elements are mostly updated together, so their counters agree: the bias correction (two powers, a square
        // root, a division) of the run's largest counter is computed once and taken by every element whose new counter
        // equals it.
        const uint32_t top   = (uint32_t)max(max(s[0], s[1]), max(s[2], s[3])) + 1u;
        const AdamRate top_r = adam_rate(h, adam_corrected_lr(h, top));
        float we[4] = {w4.x, w4.y, w4.z, w4.w}, me[4] = {m4.x, m4.y, m4.z, m4.w}, ve[4] = {v4.x, v4.y, v4.z, v4.w};
        bool others = false;  // some element with a gradient has another counter
#pragma unroll
        for (int k = 0; k < 4; ++k) others = others || (ge[k] != 0.f && (uint32_t)s[k] + 1u != top);
        const bool any_others = __ballot(others) != 0ull;
#pragma unroll
        for (int k = 0; k < 4; ++k)
        {
            const bool seen = ge[k] != 0.f;
            AdamRate r      = top_r;
            if (any_others)  // (skipped by the whole wavefront in the usual case)
            {
                asm volatile("");
                const uint32_t own = (uint32_t)s[k] + 1u;
                if (seen && own != top) r = adam_rate(h, adam_corrected_lr(h, own));
            }
            float nw = we[k], nm = me[k], nv = ve[k];
            adam_update(h, r, ge[k], nw, nm, nv);
            we[k] = seen ? nw : we[k];
            me[k] = seen ? nm : me[k];
            ve[k] = seen ? nv : ve[k];
            s[k]  = (STEP)((long long)s[k] + (seen ? 1 : 0));
        }
        nt_store(make_float4(we[0], we[1], we[2], we[3]), reinterpret_cast<float4*>(w + i0));
        nt_store(make_float4(me[0], me[1], me[2], me[3]), reinterpret_cast<float4*>(mo + i0));
        nt_store(make_float4(ve[0], ve[1], ve[2], ve[3]), reinterpret_cast<float4*>(vo + i0));
        if (sizeof(STEP) == 8)
        {
            nt_store(*reinterpret_cast<longlong2*>(&s[0]), reinterpret_cast<longlong2*>(st + i0));
            nt_store(*reinterpret_cast<longlong2*>(&s[2]), reinterpret_cast<longlong2*>(st + i0 + 2));
        }
        else
            nt_store(*reinterpret_cast<int4*>(&s[0]), reinterpret_cast<int4*>(st + i0));
        return;
    }
    for (int k = 0; k < 4; ++k)
    {
        const long long i = i0 + k;
        if (i >= T.n) break;
        float gr[1], wf;
        if (T.dtype == TRIPS_DTYPE_F64)
        {
            gr[0] = (float)reinterpret_cast<const double*>(T.grads)[i];
            wf    = (float)reinterpret_cast<double*>(T.weights)[i];
        }
        else
        {
            gr[0] = reinterpret_cast<const float*>(T.grads)[i];
            wf    = reinterpret_cast<float*>(T.weights)[i];
        }
        adam_unscale(h.loss_scale, gr);
        if (gr[0] == 0.f) continue;
        float m = mo[i], v = vo[i];
        const long long s = (long long)st[i] + 1;
        adam_update(h, adam_rate(h, adam_corrected_lr(h, (uint32_t)s)), gr[0], wf, m, v);
        mo[i] = m;
        vo[i] = v;
        st[i] = (STEP)s;
        if (T.dtype == TRIPS_DTYPE_F64)
            reinterpret_cast<double*>(T.weights)[i] = wf;
        else
            reinterpret_cast<float*>(T.weights)[i] = wf;
    }
}

__global__ __launch_bounds__(256) void adam_fused_kernel(const AdamTable tab)
{
    int ti = 0;
    while (ti + 1 < tab.n && (long long)blockIdx.x >= tab.block_start[ti + 1]) ++ti;
    if (tab.t[ti].steps_dtype == TRIPS_STEPS_I32)
        adam_block<int>(tab, ti);
    else
        adam_block<long long>(tab, ti);
}

hipError_t launch_adam(const TripsAdamTensor* tensors, int n_tensors, hipStream_t stream, Profiler* prof)
{
    ProfScope ps(prof, "adam_fused", stream);
    int done = 0;
    while (done < n_tensors)
    {
        AdamTable tab;
        tab.n           = 0;
        long long block = 0;
        while (done < n_tensors && tab.n < kAdamMaxTensors)
        {
            const TripsAdamTensor& T = tensors[done++];
            if (T.n <= 0) continue;
            tab.t[tab.n]           = T;
            tab.block_start[tab.n] = block;
            auto al16              = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
            tab.vec_ok[tab.n] = al16(T.weights) && al16(T.grads) && al16(T.first_moment) && al16(T.second_moment) &&
                                al16(T.steps);
            block += (T.n + kAdamPerBlock - 1) / kAdamPerBlock;
            tab.n += 1;
        }
        tab.block_start[tab.n] = block;
        if (tab.n == 0 || block == 0) continue;
        if (block > 0x7fffffffll) return hipErrorInvalidValue;
        hipLaunchKernelGGL(adam_fused_kernel, dim3((unsigned)block), dim3(256), 0, stream, tab);
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------------
// The four parameter tensors of a point cloud (position [N,4], size [N], descriptors [C,N], confidence [N]) stepped
// together, with the optimiser state packed per point: one row of CHUNKS x 16 bytes holding {first moment, second
// moment, step counter} of the point's 6 + C elements (position xyzw, size, descriptors, confidence). A point that
// was not seen has zero gradients everywhere and is skipped as a whole (MyAdam.cu:57-61 per element): with per-tensor
// state arrays its state shares every line with its neighbours' and travels anyway; packed, the row of a point that
// is skipped is never touched. Same arithmetic per element as adam_fused_kernel.
// One thread per point. The rows of a wavefront's live points pass through LDS so that the accesses to memory stay
// whole lines: 64 / USED rows per load instruction, lane = (row, 16-byte word).
// What bounds it: memory (6M points of four channels, 39 % of them culled: 1.30 GB in 224 us = 5.8 TB/s; a large copy runs at
// 6.2). Gradients and rows are read once and rows written whole: non-temporal (278 us without; the weights, of which
// live points write parts of lines, are not: 266 with). A third of its vector instructions were divisions by a loss scale
// of one and two loops per bias correction; without them the time of four channels stayed and that of eight, whose rows in
// LDS leave room for few wavefronts, went from 50 to 45 us at 300k points.
struct AdamPointsParams
{
    float *w_pos, *w_size, *w_tex, *w_conf;
    const float *g_pos, *g_size, *g_tex, *g_conf;
    uint4* state;  // [N][CHUNKS]
    long long tex_stride;  // elements between two descriptor rows
    int num_points;
    int scaled;        // some tensor has a loss scale other than 1
    AdamScalars h[4];  // position, size, descriptors, confidence
};

template <int C, int CHUNKS, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void adam_points_kernel(const AdamPointsParams p)
{
    constexpr int E   = 6 + C;
    constexpr int USED = (3 * E + 15) / 16 * 4;  // 16-byte words of a row that travel: whole 64-byte pieces
    constexpr int LS   = USED + 1;   // LDS row stride in 16-byte words: an odd multiple spreads the rows over the banks
    constexpr int RPP  = 64 / USED;  // rows per load instruction
    static_assert(USED <= CHUNKS, "row too short");
    __shared__ uint4 s_rows[WAVES][64 * LS];
    __shared__ unsigned char s_list[WAVES][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long long first = (long long)blockIdx.x * (64 * WAVES) + wave * 64;  // first point of this wavefront
    const long long point = first + lane;
    const bool in         = point < p.num_points;
    float g[E];
    {
        const float4 gp = in ? nt_load(reinterpret_cast<const float4*>(p.g_pos) + point) : make_float4(0.f, 0.f, 0.f, 0.f);
        g[0] = gp.x, g[1] = gp.y, g[2] = gp.z, g[3] = gp.w;
        g[4] = in ? nt_load(p.g_size + point) : 0.f;
#pragma unroll
        for (int c = 0; c < C; ++c) g[5 + c] = in ? nt_load(p.g_tex + c * p.tex_stride + point) : 0.f;
        g[5 + C] = in ? nt_load(p.g_conf + point) : 0.f;
    }
    auto tensor_of = [](int e) constexpr { return e < 4 ? 0 : e == 4 ? 1 : e < 5 + C ? 2 : 3; };
    if (p.scaled)
    {
        asm volatile("");  // (kept out of the way of the usual case, as in adam_unscale)
#pragma unroll
        for (int e = 0; e < E; ++e)
            if (p.h[tensor_of(e)].loss_scale != 1.f) g[e] = g[e] / p.h[tensor_of(e)].loss_scale;
    }
    bool live = false;
#pragma unroll
    for (int e = 0; e < E; ++e) live = live || g[e] != 0.f;
    const unsigned long long mask = __ballot(live);
    if (mask == 0) return;  // (no barrier below: a wavefront is on its own)
    const int nlive = (int)__popcll(mask);
    if (live) s_list[wave][__popcll(mask & ((1ull << lane) - 1ull))] = (unsigned char)lane;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // the weights of the live points: in flight beside the rows
    float w[E];
#pragma unroll
    for (int e = 0; e < E; ++e) w[e] = 0.f;
    if (live)
    {
        const float4 wp = reinterpret_cast<const float4*>(p.w_pos)[point];
        w[0] = wp.x, w[1] = wp.y, w[2] = wp.z, w[3] = wp.w;
        w[4] = p.w_size[point];
#pragma unroll
        for (int c = 0; c < C; ++c) w[5 + c] = p.w_tex[c * p.tex_stride + point];
        w[5 + C] = p.w_conf[point];
    }
    const int my_r = lane / USED, my_c = lane - my_r * USED;
    {
        // every load of the wavefront's rows is issued before the first one is waited for (as a loop that loads and
        // stores pass by pass the round trips to memory ran one after the other)
        constexpr int PASSES = (64 + RPP - 1) / RPP;
        uint4 v[PASSES];
        int src[PASSES];
#pragma unroll
        for (int it = 0; it < PASSES; ++it)
        {
            const int r = it * RPP + my_r;
            src[it]     = -1;
            v[it]       = make_uint4(0u, 0u, 0u, 0u);
            if (my_r < RPP && r < nlive)
            {
                src[it] = s_list[wave][r];
                v[it]   = nt_load(p.state + (first + src[it]) * CHUNKS + my_c);
            }
        }
#pragma unroll
        for (int it = 0; it < PASSES; ++it)
            if (src[it] >= 0) s_rows[wave][src[it] * LS + my_c] = v[it];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (live)
    {
        uint32_t row[4 * USED];
#pragma unroll
        for (int j = 0; j < USED; ++j)
        {
            const uint4 t = s_rows[wave][lane * LS + j];
            row[4 * j] = t.x, row[4 * j + 1] = t.y, row[4 * j + 2] = t.z, row[4 * j + 3] = t.w;
        }
        // The elements of a tensor are mostly updated together, so their counters agree: the bias correction of the
        // tensor's largest counter is computed once and taken by every element whose new counter equals it.
        int top[4] = {0, 0, 0, 0};
#pragma unroll
        for (int e = 0; e < E; ++e) top[tensor_of(e)] = max(top[tensor_of(e)], (int)row[3 * e + 2]);
        // (and tensors with the same learning rate and betas whose largest counters agree share it: usually all four)
        AdamRate top_r[4];
        const float lr0 = adam_corrected_lr(p.h[0], (uint32_t)(top[0] + 1));
        top_r[0]        = adam_rate(p.h[0], lr0);
#pragma unroll
        for (int t = 1; t < 4; ++t)
        {
            const bool same_scalars = p.h[t].lr == p.h[0].lr && p.h[t].beta1 == p.h[0].beta1 && p.h[t].beta2 == p.h[0].beta2;
            const bool shares       = same_scalars && top[t] == top[0];
            float lr                = lr0;
            if (__ballot(!shares))  // (skipped by the whole wavefront in the usual case)
            {
                if (!shares) lr = adam_corrected_lr(p.h[t], (uint32_t)(top[t] + 1));
            }
            top_r[t] = adam_rate(p.h[t], lr);
        }
        bool others = false;  // some element with a gradient has a counter of its own
#pragma unroll
        for (int e = 0; e < E; ++e) others = others || (g[e] != 0.f && (int)row[3 * e + 2] != top[tensor_of(e)]);
        const bool any_others = __ballot(others) != 0ull;
#pragma unroll
        for (int e = 0; e < E; ++e)
        {
            const int t     = tensor_of(e);
            const bool seen = g[e] != 0.f;
            AdamRate r      = top_r[t];
            if (any_others)  // (skipped by the whole wavefront in the usual case)
            {
                asm volatile("");
                const uint32_t own = row[3 * e + 2];
                if (seen && (int)own != top[t]) r = adam_rate(p.h[t], adam_corrected_lr(p.h[t], own + 1u));
            }
            float nw = w[e], nm = __uint_as_float(row[3 * e]), nv = __uint_as_float(row[3 * e + 1]);
            adam_update(p.h[t], r, g[e], nw, nm, nv);
            w[e]           = seen ? nw : w[e];
            row[3 * e]     = seen ? __float_as_uint(nm) : row[3 * e];
            row[3 * e + 1] = seen ? __float_as_uint(nv) : row[3 * e + 1];
            row[3 * e + 2] += seen ? 1u : 0u;
        }
        reinterpret_cast<float4*>(p.w_pos)[point] = make_float4(w[0], w[1], w[2], w[3]);
        p.w_size[point]                          = w[4];
#pragma unroll
        for (int c = 0; c < C; ++c) p.w_tex[c * p.tex_stride + point] = w[5 + c];
        p.w_conf[point] = w[5 + C];
#pragma unroll
        for (int j = 0; j < USED; ++j)
            s_rows[wave][lane * LS + j] = make_uint4(row[4 * j], row[4 * j + 1], row[4 * j + 2], row[4 * j + 3]);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int base = 0; base < nlive; base += RPP)
    {
        const int r = base + my_r;
        if (my_r < RPP && r < nlive)
        {
            const int src                          = s_list[wave][r];
            nt_store(s_rows[wave][src * LS + my_c], p.state + (first + src) * CHUNKS + my_c);
        }
    }
}

// 16-byte chunks of a packed state row: 12 bytes per element, rounded up to whole 128-byte lines
int adam_points_row_chunks(int channels) { return ((6 + channels) * 12 + 127) / 128 * 8; }

hipError_t launch_adam_points(const TripsAdamTensor tensors[4], int num_points, int channels, void* state, hipStream_t stream,
                              Profiler* prof)
{
    ProfScope ps(prof, "adam_fused", stream);
    if (num_points <= 0) return hipSuccess;
    AdamPointsParams p;
    p.w_pos = (float*)tensors[0].weights, p.w_size = (float*)tensors[1].weights, p.w_tex = (float*)tensors[2].weights,
    p.w_conf = (float*)tensors[3].weights;
    p.g_pos = (const float*)tensors[0].grads, p.g_size = (const float*)tensors[1].grads, p.g_tex = (const float*)tensors[2].grads,
    p.g_conf = (const float*)tensors[3].grads;
    p.state      = reinterpret_cast<uint4*>(state);
    p.tex_stride = num_points;
    p.num_points = num_points;
    p.scaled     = 0;
    for (int i = 0; i < 4; ++i)
    {
        const TripsAdamTensor& T = tensors[i];
        if (T.loss_scale != 1.f) p.scaled = 1;
        p.h[i] = AdamScalars{T.lr, T.beta1, T.beta2, T.eps, T.relative_weight_decay, T.absolute_weight_decay,
                             T.weight_clipping_magnitude, T.lower_lr_bound, T.upper_lr_bound, T.loss_scale};
    }
    // (a wavefront keeps to itself: with sixteen channels its rows take 22 KB of LDS, and workgroups of one wavefront fit
    // seven to a CU where those of four fit one)
    const unsigned blocks = (unsigned)((num_points + 255) / 256), blocks64 = (unsigned)((num_points + 63) / 64);
    switch (channels)
    {
        case 3: hipLaunchKernelGGL((adam_points_kernel<3, 8, 4>), dim3(blocks), dim3(256), 0, stream, p); break;
        case 4: hipLaunchKernelGGL((adam_points_kernel<4, 8, 4>), dim3(blocks), dim3(256), 0, stream, p); break;
        case 6: hipLaunchKernelGGL((adam_points_kernel<6, 16, 4>), dim3(blocks), dim3(256), 0, stream, p); break;
        case 8: hipLaunchKernelGGL((adam_points_kernel<8, 16, 4>), dim3(blocks), dim3(256), 0, stream, p); break;
        case 16: hipLaunchKernelGGL((adam_points_kernel<16, 24, 1>), dim3(blocks64), dim3(64), 0, stream, p); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// pose <- se3_exp(t with rotation * 0.1) * pose; t <- 0. Sophus' exp restated (quaternion half-angle form,
// V = I + (1-cos)/th^2 W + (th-sin)/th^3 W^2, first-order renormalisation of the product quaternion).
__global__ __launch_bounds__(128) void apply_tangent_kernel(double* tangent, double* poses, int n)
{
    const int i = blockIdx.x * 128 + threadIdx.x;
    if (i >= n) return;
    double* t = tangent + 6 * (size_t)i;
    double* p = poses + 8 * (size_t)i;
    const double u[3] = {t[0], t[1], t[2]};
    const double w[3] = {t[3] * 0.1, t[4] * 0.1, t[5] * 0.1};
    const double th2  = w[0] * w[0] + w[1] * w[1] + w[2] * w[2];
    const double th   = sqrt(th2);
    double imag, real;
    if (th < 1e-10)
    {
        const double th4 = th2 * th2;
        imag             = 0.5 - th2 / 48.0 + th4 / 3840.0;
        real             = 1.0 - th2 / 8.0 + th4 / 384.0;
    }
    else
    {
        imag = sin(0.5 * th) / th;
        real = cos(0.5 * th);
    }
    const double x1 = imag * w[0], y1 = imag * w[1], z1 = imag * w[2], w1 = real;
    const double W[9] = {0, -w[2], w[1], w[2], 0, -w[0], -w[1], w[0], 0};
    double W2[9];
    for (int r = 0; r < 3; ++r)
        for (int c = 0; c < 3; ++c)
        {
            double s = 0;
            for (int k = 0; k < 3; ++k) s += W[3 * r + k] * W[3 * k + c];
            W2[3 * r + c] = s;
        }
    const double R1[9] = {1 - 2 * (y1 * y1 + z1 * z1), 2 * (x1 * y1 - z1 * w1),     2 * (x1 * z1 + y1 * w1),
                          2 * (x1 * y1 + z1 * w1),     1 - 2 * (x1 * x1 + z1 * z1), 2 * (y1 * z1 - x1 * w1),
                          2 * (x1 * z1 - y1 * w1),     2 * (y1 * z1 + x1 * w1),     1 - 2 * (x1 * x1 + y1 * y1)};
    double Vm[9];
    if (th < 1e-10)
    {
        for (int k = 0; k < 9; ++k) Vm[k] = R1[k];
    }
    else
    {
        const double a = (1 - cos(th)) / th2, b = (th - sin(th)) / (th2 * th);
        for (int k = 0; k < 9; ++k) Vm[k] = (k % 4 == 0 ? 1.0 : 0.0) + a * W[k] + b * W2[k];
    }
    double t1[3];
    for (int r = 0; r < 3; ++r) t1[r] = Vm[3 * r] * u[0] + Vm[3 * r + 1] * u[1] + Vm[3 * r + 2] * u[2];
    const double x2 = p[0], y2 = p[1], z2 = p[2], w2 = p[3];
    double q[4] = {w1 * x2 + x1 * w2 + y1 * z2 - z1 * y2, w1 * y2 - x1 * z2 + y1 * w2 + z1 * x2,
                   w1 * z2 + x1 * y2 - y1 * x2 + z1 * w2, w1 * w2 - x1 * x2 - y1 * y2 - z1 * z2};
    const double sn = q[0] * q[0] + q[1] * q[1] + q[2] * q[2] + q[3] * q[3];
    if (sn != 1.0)
    {
        const double sc = 2.0 / (1.0 + sn);
        for (int k = 0; k < 4; ++k) q[k] *= sc;
    }
    double tn[3];
    for (int r = 0; r < 3; ++r) tn[r] = t1[r] + R1[3 * r] * p[4] + R1[3 * r + 1] * p[5] + R1[3 * r + 2] * p[6];
    for (int k = 0; k < 4; ++k) p[k] = q[k];
    for (int k = 0; k < 3; ++k) p[4 + k] = tn[k];
    for (int k = 0; k < 6; ++k) t[k] = 0.0;
}

hipError_t launch_apply_tangent(double* tangent, double* poses, int n, hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(apply_tangent_kernel, dim3((n + 127) / 128), dim3(128), 0, stream, tangent, poses, n);
    return hipGetLastError();
}

// ---- exports from the saved state ----
// (the records are kept per valid point, at its compact number)
__global__ __launch_bounds__(256) void export_points_kernel(const float* __restrict__ rec, int rec_floats,
                                                            const float* __restrict__ prec, const int32_t* __restrict__ cid_of,
                                                            int n, float* ip, float* depth, float* size_px, int32_t* max_layer)
{
    const int pid = blockIdx.x * 256 + threadIdx.x;
    if (pid >= n) return;
    const int cid   = cid_of[pid];
    const bool ok   = cid >= 0;
    const float* r  = rec + (size_t)(ok ? cid : 0) * rec_floats;
    // {depth, layers written | .. << 4, softplus'(raw size), size_px}
    const float4 tl = ok ? reinterpret_cast<const float4*>(prec)[cid] : make_float4(-1.f, 0.f, 0.f, 0.f);
    if (ip)
    {
        ip[2 * (size_t)pid]     = ok ? r[0] : 0.f;
        ip[2 * (size_t)pid + 1] = ok ? r[1] : 0.f;
    }
    if (depth) depth[pid] = tl.x;
    if (size_px) size_px[pid] = ok ? tl.w : 0.f;
    if (max_layer) max_layer[pid] = ok ? (int)(__float_as_uint(tl.y) & kLayersMask) : 0;
}

hipError_t launch_export_points(const float* rec, int rec_floats, const float* prec, const int32_t* cid_of, int n, float* ip,
                                float* depth, float* size_px, int32_t* max_layer, hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(export_points_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, rec, rec_floats, prec, cid_of, n, ip,
                       depth, size_px, max_layer);
    return hipGetLastError();
}

// Saved tables are tile-major (padded); the exports are row-major, layer by layer. Bound by the scattered requests of the search for a
// list entry's point: a lane makes four searches side by side. us, with an array of the points by number, which the forward then had
// to write; searched by halves, an entry at a time; and so: 6M points in no order at 1920 x 1080 570, 1500 and 524, in Morton
// order 482, 760 and 406, 300k at 641 x 479 18, 48 and 19, 4M in tight clusters 205, 271 and 43.
__global__ __launch_bounds__(256) void export_lists_kernel(const PyramidGeom g, int K, const int32_t* __restrict__ lists,
                                                           const int32_t* __restrict__ retained,
                                                           const int32_t* __restrict__ cid_of,
                                                           const int32_t* __restrict__ chunk_valid, int num_points,
                                                           int points_per_block, int32_t* out_lists, int32_t* out_retained,
                                                           int32_t* out_lengths)
{
    // four positions of a pixel's list
    const int P = g.off[g.num_layers], quads = K >> 2;
    const long long item = (long long)blockIdx.x * 256 + threadIdx.x;
    const int r = (int)(item / quads), q = (int)(item - (long long)r * quads);
    if (r >= P) return;
    int layer = 0;
    while (layer + 1 < g.num_layers && r >= g.off[layer + 1]) ++layer;
    const int local = r - g.off[layer];
    const int x = local % g.w[layer], y = local / g.w[layer];
    const int ip = pix_index(g, layer, x, y);
    const unsigned word = (unsigned)retained[ip];  // retained entries | filled list positions << 5 | list length << 10
    const int filled    = (int)((word >> kRetainedBits) & kRetainedMask);
    if (out_retained && q == 0) out_retained[r] = (int)(word & kRetainedMask);
    if (out_lengths && q == 0) out_lengths[r] = (int)(word >> (2 * kRetainedBits));
    if (!out_lists) return;
    // The points of the four compact numbers. cid_of counts on over culled points (~number of the next valid one), so an entry g of
    // it, as a number, says that the point lies at least |cid - g| positions further on or back. A search goes on by that distance
    // times the chunk's points per valid point (of a culled point half of that further), and every other time to the middle of what
    // is left.
    const int4 four = 4 * q < filled ? *reinterpret_cast<const int4*>(lists + list_word((unsigned)ip, 4 * q, K)) : make_int4(0, 0, 0, 0);
    const int cid[4] = {four.x, four.y, four.z, four.w};
    int lo[4], hi[4], at[4], point[4];  // a point is in [lo, hi)
    float spread[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
    {
        point[i] = -1, lo[i] = hi[i] = at[i] = 0, spread[i] = 1.f;
        if (4 * q + i >= filled) continue;
        const int chunk = cid[i] / points_per_block, begin = chunk * points_per_block, end = min(num_points, begin + points_per_block);
        const int valid = chunk_valid[chunk];
        spread[i] = (float)(end - begin) / (float)max(valid, 1);
        lo[i]     = cid[i];
        hi[i]     = end - (begin + valid - 1 - cid[i]);  // (valid points behind it are as many positions)
        at[i]     = begin + (int)((float)(cid[i] - begin) * spread[i]);
    }
    for (int turn = 1; lo[0] < hi[0] || lo[1] < hi[1] || lo[2] < hi[2] || lo[3] < hi[3]; ++turn)
    {
        int c[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
        {
            at[i] = min(max(at[i], lo[i]), hi[i] - 1);
            c[i]  = lo[i] < hi[i] ? cid_of[at[i]] : 0;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
        {
            if (lo[i] >= hi[i]) continue;
            const int away = cid[i] - (c[i] < 0 ? ~c[i] : c[i]);
            if (c[i] == cid[i])
                point[i] = at[i], hi[i] = lo[i];
            else if (away >= 0)
                lo[i] = at[i] + away + (c[i] < 0 ? 1 : 0);
            else
                hi[i] = at[i] + away + 1;
            at[i] = turn % 2 == 0 ? lo[i] + (hi[i] - lo[i]) / 2 : at[i] + (int)(((float)away + (c[i] < 0 ? 0.5f : 0.f)) * spread[i]);
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) out_lists[(size_t)r * K + 4 * q + i] = point[i];
}

hipError_t launch_export_lists(const PyramidGeom& g, int K, const int32_t* lists, const int32_t* retained,
                               const int32_t* cid_of, const int32_t* chunk_valid, int num_points, int points_per_block, int32_t* out_lists,
                               int32_t* out_retained, int32_t* out_lengths, hipStream_t stream)
{
    const int P = g.off[g.num_layers];
    if (P <= 0) return hipSuccess;
    const long long items = (long long)P * (K >> 2);  // (lists of 8 or 16)
    hipLaunchKernelGGL(export_lists_kernel, dim3((unsigned)((items + 255) / 256)), dim3(256), 0, stream, g, K, lists, retained, cid_of,
                       chunk_valid, num_points, points_per_block, out_lists, out_retained, out_lengths);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void sum_i32_kernel(const int32_t* __restrict__ v, long long n, unsigned mask,
                                                      unsigned long long* out)
{
    __shared__ unsigned long long s[4];
    unsigned long long acc = 0;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256)
        acc += (unsigned long long)((unsigned)v[i] & mask);
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(out, s[0] + s[1] + s[2] + s[3]);
}

// *out = sum of (v[i] & mask)
hipError_t launch_sum_i32(const int32_t* v, long long n, unsigned mask, unsigned long long* out, hipStream_t stream)
{
    hipError_t e = hipMemsetAsync(out, 0, sizeof(unsigned long long), stream);
    if (e != hipSuccess) return e;
    if (n <= 0) return hipSuccess;
    int blocks = (int)((n + 255) / 256);
    if (blocks > 1024) blocks = 1024;
    hipLaunchKernelGGL(sum_i32_kernel, dim3(blocks), dim3(256), 0, stream, v, n, mask, out);
    return hipGetLastError();
}

}  // namespace trips
