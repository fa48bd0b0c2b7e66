// Device-side scalar math of the splat path (gfx950). Compiled with -ffp-contract=off: positions,
// depths and sizes feed integer decisions (pixel, layer, sort key), so every expression below is
// evaluated exactly in the order written, with IEEE single-precision operations.
//
// Reference lines restated here (paths relative to the reference checkout):
//   softplus / derivative     src/lib/rendering/RenderForward.cu:154-159, RenderBackward.cu:71-83
//   layer factor              src/lib/rendering/PointBlending.h:81-149
//   bilinear weights          src/lib/rendering/PointBlending.h:211-264
//   pinhole projection        src/lib/rendering/PointRendererHelper.h:232-253, RenderForward.cu:69-76,302-303
//   projection backward       src/lib/rendering/PointRendererHelper.h:434-494
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#pragma clang fp contract(off)

namespace trips
{
constexpr float kAlphaDestCutoff = 0.001f;  // ALPHA_DEST_CUTOFF, RenderForward.cu:907

// exp / log evaluated in double and rounded once, so that results do not depend on a libm's float path. The projection is bound by
// its vector instructions, and the two functions for any double were a third of them: a float's exponential and the logarithm
// of 1 + exp(x) need no second word of the argument, no range tests and, with a table of reciprocals, no division. Their errors
// stay below 2^-51 of the value, and the rounded results are those of exp() and log() in double: of exp for every float from -200 to
// 200, of log for every z = 1 + exp(x) of a float x, its only arguments. (Of the other floats up to there two have a logarithm that
// close to the middle between two floats: z = 0x1.cb534cp+13 and 0x1.c09d7cp+27, rounded the other way than by the libm.)

// A constant kept in scalar registers: as an operand of a multiply-add it then costs nothing, where the compiler would copy
// it into two vector registers first.
__device__ __forceinline__ double scalar_const(double c)
{
    asm("" : "+s"(c));
    return c;
}

// exp(x) for -200 <= x <= 200 (or NaN): 2^n 2^f with n = rint(x log2 e), |f| <= 1/2, and for 2^f a polynomial that interpolates
// it in the Chebyshev nodes (relative error 2^-55).
__device__ __forceinline__ float exp_rn(float x)
{
    const double xd = (double)x, log2e = scalar_const(0x1.71547652b82fep+0);
    const double n = rint(xd * log2e);
    const double f = fma(xd, scalar_const(0x1.777d0ffda0d24p-56), fma(xd, log2e, -n));
    double q       = scalar_const(0x1.e9d3fe3952179p-32);
    q              = fma(q, f, scalar_const(0x1.e6063f7217bc6p-28));
    q              = fma(q, f, scalar_const(0x1.b524fae627834p-24));
    q              = fma(q, f, scalar_const(0x1.62bfd47773353p-20));
    q              = fma(q, f, scalar_const(0x1.ffcbfc670dcd4p-17));
    q              = fma(q, f, scalar_const(0x1.430913096fd9fp-13));
    q              = fma(q, f, scalar_const(0x1.5d87fe78a5276p-10));
    q              = fma(q, f, scalar_const(0x1.3b2ab6fba1ddap-7));
    q              = fma(q, f, scalar_const(0x1.c6b08d704a0c2p-5));
    q              = fma(q, f, scalar_const(0x1.ebfbdff82c598p-3));
    q              = fma(q, f, scalar_const(0x1.62e42fefa39efp-1));
    return (float)__builtin_amdgcn_ldexp(fma(q, f, 1.0), (int)n);
}

// {c, -log c} for c = 1 / (1 + i / 128) rounded to float, which makes the product with another float exact in double
constexpr int kLogTable = 128;
__device__ __forceinline__ double2 log_table_entry(int i)
{
    const double c = (double)(float)(1.0 / (1.0 + (double)i / kLogTable));
    return make_double2(c, -log(c));
}

// log(z) for finite z >= 1 (or NaN): with z = 2^k m, m in [1 - 2^-8, 2 - 2^-8), and the table's c next to 1 / m,
// k log 2 - log c + log(1 + r), r = m c - 1 (exact), |r| <= 2^-7, and the series of log(1 + r) to the eighth power
__device__ __forceinline__ float log_rn(float z, const double2* table)
{
    const uint32_t u = __float_as_uint(z) + 0x8000u;
    const int minus_k = 127 - (int)(u >> 23);
    const double2 t   = table[(u >> 16) & (kLogTable - 1)];
    const double r    = fma(__builtin_amdgcn_ldexp((double)z, minus_k), t.x, -1.0);
    double q          = scalar_const(-1.0 / 8);
    q                 = fma(q, r, scalar_const(1.0 / 7));
    q                 = fma(q, r, scalar_const(-1.0 / 6));
    q                 = fma(q, r, scalar_const(1.0 / 5));
    q                 = fma(q, r, scalar_const(-1.0 / 4));
    q                 = fma(q, r, scalar_const(1.0 / 3));
    q                 = fma(q, r, -0.5);
    return (float)(fma((double)minus_k, scalar_const(-0x1.62e42fefa39efp-1), t.y) + fma(r * r, q, r));
}

// 1 / b in double for a float b > 0, within two units of the last place: the hardware's reciprocal (an error e of 2^-23) times
// 1 + e + e^2. A float times it is within 2^-51 of the quotient, which is never that close to the middle between two
// floats (25-bit numbers; quotients of floats keep 2^-49 of themselves away from these): rounded to float it is the IEEE quotient,
// where that is a normal number. Quotients by the same number share it: three operations each instead of eleven.
__device__ __forceinline__ double reciprocal_of(float b)
{
    const double bd = (double)b;
    if (!(b > 0x1p-60f && b < 0x1p60f)) return 1.0 / bd;  // where the hardware's has no more to give (infinity among them)
    const double r = (double)__builtin_amdgcn_rcpf(b);
    const double e = fma(-bd, r, 1.0);
    return fma(r, fma(e, e, e), r);
}
__device__ __forceinline__ float quotient(float a, double reciprocal) { return (float)((double)a * reciprocal); }
// The IEEE quotient also below the normal numbers, where floats are wider apart and it can itself be the middle between two: there it
// is divided out.
__device__ __forceinline__ float quotient_of_any_size(float a, float b, double reciprocal)
{
    const double q = (double)a * reciprocal;
    if (fabs(q) < 0x1p-126 && a != 0.f) return (float)((double)a / (double)b);
    return (float)q;
}

// softplus and its derivative, with the one exponential that they share (derivative may be nullptr)
__device__ __forceinline__ float softplus(float x, const double2* table, float* derivative)
{
    const float z   = exp_rn(x < -200.f ? -200.f : x > 20.f ? 20.f : x);
    const float sum = 1.f + z;
    if (derivative) *derivative = x > 20.f ? 1.f : z / sum;
    const float y = log_rn(sum, table);
    return x > 20.f ? x : y;
}

// floor(log2 s), ceil(log2 s) for finite s > 0 from the bit pattern (exact; the reference rounds log2f first)
__device__ __forceinline__ void log2_floor_ceil(float s, int& lo, int& hi)
{
    uint32_t u   = __float_as_uint(s);
    int e        = int((u >> 23) & 0xff);
    uint32_t man = u & 0x7fffffu;
    if (e == 0)
    {
        lo = -127;
        hi = -126;
        return;
    }
    lo = e - 127;
    hi = lo + (man != 0 ? 1 : 0);
}

// compute_point_size_fac (PointBlending.h:81-149) for s > 1 and more than one layer, the branch that interpolates
// between two layers. (The other branch, 0.75 exp(s - 1) + 0.25 for a point that lands in layer 0 only, is evaluated once
// per point by encode_size_field below.) `layer` must be one that the point is written to: at most ceil(log2 s).
// With q = s / 2^layer (exact) the reference's cases are: q >= 2, a layer below both, 1; 1 <= q < 2, the lower layer,
// 1 - (s - 2^layer) / 2^layer = 2 - q with the same rounding, or 1 if it is the last layer, where both are clamped to it;
// 1/2 < q < 1, the higher layer, (s - 2^(layer - 1)) / 2^(layer - 1) = 2 q - 1, exact. The reference's derivative where the
// two layers are the same is 1. (Size and layer are compared through q instead of through the bits of log2 s: 9 vector
// instructions instead of 20, once per list entry of every pixel.)
__device__ __forceinline__ float layer_factor_interpolated(float s, int layer, int max_layers, float* grad)
{
    const float m   = __uint_as_float((uint32_t)(127 - layer) << 23);  // 2^-layer
    const float q   = s * m;
    const bool last = layer == max_layers - 1;
    float f         = (q < 2.f && !last) ? 2.f - q : 1.f;
    f               = q < 1.f ? 2.f * q - 1.f : f;
    if (grad)
    {
        float J = q < 2.f ? -m : 0.f;
        J       = (q == 1.f || last) ? 1.f : J;
        *grad   = q < 1.f ? 2.f * m : J;
    }
    return f;
}

// The "small point" branch of the layer factor (layer_higher == 0, i.e. size <= 1 pixel or a single layer) is the
// only one that needs exp(), and it does not depend on the layer (such a point lands in layer 0 only). The
// projection kernel evaluates it once per point and stores it NEGATED in the size slot of the per-point record;
// the blend and the backward then read the factor instead of re-evaluating a double-precision exp per list entry.
__device__ __forceinline__ float encode_size_field(float size_px, int max_layers)
{
    const bool small_branch = !(size_px > 1.f) || max_layers == 1;
    const float x = size_px - 1.f;
    return small_branch ? -(0.75f * exp_rn(x < -200.f ? -200.f : x > 200.f ? 200.f : x) + 0.25f) : size_px;
}

// layer factor from the encoded size field
__device__ __forceinline__ float layer_factor_encoded(float field, int layer, int max_layers)
{
    if (field < 0.f) return -field;
    return layer_factor_interpolated(field, layer, max_layers, nullptr);
}

// same with the reference's gradient; true_size is the un-encoded projected size
__device__ __forceinline__ float layer_factor_encoded_grad(float field, float true_size, int layer, int max_layers,
                                                           float* grad)
{
    if (field < 0.f)
    {
        *grad = 0.27591f * true_size;
        return -field;
    }
    return layer_factor_interpolated(field, layer, max_layers, grad);
}

// alpha of a list entry (r0: the first four floats of its point's blend record) at pixel (gx, gy) of `layer`
// (RenderForward.cu:875-899: bilinear weight x confidence x layer factor)
__device__ __forceinline__ float entry_alpha(const float4& r0, int layer, int num_layers, int gx, int gy)
{
    const float m  = __uint_as_float((uint32_t)(127 - layer) << 23);  // 2^-layer
    const float ux = r0.x * m, uy = r0.y * m;
    // (the reference's test for a distance above 1 never holds: the pixel is one of the four around (ux, uy))
    const float w = (1.f - fabsf(ux - float(gx))) * (1.f - fabsf(uy - float(gy)));
    float a       = w * r0.w;
    a *= layer_factor_encoded(r0.z, layer, num_layers);
    return a;
}

struct Pose
{
    float qx, qy, qz, qw, tx, ty, tz;
};

// Sophus::SE3d memory (quaternion xyzw, translation, pad) cast to float (RenderConstants.h:88)
__device__ __forceinline__ Pose load_pose(const double* p)
{
    Pose P;
    P.qx = (float)p[0];
    P.qy = (float)p[1];
    P.qz = (float)p[2];
    P.qw = (float)p[3];
    P.tx = (float)p[4];
    P.ty = (float)p[5];
    P.tz = (float)p[6];
    return P;
}

// SE3f * point; rotation in the form of Eigen's QuaternionBase::_transformVector
__device__ __forceinline__ void transform_point(const Pose& V, float px, float py, float pz, float out[3])
{
    float ux = V.qy * pz - V.qz * py;
    float uy = V.qz * px - V.qx * pz;
    float uz = V.qx * py - V.qy * px;
    ux += ux;
    uy += uy;
    uz += uz;
    float cx = V.qy * uz - V.qz * uy;
    float cy = V.qz * ux - V.qx * uz;
    float cz = V.qx * uy - V.qy * ux;
    out[0]   = (px + V.qw * ux + cx) + V.tx;
    out[1]   = (py + V.qw * uy + cy) + V.ty;
    out[2]   = (pz + V.qw * uz + cz) + V.tz;
}

// Eigen's QuaternionBase::toRotationMatrix, row-major
__device__ __forceinline__ void rotation_matrix(const Pose& V, float R[9])
{
    float tx = 2.f * V.qx, ty = 2.f * V.qy, tz = 2.f * V.qz;
    float twx = tx * V.qw, twy = ty * V.qw, twz = tz * V.qw;
    float txx = tx * V.qx, txy = ty * V.qx, txz = tz * V.qx;
    float tyy = ty * V.qy, tyz = tz * V.qy, tzz = tz * V.qz;
    R[0]      = 1.f - (tyy + tzz);
    R[1]      = txy - twz;
    R[2]      = txz + twy;
    R[3]      = txy + twz;
    R[4]      = 1.f - (txx + tzz);
    R[5]      = tyz - twx;
    R[6]      = txz - twy;
    R[7]      = tyz + twx;
    R[8]      = 1.f - (txx + tyy);
}

// 8-parameter distortion (k1..k6 rational radial, p1 p2 tangential) of Saiga's distortNormalizedPoint,
// sentinel (100000,100000) beyond the cut-off radius. Jp: 2x2 row-major, Jd: 2x8 row-major; may be nullptr.
__device__ __forceinline__ void distort(float x, float y, const float* c, float cutoff, float& xd, float& yd,
                                        float* Jp, float* Jd)
{
    float k1 = c[0], k2 = c[1], k3 = c[2], k4 = c[3], k5 = c[4], k6 = c[5], p1 = c[6], p2 = c[7];
    float x2 = x * x, y2 = y * y;
    float r2 = x2 + y2, _2xy = 2.f * x * y;
    float r4 = r2 * r2, r6 = r4 * r2;
    float U   = 1.f + k1 * r2 + k2 * r4 + k3 * r6;
    float Vv  = 1.f + k4 * r2 + k5 * r4 + k6 * r6;
    float iV  = 1.f / Vv;
    float rad = U * iV;
    float tX  = p1 * _2xy + p2 * (r2 + 2.f * x2);
    float tY  = p1 * (r2 + 2.f * y2) + p2 * _2xy;
    xd        = x * rad + tX;
    yd        = y * rad + tY;
    if (Jp)
    {
        float dU   = k1 + 2.f * k2 * r2 + 3.f * k3 * r4;
        float dV   = k4 + 2.f * k5 * r2 + 3.f * k6 * r4;
        float drad = (dU * Vv - U * dV) * iV * iV;
        Jp[0]      = rad + x * drad * 2.f * x + (2.f * p1 * y + 6.f * p2 * x);
        Jp[1]      = x * drad * 2.f * y + (2.f * p1 * x + 2.f * p2 * y);
        Jp[2]      = y * drad * 2.f * x + (2.f * p1 * x + 2.f * p2 * y);
        Jp[3]      = rad + y * drad * 2.f * y + (6.f * p1 * y + 2.f * p2 * x);
    }
    if (Jd)
    {
        float uv2 = U * iV * iV;
        Jd[0]     = x * r2 * iV;
        Jd[1]     = x * r4 * iV;
        Jd[2]     = x * r6 * iV;
        Jd[3]     = -x * uv2 * r2;
        Jd[4]     = -x * uv2 * r4;
        Jd[5]     = -x * uv2 * r6;
        Jd[6]     = _2xy;
        Jd[7]     = r2 + 2.f * x2;
        Jd[8]     = y * r2 * iV;
        Jd[9]     = y * r4 * iV;
        Jd[10]    = y * r6 * iV;
        Jd[11]    = -y * uv2 * r2;
        Jd[12]    = -y * uv2 * r4;
        Jd[13]    = -y * uv2 * r6;
        Jd[14]    = r2 + 2.f * y2;
        Jd[15]    = _2xy;
    }
    if (r2 > cutoff * cutoff)
    {
        xd = 100000.f;
        yd = 100000.f;
        if (Jp) Jp[0] = Jp[1] = Jp[2] = Jp[3] = 0.f;
        if (Jd)
            for (int i = 0; i < 16; ++i) Jd[i] = 0.f;
    }
}

// Camera constants of one view, gathered once per thread from uniform memory.
struct Camera
{
    Pose V;
    float fx, fy, cx, cy, s;
    float dist[8];
    bool no_distortion;            // all of dist[] are zero (wave-uniform: the forward then skips the rational model)
    float cfx, cfy, ccx, ccy, cs;  // crop transform
    float r00, r01, r10, r11;      // crop rotation
    float centre_x, centre_y;      // float(w/2), float(h/2), integer division
    float dist_cutoff;
};

struct Projected
{
    float ipx, ipy, z, scale;  // scale = K.fx * crop.fx (divide by z after multiplying with a radius)
    double iz;                 // 1 / z where z > 0
};

__device__ __forceinline__ Projected project(const Camera& cam, float px, float py, float pz)
{
    float view[3];
    transform_point(cam.V, px, py, pz, view);
    float z  = fmaxf(view[2], 0.f);
    const double izd = reciprocal_of(view[2]);  // (a point that is not in front of the camera is culled, wherever it falls)
    const float iz   = (float)izd;
    float nx = view[0] * iz, ny = view[1] * iz;
    float dx, dy;
    if (cam.no_distortion)
    {
        // all eight coefficients are zero: the model is x * (1 / 1) + 0 in float arithmetic, which is x + 0 (the
        // addition turns a negative zero into a positive one, as the full expression does); the cut-off stays
        dx = nx + 0.f;
        dy = ny + 0.f;
        if (nx * nx + ny * ny > cam.dist_cutoff * cam.dist_cutoff) dx = dy = 100000.f;
    }
    else
        distort(nx, ny, cam.dist, cam.dist_cutoff, dx, dy, nullptr, nullptr);
    if (dx == 100000.f) z = 0.f;
    float ix = cam.fx * dx + cam.s * dy + cam.cx;
    float iy = cam.fy * dy + cam.cy;
    float jx = cam.cfx * ix + cam.cs * iy + cam.ccx;
    float jy = cam.cfy * iy + cam.ccy;
    jx -= cam.centre_x;
    jy -= cam.centre_y;
    float rx = cam.r00 * jx + cam.r01 * jy;
    float ry = cam.r10 * jx + cam.r11 * jy;
    Projected P;
    P.ipx   = rx + cam.centre_x;
    P.ipy   = ry + cam.centre_y;
    P.z     = z;
    P.scale = cam.fx * cam.cfx;
    P.iz    = izd;
    return P;
}

// image-space gradient (g0,g1) -> point (3), pose (6), K (5), distortion (8); view-space point given
__device__ __forceinline__ void project_backward(const Camera& cam, const float R[9], float vx, float vy, float vz,
                                                 float g0, float g1, float g_point[3], float g_pose[6], float g_k[5],
                                                 float g_dis[8], bool want_intrinsics)
{
    float iz = 1.f / vz, iz2 = 1.f / (vz * vz);
    float nx = vx * iz, ny = vy * iz;
    float gr0 = cam.r00 * g0 + cam.r10 * g1;
    float gr1 = cam.r01 * g0 + cam.r11 * g1;
    float a   = cam.cfx * gr0;
    float b   = cam.cs * gr0 + cam.cfy * gr1;
    float k0  = cam.fx * a;
    float k1  = cam.s * a + cam.fy * b;
    float dx, dy, d0, d1;
    if (cam.no_distortion)
    {
        // all eight coefficients are zero: the distortion is the identity, and of the Jacobian of its coefficients only the
        // powers of the radius are left (the same bits as through distort() and its matrices, whose zeros stay in the
        // sums: they carry a gradient of one axis that is not finite to the other)
        const bool cut = nx * nx + ny * ny > cam.dist_cutoff * cam.dist_cutoff;  // (never of a point that the projection kept)
        dx = cut ? 100000.f : nx;
        dy = cut ? 100000.f : ny;
        const float j = cut ? 0.f : 1.f;
        d0 = j * k0 + 0.f * k1;
        d1 = 0.f * k0 + j * k1;
        if (want_intrinsics)
        {
            const float x = cut ? 0.f : nx, y = cut ? 0.f : ny;
            const float x2 = x * x, y2 = y * y, r2 = x2 + y2, r4 = r2 * r2, r6 = r4 * r2, xy2 = 2.f * x * y;
            g_dis[0] = x * r2 * k0 + y * r2 * k1;
            g_dis[1] = x * r4 * k0 + y * r4 * k1;
            g_dis[2] = x * r6 * k0 + y * r6 * k1;
            g_dis[3] = -g_dis[0];
            g_dis[4] = -g_dis[1];
            g_dis[5] = -g_dis[2];
            g_dis[6] = xy2 * k0 + (r2 + 2.f * y2) * k1;
            g_dis[7] = (r2 + 2.f * x2) * k0 + xy2 * k1;
        }
    }
    else
    {
        float Jp[4], Jd[16];
        distort(nx, ny, cam.dist, cam.dist_cutoff, dx, dy, Jp, Jd);  // a pointer chosen at run time would put the arrays in scratch memory
        d0 = Jp[0] * k0 + Jp[2] * k1;
        d1 = Jp[1] * k0 + Jp[3] * k1;
        if (want_intrinsics)
            for (int i = 0; i < 8; ++i) g_dis[i] = Jd[i] * k0 + Jd[8 + i] * k1;
    }
    float v0  = iz * d0;
    float v1  = iz * d1;
    float v2  = (-vx * iz2) * d0 + (-vy * iz2) * d1;
    g_point[0] = R[0] * v0 + R[3] * v1 + R[6] * v2;
    g_point[1] = R[1] * v0 + R[4] * v1 + R[7] * v2;
    g_point[2] = R[2] * v0 + R[5] * v1 + R[8] * v2;
    g_pose[0]  = v0;
    g_pose[1]  = v1;
    g_pose[2]  = v2;
    g_pose[3]  = vy * v2 - vz * v1;
    g_pose[4]  = vz * v0 - vx * v2;
    g_pose[5]  = vx * v1 - vy * v0;
    if (want_intrinsics)
    {
        g_k[0] = dx * a;
        g_k[1] = dy * b;
        g_k[2] = a;
        g_k[3] = b;
        g_k[4] = dy * a;
    }
}

// saturating float -> int (what v_cvt_i32_f32 does); NaN -> 0
__device__ __forceinline__ int trunc_sat(float v)
{
    if (!(v == v)) return 0;
    if (v >= 2147483648.f) return 2147483647;
    if (v <= -2147483648.f) return -2147483647 - 1;
    return (int)v;
}

}  // namespace trips
