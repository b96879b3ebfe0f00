// Device pieces shared by the query kernels: the point's mesh, exact triangle solid angles, the far
// field of a slot and the node fetch into LDS.  Every kernel that answers a query uses these, so
// a point's terms have the same bits in each.
#pragma once

#include "fwn_internal.h"

namespace fwn {
namespace {

__device__ __forceinline__ int mesh_of64(const int64_t* off, int M, int64_t t)
{
    int lo = 0, hi = M - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (off[mid] <= t) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// Exact triangle solid angles.  Every rounding stands in the source (explicit fma, no contraction by the
// compiler, which fuses a product and a sum only where both lie in one basic block): a leaf's value has
// the same bits in every kernel, whatever else is compiled around it.

// FP32, normalised-vector van Oosterom-Strackee form
__device__ __forceinline__ float tri_f32(const float* __restrict__ t, float qx, float qy, float qz)
{
#pragma clang fp contract(off)
    float ax = t[0] - qx, ay = t[1] - qy, az = t[2] - qz;
    float bx = t[3] - qx, by = t[4] - qy, bz = t[5] - qz;
    float cx = t[6] - qx, cy = t[7] - qy, cz = t[8] - qz;
    float la2 = fmaf(ax, ax, fmaf(ay, ay, az * az));
    float lb2 = fmaf(bx, bx, fmaf(by, by, bz * bz));
    float lc2 = fmaf(cx, cx, fmaf(cy, cy, cz * cz));
    // a zero where a corner or the plane is hit, selected at the end: two branches around the rest cost
    // more than they save
    const bool corner = la2 == 0.0f || lb2 == 0.0f || lc2 == 0.0f;
    float ia = __builtin_amdgcn_rsqf(la2), ib = __builtin_amdgcn_rsqf(lb2), ic = __builtin_amdgcn_rsqf(lc2);
    ax *= ia; ay *= ia; az *= ia;
    float ux = fmaf(bx, ib, -ax), uy = fmaf(by, ib, -ay), uz = fmaf(bz, ib, -az);
    float vx = fmaf(cx, ic, -ax), vy = fmaf(cy, ic, -ay), vz = fmaf(cz, ic, -az);
    bx *= ib; by *= ib; bz *= ib;
    cx *= ic; cy *= ic; cz *= ic;
    float nx = fmaf(uy, vz, -uz * vy);
    float ny = fmaf(uz, vx, -ux * vz);
    float nz = fmaf(ux, vy, -uy * vx);
    float num = fmaf(ax, nx, fmaf(ay, ny, az * nz));
    float ab = fmaf(ax, bx, fmaf(ay, by, az * bz));
    float ac = fmaf(ax, cx, fmaf(ay, cy, az * cz));
    float bc = fmaf(bx, cx, fmaf(by, cy, bz * cz));
    float den = 1.0f + ab + ac + bc;
    return corner || num == 0.0f ? 0.0f : 2.0f * atan2f(num, den);
}

// a.b in FP64: products of the three axes, two of them fused into the sum
__device__ __forceinline__ double dot_f64(double ax, double ay, double az, double bx, double by, double bz)
{
    return fma(az, bz, fma(ax, bx, ay * by));
}

// FP64, 2 atan2(a.(b x c), |a||b||c| + (a.b)|c| + (b.c)|a| + (c.a)|b|)
__device__ __forceinline__ double tri_f64(const float* __restrict__ t, float qx, float qy, float qz)
{
#pragma clang fp contract(off)
    double q0 = qx, q1 = qy, q2 = qz;
    double ax = (double)t[0] - q0, ay = (double)t[1] - q1, az = (double)t[2] - q2;
    double bx = (double)t[3] - q0, by = (double)t[4] - q1, bz = (double)t[5] - q2;
    double cx = (double)t[6] - q0, cy = (double)t[7] - q1, cz = (double)t[8] - q2;
    double la = sqrt(dot_f64(ax, ay, az, ax, ay, az));
    double lb = sqrt(dot_f64(bx, by, bz, bx, by, bz));
    double lc = sqrt(dot_f64(cx, cy, cz, cx, cy, cz));
    if (la == 0.0 || lb == 0.0 || lc == 0.0) return 0.0;
    double num = dot_f64(ax, ay, az, fma(by, cz, -(bz * cy)), fma(bz, cx, -(bx * cz)), fma(bx, cy, -(by * cx)));
    if (num == 0.0) return 0.0;
    double den = fma(la * lb, lc, dot_f64(ax, ay, az, bx, by, bz) * lc);
    den = fma(la, dot_f64(bx, by, bz, cx, cy, cz), den);
    den = fma(lb, dot_f64(cx, cy, cz, ax, ay, az), den);
    return 2.0 * atan2(num, den);
}

// order-2 far field of one slot, split into t and inv3 (the caller adds fmaf(t, inv3, omega)):
//   omega += inv3 (o0 + inv2 (q1 + inv2 q2)),  inv = 1 / |d|,
// o0 = d.N, q1 = d^T A d, q2 = B(d, d, d).  The build folds the constant terms (tr M1 of o0 and
// C.d of q1) into A and B through |d|^2 / |d|^2, so every product has one coefficient operand
// and no coefficient needs a move into a vector register; q1 and q2 are evaluated in Horner form
// over the packed coefficients (no monomials needed).  W(k) reads slot word k: scalar registers
// in the batched traversal, per-lane registers in the single-point kernel (the same operations,
// so the same bits).
template <class W>
__device__ __forceinline__ void far_field_terms(const W& w, float dx, float dy, float dz, float d2, float& t,
                                                float& inv3)
{
    const float inv = __builtin_amdgcn_rsqf(d2);
    const float inv2 = inv * inv;
    inv3 = inv2 * inv;
    const float o0 = fmaf(dx, w(FWN_W_NX), fmaf(dy, w(FWN_W_NY), dz * w(FWN_W_NZ)));
    const float zz = dz * dz; // shared with the slot test's |d|^2
    // A: xx yy zz xy yz zx;  q1 = A_zz zz + x (A_xx x + A_xy y + A_zx z) + y (A_yy y + A_yz z)
    const float a1 = fmaf(w(FWN_W_A), dx, fmaf(w(FWN_W_A + 3), dy, w(FWN_W_A + 5) * dz));
    const float b1 = fmaf(w(FWN_W_A + 1), dy, w(FWN_W_A + 4) * dz);
    const float q1 = fmaf(dy, b1, fmaf(dx, a1, w(FWN_W_A + 2) * zz));
    // B: xxx yyy zzz xxy xxz yyx yyz zzx zzy xyz;
    // q2 = zz (B_zzx x + B_zzy y + B_zzz z) + x (x (B_xxx x + B_xxy y + B_xxz z) + y (B_yyx y + B_xyz z))
    //      + y y (B_yyy y + B_yyz z)
    const float L = fmaf(w(FWN_W_B + 7), dx, fmaf(w(FWN_W_B + 8), dy, w(FWN_W_B + 2) * dz));
    const float P = fmaf(w(FWN_W_B), dx, fmaf(w(FWN_W_B + 3), dy, w(FWN_W_B + 4) * dz));
    const float Qv = fmaf(w(FWN_W_B + 5), dy, w(FWN_W_B + 9) * dz);
    const float X = fmaf(dy, Qv, dx * P);
    const float R = fmaf(w(FWN_W_B + 1), dy, w(FWN_W_B + 6) * dz);
    const float q2 = fmaf(dy * dy, R, fmaf(dx, X, zz * L));
    t = fmaf(inv2, fmaf(inv2, q2, q1), o0);
}

struct LaneWords {
    const float* w;
    __device__ __forceinline__ float operator()(int k) const { return w[k]; }
};

// one node (width x 96 bytes) into LDS: lane l < width * 6 copies 16 bytes
__device__ __forceinline__ void fetch_node(const uint32_t* __restrict__ nb, uint4* lds, int width, int lane)
{
    if (lane < width * (kSlotWords / 4))
        __builtin_amdgcn_global_load_lds(reinterpret_cast<const uint4*>(nb) + lane, lds, 16, 0, 0);
}

} // namespace
} // namespace fwn
