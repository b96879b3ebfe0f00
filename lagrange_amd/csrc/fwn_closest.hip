// Closest point on the mesh (unsigned distance) over the same tree as the winding-number
// engine: the query of lagrange::bvh::TriangleAABBTree::get_closest_point
// (modules/bvh/src/TriangleAABBTree.cpp:86-127), whose tree walk is AABB::get_closest_element
// (modules/bvh/src/AABB.cpp:187-250) and whose per-triangle distance is
// lagrange::point_triangle_squared_distance
// (modules/core/include/lagrange/utils/point_triangle_squared_distance.h), Eberly's region
// method evaluated in double.
//
// One wave64 walks the tree for 64 Morton-sorted points.  The wave stack holds (node, lane mask)
// entries as in the winding-number traversal; a lane takes part in a slot while the slot's box is
// nearer than the lane's best distance so far.  Leaf slots are evaluated before a node's children
// are pushed (to tighten the bounds early) and children are pushed farthest first, ordered by the
// box distance of each slot's first participating lane, so the nearest is walked next.  A slot that
// no participating lane's best reaches by its disk (a slab around the triangles: a box is fat where
// the surface runs askew, and deep inside a mesh the box walk opened nearly every leaf) is left out
// as a whole, which changes neither a mask nor a best distance anywhere else: the facet of an exact
// tie is the first in the walk's order, with or without the disks.  Inside a leaf bucket, a triangle
// is evaluated only for lanes whose best distance its vertex box does not exceed.
//
// Bound: issue and latency of the longest waves (points deep inside, whose 64 lanes' nearest
// triangles lie on all sides): 400,000 points over 200k triangles keep 3.3 waves of a compute unit in
// flight on average, and an average wave issues 87k vector and 52k scalar instructions.  Against the
// walk with double box distances from vector loads and no disks (333k and 330k), that call takes
// 4.1 ms instead of 43.2: 16.1 ms with the float box distances and record loads below, 12.7 with
// disks of single triangles, 4.3 with the disks of the inner slots, the rest by the blocks' order.
#include <hip/hip_runtime.h>

#include <cmath>

#include "fwn_internal.h"

namespace fwn {
namespace {

// Squared distance from q to the triangle (v0, v1, v2) and the parameters (s, t) of the closest
// point v0 + s (v1 - v0) + t (v2 - v0); every operation rounded as written (no contraction).
__device__ double tri_closest_f64(const float* __restrict__ tw, double qx, double qy, double qz, double& so,
                                  double& to)
{
#pragma clang fp contract(off)
    const double v0[3] = {tw[0], tw[1], tw[2]};
    const double v1[3] = {tw[3], tw[4], tw[5]};
    const double v2[3] = {tw[6], tw[7], tw[8]};
    const double q[3] = {qx, qy, qz};
    double df[3], e0[3], e1[3];
    for (int d = 0; d < 3; ++d) {
        df[d] = v0[d] - q[d];
        e0[d] = v1[d] - v0[d];
        e1[d] = v2[d] - v0[d];
    }
    const double a00 = e0[0] * e0[0] + e0[1] * e0[1] + e0[2] * e0[2];
    const double a01 = e0[0] * e1[0] + e0[1] * e1[1] + e0[2] * e1[2];
    const double a11 = e1[0] * e1[0] + e1[1] * e1[1] + e1[2] * e1[2];
    const double b0 = df[0] * e0[0] + df[1] * e0[1] + df[2] * e0[2];
    const double b1 = df[0] * e1[0] + df[1] * e1[1] + df[2] * e1[2];
    const double c = df[0] * df[0] + df[1] * df[1] + df[2] * df[2];
    const double det = fabs(a00 * a11 - a01 * a01);
    double s = a01 * b1 - a11 * b0;
    double t = a01 * b0 - a00 * b1;
    double r;
    if (det < 1e-30) {
        // degenerate triangle: nearest of the three edges (v0 v1), (v0 v2), (v1 v2)
        const double* P[3][2] = {{v0, v1}, {v0, v2}, {v1, v2}};
        r = INFINITY;
        for (int k = 0; k < 3; ++k) {
            const double* A = P[k][0];
            const double* B = P[k][1];
            double ab[3], aq[3];
            for (int d = 0; d < 3; ++d) {
                ab[d] = B[d] - A[d];
                aq[d] = q[d] - A[d];
            }
            const double l2 = ab[0] * ab[0] + ab[1] * ab[1] + ab[2] * ab[2];
            const double tp = aq[0] * ab[0] + aq[1] * ab[1] + aq[2] * ab[2];
            double u = 0.0;
            if (!(tp <= 0.0 || l2 == 0.0)) u = tp > l2 ? 1.0 : tp / l2;
            double dd = 0.0;
            for (int d = 0; d < 3; ++d) {
                const double x = q[d] - (A[d] + u * ab[d]);
                dd += x * x;
            }
            if (dd < r) {
                r = dd;
                // express the point in (s, t) of the triangle: edge k interpolates its endpoints
                so = k == 0 ? u : (k == 1 ? 0.0 : 1.0 - u);
                to = k == 0 ? 0.0 : (k == 1 ? u : u);
            }
        }
        return r;
    }
    if (s + t <= det) {
        if (s < 0.0) {
            if (t < 0.0) { // region 4
                if (b0 < 0.0) {
                    t = 0.0;
                    if (-b0 >= a00) {
                        s = 1.0;
                        r = a00 + 2.0 * b0 + c;
                    } else {
                        s = -b0 / a00;
                        r = b0 * s + c;
                    }
                } else {
                    s = 0.0;
                    if (b1 >= 0.0) {
                        t = 0.0;
                        r = c;
                    } else if (-b1 >= a11) {
                        t = 1.0;
                        r = a11 + 2.0 * b1 + c;
                    } else {
                        t = -b1 / a11;
                        r = b1 * t + c;
                    }
                }
            } else { // region 3: edge s = 0
                s = 0.0;
                if (b1 >= 0.0) {
                    t = 0.0;
                    r = c;
                } else if (-b1 >= a11) {
                    t = 1.0;
                    r = a11 + 2.0 * b1 + c;
                } else {
                    t = -b1 / a11;
                    r = b1 * t + c;
                }
            }
        } else if (t < 0.0) { // region 5: edge t = 0
            t = 0.0;
            if (b0 >= 0.0) {
                s = 0.0;
                r = c;
            } else if (-b0 >= a00) {
                s = 1.0;
                r = a00 + 2.0 * b0 + c;
            } else {
                s = -b0 / a00;
                r = b0 * s + c;
            }
        } else { // region 0: interior
            const double inv = 1.0 / det;
            s = s * inv;
            t = t * inv;
            r = s * (a00 * s + a01 * t + 2.0 * b0) + t * (a01 * s + a11 * t + 2.0 * b1) + c;
        }
    } else {
        if (s < 0.0) { // region 2
            const double tmp0 = a01 + b0, tmp1 = a11 + b1;
            if (tmp1 > tmp0) {
                const double numer = tmp1 - tmp0, denom = a00 - 2.0 * a01 + a11;
                if (numer >= denom) {
                    s = 1.0;
                    t = 0.0;
                    r = a00 + 2.0 * b0 + c;
                } else {
                    s = numer / denom;
                    t = 1.0 - s;
                    r = s * (a00 * s + a01 * t + 2.0 * b0) + t * (a01 * s + a11 * t + 2.0 * b1) + c;
                }
            } else {
                s = 0.0;
                if (tmp1 <= 0.0) {
                    t = 1.0;
                    r = a11 + 2.0 * b1 + c;
                } else if (b1 >= 0.0) {
                    t = 0.0;
                    r = c;
                } else {
                    t = -b1 / a11;
                    r = b1 * t + c;
                }
            }
        } else if (t < 0.0) { // region 6
            const double tmp0 = a01 + b1, tmp1 = a00 + b0;
            if (tmp1 > tmp0) {
                const double numer = tmp1 - tmp0, denom = a00 - 2.0 * a01 + a11;
                if (numer >= denom) {
                    t = 1.0;
                    s = 0.0;
                    r = a11 + 2.0 * b1 + c;
                } else {
                    t = numer / denom;
                    s = 1.0 - t;
                    r = s * (a00 * s + a01 * t + 2.0 * b0) + t * (a01 * s + a11 * t + 2.0 * b1) + c;
                }
            } else {
                t = 0.0;
                if (tmp1 <= 0.0) {
                    s = 1.0;
                    r = a00 + 2.0 * b0 + c;
                } else if (b0 >= 0.0) {
                    s = 0.0;
                    r = c;
                } else {
                    s = -b0 / a00;
                    r = b0 * s + c;
                }
            }
        } else { // region 1: edge s + t = 1
            const double numer = a11 + b1 - a01 - b0;
            if (numer <= 0.0) {
                s = 0.0;
                t = 1.0;
                r = a11 + 2.0 * b1 + c;
            } else {
                const double denom = a00 - 2.0 * a01 + a11;
                if (numer >= denom) {
                    s = 1.0;
                    t = 0.0;
                    r = a00 + 2.0 * b0 + c;
                } else {
                    s = numer / denom;
                    t = 1.0 - s;
                    r = s * (a00 * s + a01 * t + 2.0 * b0) + t * (a01 * s + a11 * t + 2.0 * b1) + c;
                }
            }
        }
    }
    so = s;
    to = t;
    return r < 0.0 ? 0.0 : r;
}

// v0 + s (v1 - v0) + t (v2 - v0) in double, rounded as written
__device__ __forceinline__ void closest_on(const float* __restrict__ tw, double s, double t, double* cp)
{
#pragma clang fp contract(off)
    for (int d = 0; d < 3; ++d) {
        const double v0 = tw[d];
        cp[d] = v0 + s * ((double)tw[3 + d] - v0) + t * ((double)tw[6 + d] - v0);
    }
}

// squared distance from q to the box (lo[3], hi[3]); 0 inside
__device__ __forceinline__ double box_dist2(const float* __restrict__ b, double qx, double qy, double qz)
{
    const double q[3] = {qx, qy, qz};
    double r = 0.0;
    for (int d = 0; d < 3; ++d) {
        const double lo = b[d], hi = b[3 + d];
        const double x = q[d] < lo ? lo - q[d] : (q[d] > hi ? q[d] - hi : 0.0);
        r = fma(x, x, r);
    }
    return r;
}

// Squared distance from q to the box of the triangle's vertices: a lower bound on the squared
// distance to the triangle
__device__ __forceinline__ double tri_box_dist2(const float* __restrict__ tw, double qx, double qy, double qz)
{
    float b[6];
    for (int d = 0; d < 3; ++d) {
        b[d] = fminf(fminf(tw[d], tw[3 + d]), tw[6 + d]);
        b[3 + d] = fmaxf(fmaxf(tw[d], tw[3 + d]), tw[6 + d]);
    }
    return box_dist2(b, qx, qy, qz);
}

// the same in float, within 3e-7 of it
__device__ __forceinline__ float tri_box_dist2f(const float* __restrict__ tw, float fx, float fy, float fz)
{
    const float f[3] = {fx, fy, fz};
    float r = 0.0f;
    for (int d = 0; d < 3; ++d) {
        const float lo = fminf(fminf(tw[d], tw[3 + d]), tw[6 + d]), hi = fmaxf(fmaxf(tw[d], tw[3 + d]), tw[6 + d]);
        const float x = fmaxf(fmaxf(lo - f[d], f[d] - hi), 0.0f);
        r = fmaf(x, x, r);
    }
    return r;
}

typedef float v16f __attribute__((ext_vector_type(16)));
typedef v16f v16f_a4 __attribute__((aligned(4)));

// A lane's FP64 best distance as float bounds: a float box distance below `lo` is certainly below
// the best, one above `hi` certainly not (the float distance is within 3e-7 of the double one, the
// bounds leave 1e-6); between them, and where the best is too small or too large for that, the
// double distance decides.
struct BestBounds {
    float lo = INFINITY, hi = INFINITY;
    __device__ __forceinline__ void set(double best)
    {
        const float b = (float)best;
        lo = b > 1e-30f && b < 1e38f ? b * (1.0f - 1e-6f) : 0.0f;
        hi = b < 1e38f ? (b > 1e-30f ? b * (1.0f + 1e-6f) : 1e-29f) : INFINITY;
    }
};

// Lower bound on the squared distance from q to what a slot's disk holds (its triangles: within t of
// the plane through c normal to n, and within R of the axis), less the float arithmetic's error.  With
// r = c - q, h its part along n and rho the one along the plane, the distance is at least |h| - t along
// n and rho - R along the plane.  The float results are within 2.4e-6 |r|^2 (six roundings of relative
// 2^-24 in h, three in |r|^2, and (rho - R) / rho <= 1 for the square root); 4e-6 |r|^2 is taken off,
// and 1e-13 R^2 for the rounding of the exact evaluation this stands for.  t = R = infinity bounds
// nothing, and NaN (overflow) compares as no bound.
__device__ __forceinline__ float disk_bound(float t, float cx, float cy, float cz, float R, float nx, float ny,
                                            float nz, float fx, float fy, float fz)
{
    const float rx = cx - fx, ry = cy - fy, rz = cz - fz;
    const float r2 = fmaf(rx, rx, fmaf(ry, ry, rz * rz));
    const float hc = fmaf(rx, nx, fmaf(ry, ny, rz * nz));
    const float h = fmaxf(fabsf(hc) - t, 0.0f);
    const float out = fmaxf(__builtin_amdgcn_sqrtf(fmaxf(fmaf(-hc, hc, r2), 0.0f)) - R, 0.0f);
    return fmaf(-4e-6f, r2, fmaf(-1e-13f * R, R, fmaf(out, out, h * h)));
}

// One wave per 64 sorted points; W = tree width.  Decisions (which lanes take part in a slot, the
// order of the children, which triangle wins) are those of the double arithmetic throughout; float
// distances settle all but the closest calls: 14 instructions a box instead of 40, its operands
// straight from scalar registers.  A slot's box, link and disk are one 64-byte scalar load.
// (Measured and not taken: the disks of a node's leaves all tested before any is evaluated, 13.1 ms
// for 12.7; one selected division and evaluation in place of the region branches, 4.80 for 4.28.)
template <int NB, int W>
__global__ __launch_bounds__(64) void k_closest(const float* __restrict__ boxes, const uint32_t* __restrict__ tris,
                                                int32_t root, int32_t root_ns, const float* __restrict__ Q,
                                                const uint32_t* __restrict__ perm, int64_t nQ,
                                                double* __restrict__ d2_out, int32_t* __restrict__ tri_out,
                                                double* __restrict__ cp_out, int32_t* __restrict__ flag)
{
    const int lane = threadIdx.x;
    // runs of 256 waves: the expensive waves lie together (400k points: 4.20 ms in one run per XCD,
    // 3.96 in runs of 64, 3.88 of 256, 4.25 of 1,024)
    const int64_t batch = xcd_remap_runs(blockIdx.x, gridDim.x, 256u);
    const int64_t jpos = batch * 64 + lane;
    const bool valid = jpos < nQ;
    const uint32_t orig = valid ? perm[jpos] : 0u;
    const float fx = valid ? Q[3 * (int64_t)orig] : 0.0f;
    const float fy = valid ? Q[3 * (int64_t)orig + 1] : 0.0f;
    const float fz = valid ? Q[3 * (int64_t)orig + 2] : 0.0f;
    const double qx = fx, qy = fy, qz = fz;
    double best = INFINITY, bs = 0.0, bt = 0.0;
    BestBounds bb;
    int32_t btri = -1;
    if (root >= 0) {
        WaveStack<NB> S;
        S.push(0, lane, ((uint32_t)root << 4) | (uint32_t)root_ns, __ballot(valid));
        int sp = 1;
        bool overflow = false;
        while (sp > 0) {
            --sp;
            uint32_t e;
            uint64_t mk;
            S.pop(sp, e, mk);
            const float* nbx = boxes + (size_t)(e >> 4) * (size_t)(W * kBoxWords);
            float db[W];     // squared box distances
            int32_t link[W]; // negative: a leaf, -1: unoccupied (its box is zeros)
            v16f rec[W];
#pragma unroll
            for (int s = 0; s < W; ++s) {
                const v16f b = *reinterpret_cast<const v16f_a4*>(nbx + kBoxWords * s); // one scalar load
                const float x = fmaxf(fmaxf(b[0] - fx, fx - b[3]), 0.0f);
                const float y = fmaxf(fmaxf(b[1] - fy, fy - b[4]), 0.0f);
                const float z = fmaxf(fmaxf(b[2] - fz, fz - b[5]), 0.0f);
                db[s] = fmaf(z, z, fmaf(y, y, x * x));
                link[s] = __float_as_int(b[6]);
                rec[s] = b;
            }
            // lanes of the node whose double box distance to slot s is below their best
            auto nearer = [&](int s, float d) __attribute__((always_inline)) -> uint64_t {
                const uint64_t yes = __ballot(d < bb.lo);
                const uint64_t open = mk & ~yes & ~__ballot(d > bb.hi);
                if (open == 0ull) return mk & yes;
                return mk & __ballot(box_dist2(nbx + kBoxWords * s, qx, qy, qz) < best);
            };
            // of lanes m, those whose best the slot's disk may reach
            auto reached = [&](int s, uint64_t m) __attribute__((always_inline)) -> uint64_t {
                const v16f b = rec[s];
                const float d = disk_bound(b[7], b[8], b[9], b[10], b[11], b[12], b[13], b[14], fx, fy, fz);
                return m & ~__ballot(d > bb.hi);
            };
            // leaf slots first
#pragma unroll
            for (int s = 0; s < W; ++s) {
                if (link[s] >= -1) continue;
                uint64_t lanes = nearer(s, db[s]);
                if (lanes == 0ull) continue;
                lanes = reached(s, lanes);
                if (lanes == 0ull) continue;
                const int32_t first = (int32_t)(((uint32_t)link[s] & ~FWN_LINK_LEAF) >> 3);
                const int32_t cnt = (link[s] & 7) + 1;
                for (int32_t t = first; t < first + cnt; ++t) {
                    const float* tw = reinterpret_cast<const float*>(tris + (size_t)t * kTriWords);
                    // a triangle whose box is farther than the lane's best cannot improve it; the 1e-12
                    // margin is far above the rounding of the bound and of the exact evaluation, so the
                    // nearest triangle (and the first of equally near ones) is always evaluated and results
                    // do not change.  Float distances settle all but the closest calls, as for slots (16.7M
                    // grid points, F = 953,344, leaf 8: 29.7 ms by double distances alone, 27.6 so).
                    // A single triangle's box is the slot's, already compared
                    uint64_t m = lanes;
                    if (cnt > 1) {
                        const float d = tri_box_dist2f(tw, fx, fy, fz);
                        m &= ~__ballot(d > bb.hi);
                        if ((m & ~__ballot(d < bb.lo)) != 0ull)
                            m &= __ballot(tri_box_dist2(tw, qx, qy, qz) <= best * (1.0 + 1e-12));
                    }
                    if (m == 0ull) continue;
                    if (__builtin_amdgcn_inverse_ballot_w64(m)) {
                        double ss, tt;
                        const double d = tri_closest_f64(tw, qx, qy, qz, ss, tt);
                        if (d < best) {
                            best = d;
                            btri = t;
                            bs = ss;
                            bt = tt;
                            bb.set(best);
                        }
                    }
                }
            }
            // inner slots: pushed farthest first so the nearest is walked next, ordered by the box
            // distance (rounded to float, the later slot first among equals) that the slot's first
            // participating lane sees (the wave's points are close together; the order only steers
            // the walk).  A slot goes to the stack position its rank gives
            uint64_t pm[W];
            int32_t key[W]; // bits of a non-negative float; -1: not pushed
            int n = 0;
#pragma unroll
            for (int s = 0; s < W; ++s) {
                pm[s] = link[s] >= 0 ? nearer(s, db[s]) : 0ull;
                if (pm[s] != 0ull && reached(s, pm[s]) == 0ull) pm[s] = 0ull;
                key[s] = pm[s] ? __builtin_amdgcn_readlane(__float_as_int(db[s]), (int)__builtin_ctzll(pm[s])) : -1;
                n += pm[s] ? 1 : 0;
            }
            if (n == 0) continue;
            if (n > 1) {
                // float distances a few units apart may be in the other order in double (a zero is exact)
                bool close = false;
#pragma unroll
                for (int s = 0; s < W; ++s)
#pragma unroll
                    for (int t = s + 1; t < W; ++t)
                        close |= key[s] >= 0 && key[t] >= 0 && (key[s] | key[t]) != 0 &&
                                 (uint32_t)(key[t] - key[s] + 32) <= 64u;
                if (close) {
#pragma unroll
                    for (int s = 0; s < W; ++s)
                        if (pm[s] != 0ull)
                            key[s] = __builtin_amdgcn_readlane(
                                __float_as_int((float)box_dist2(nbx + kBoxWords * s, qx, qy, qz)),
                                (int)__builtin_ctzll(pm[s]));
                }
            }
            if (sp + n <= WaveStack<NB>::kCap) {
#pragma unroll
                for (int s = 0; s < W; ++s) {
                    int rank = 0;
#pragma unroll
                    for (int t = 0; t < W; ++t)
                        if (t != s) rank += (t > s ? key[t] >= key[s] : key[t] > key[s]) ? 1 : 0;
                    if (pm[s] != 0ull) S.push(sp + rank, lane, (uint32_t)link[s], pm[s]); // (child << 4) | its slots
                }
                sp += n;
            } else {
                overflow = true;
            }
        }
        if (overflow && lane == 0) atomicOr(flag, 1);
    }
    if (valid) {
        d2_out[orig] = best;
        int32_t fid = -1;
        double cp[3] = {NAN, NAN, NAN};
        if (btri >= 0) {
            fid = (int32_t)tris[(size_t)btri * kTriWords + FWN_T_FACET];
            closest_on(reinterpret_cast<const float*>(tris + (size_t)btri * kTriWords), bs, bt, cp);
        }
        tri_out[orig] = fid;
        if (cp_out) {
            cp_out[3 * (int64_t)orig] = cp[0];
            cp_out[3 * (int64_t)orig + 1] = cp[1];
            cp_out[3 * (int64_t)orig + 2] = cp[2];
        }
    }
}

} // namespace

void run_closest(Engine& e, const float* Q, int64_t nQ, double* d2, int32_t* tri, double* cp, bool dev)
{
    if (e.n_meshes != 1) fail(FWN_INVALID_ARGUMENT, "closest point needs a single-mesh engine");
    if (nQ < 0) fail(FWN_INVALID_ARGUMENT, "negative point count");
    if (nQ == 0) return;
    if (!Q || !d2 || !tri) fail(FWN_INVALID_ARGUMENT, "NULL points or output");
    const int banks = stack_banks(e.width, e.max_depth);
    if (banks == 0) fail(FWN_LIMIT_EXCEEDED, "tree deeper than the traversal stack supports");
    hipStream_t s = e.stream;
    const float* dQ = Q;
    double* dD = d2;
    int32_t* dT = tri;
    double* dC = cp;
    if (!dev) {
        e.q_in.reserve(sizeof(float) * 3 * nQ);
        e.d_d2.reserve(sizeof(double) * nQ);
        e.d_tri.reserve(sizeof(int32_t) * nQ);
        FWN_HIP(hipMemcpyAsync(e.q_in.p, Q, sizeof(float) * 3 * nQ, hipMemcpyHostToDevice, s));
        dQ = e.q_in.as<float>();
        dD = e.d_d2.as<double>();
        dT = e.d_tri.as<int32_t>();
        if (cp) {
            e.d_cp.reserve(sizeof(double) * 3 * nQ);
            dC = e.d_cp.as<double>();
        }
    }
    const uint32_t* perm = sort_points_single(e, dQ, nQ);
    e.q_flag.reserve(3 * sizeof(int32_t));
    int32_t* dflag = e.q_flag.as<int32_t>();
    FWN_HIP(hipMemsetAsync(dflag, 0, sizeof(int32_t), s));
    const int64_t nb = (nQ + 63) / 64;
    if (nb > INT32_MAX) fail(FWN_LIMIT_EXCEEDED, "too many point batches");
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)nb), dim3(64), 0, s, e.boxes.as<float>(), e.tris.as<uint32_t>(),
                           e.h_roots[0], e.h_roots[1], dQ, perm, nQ, dD, dT, dC, dflag);
        FWN_LAUNCH_CHECK("k_closest");
    };
    if (e.width == 4) go(banks == 1 ? k_closest<1, 4> : k_closest<3, 4>);
    else if (e.width == 2) go(banks == 1 ? k_closest<1, 2> : k_closest<3, 2>);
    else go(banks == 1 ? k_closest<1, 8> : k_closest<3, 8>);
    int32_t h_flag = 0;
    FWN_HIP(hipMemcpyAsync(&h_flag, dflag, sizeof(int32_t), hipMemcpyDeviceToHost, s));
    if (!dev) {
        FWN_HIP(hipMemcpyAsync(d2, dD, sizeof(double) * nQ, hipMemcpyDeviceToHost, s));
        FWN_HIP(hipMemcpyAsync(tri, dT, sizeof(int32_t) * nQ, hipMemcpyDeviceToHost, s));
        if (cp) FWN_HIP(hipMemcpyAsync(cp, dC, sizeof(double) * 3 * nQ, hipMemcpyDeviceToHost, s));
    }
    FWN_HIP(hipStreamSynchronize(s));
    if (h_flag) fail(FWN_LIMIT_EXCEEDED, "traversal stack overflow");
}

} // namespace fwn
