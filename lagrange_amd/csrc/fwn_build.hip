// GPU tree build for the fast winding number engine (gfx950).
//
// Replaces UT_SolidAngle<float,float>::init, called by the reference at
// modules/winding/src/FastWindingNumber.cpp:57 after the float/int copy of :39-52.  That
// dependency builds a 4-ary box-area BVH on the CPU and accumulates order-2 moments per child;
// here the same per-node quantities are produced by a Morton-code LBVH built on the GPU:
//
//   k_tri_setup     centroids, per-mesh centroid/vertex boxes (wave-reduced atomics), input checks
//   k_box_final     per-mesh Morton box, query box, FP64 near-field distance tau
//   k_tri_keys      key = mesh << 32 | 30-bit Morton code of the centroid
//   radix sort      (fwn_sort.hip)
//   k_karras        binary radix tree over the sorted keys (Karras 2012), ties broken by index
//   k_find_roots    the node covering exactly one mesh's triangles is that mesh's root
//   k_leaf_records  sorted triangle records + FP32 per-triangle moments
//   k_merge_mid, k_merge_top
//                   SAH trees: moments of subtrees of up to 1,024 triangles, a workgroup each, then
//                   of the nodes above them; each node merges its two children, FP32 for small
//                   nodes and FP64 for nodes with >= fp64_moment_min triangles
//   k_node_depth, k_depth_bucket, k_merge_level
//                   Morton trees: the same merges level by level from the deepest internal nodes up
//                   (kernel boundaries order the levels)
//   k_bottom_up     the same merges by an arrival-counter walk to the roots, for trees deeper
//                   than kMaxLevels
//   k_collapse_*    level by level, each wide node takes the binary node's children and
//                   repeatedly opens the largest non-leaf slot until it has tree_width slots (Morton
//                   trees), or whole binary levels (SAH trees)
//   k_write_slots   FP64 records -> the 24-word FP32 slot format of fwn.h, plus each slot's 64-byte
//                   record for distance queries: its box (6 floats, rounded outward) and link
//   k_slot_disks    each slot's disk (a slab around its triangles) for distance queries
//
// Several meshes are built together: their keys carry the mesh id above the Morton bits, so
// each mesh is one subtree of a single radix tree and every kernel runs once for all meshes.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "fwn_internal.h"

namespace fwn {

namespace {

constexpr int BT = 256; // threads per block for build kernels

__device__ __forceinline__ int mesh_of(const int64_t* off, int M, int64_t t)
{
    // largest m with off[m] <= t (off has M+1 entries, non-decreasing)
    int lo = 0, hi = M - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (off[mid] <= t) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

__global__ void k_init(int32_t* __restrict__ boxes, int M, int32_t* __restrict__ err)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    // 12 ints per mesh: cen lo[3] hi[3], vert lo[3] hi[3] (order-preserving ints)
    if (i < 12 * M) {
        int k = i % 12;
        bool is_lo = (k % 6) < 3;
        boxes[i] = is_lo ? INT32_MAX : INT32_MIN;
    }
    if (i == 0) *err = 0;
}

__device__ __forceinline__ float wave_min(float v)
{
    for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o));
    return v;
}
__device__ __forceinline__ float wave_max(float v)
{
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    return v;
}

// Per-triangle centroid (and box, for the SAH builder), per-mesh centroid and vertex bounds.
// The bounds are reduced per wave, then across the workgroup's 16 waves in LDS, so a
// single-mesh block issues 12 atomics; a wave that straddles a mesh boundary falls back to
// per-lane atomics.
constexpr int TS = 1024; // threads per k_tri_setup block
__global__ __launch_bounds__(TS) void k_tri_setup(const float* __restrict__ V, const int32_t* __restrict__ F,
                                                  int64_t nF, const int64_t* __restrict__ f_off,
                                                  const int64_t* __restrict__ v_off, int M,
                                                  float* __restrict__ cen, int32_t* __restrict__ boxes,
                                                  float* __restrict__ tbox, int32_t* __restrict__ err)
{
    __shared__ int32_t part[TS / 64][13]; // per wave: mesh (-1: nothing to add), 12 bound words
    int64_t t = (int64_t)blockIdx.x * TS + threadIdx.x;
    bool valid = t < nF;
    int m = valid ? mesh_of(f_off, M, t) : 0;
    float c[3] = {0, 0, 0}, lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    if (valid) {
        int64_t nv = v_off[m + 1] - v_off[m];
        float v[3][3];
        for (int k = 0; k < 3; ++k) {
            int32_t idx = F[3 * t + k];
            if (idx < 0 || (int64_t)idx >= nv) {
                atomicOr(err, 1);
                idx = 0;
                if (nv == 0) {
                    v[k][0] = v[k][1] = v[k][2] = 0.0f;
                    continue;
                }
            }
            int64_t g = v_off[m] + idx;
            v[k][0] = V[3 * g];
            v[k][1] = V[3 * g + 1];
            v[k][2] = V[3 * g + 2];
        }
        for (int d = 0; d < 3; ++d) {
            c[d] = ((v[0][d] + v[1][d]) + v[2][d]) * (1.0f / 3.0f);
            lo[d] = fminf(v[0][d], fminf(v[1][d], v[2][d]));
            hi[d] = fmaxf(v[0][d], fmaxf(v[1][d], v[2][d]));
            if (!isfinite(v[0][d]) || !isfinite(v[1][d]) || !isfinite(v[2][d])) atomicOr(err, 2);
            cen[3 * t + d] = c[d];
            if (tbox) {
                tbox[6 * t + d] = lo[d];
                tbox[6 * t + 3 + d] = hi[d];
            }
        }
    }
    float clo[3], chi[3];
    for (int d = 0; d < 3; ++d) {
        clo[d] = valid ? c[d] : INFINITY;
        chi[d] = valid ? c[d] : -INFINITY;
    }
    const int w = threadIdx.x >> 6;
    int m0 = __builtin_amdgcn_readfirstlane(m);
    const bool any = __ballot(valid) != 0ull;
    bool same = __ballot(valid && m != m0) == 0ull;
    if (same) {
        for (int d = 0; d < 3; ++d) {
            clo[d] = wave_min(clo[d]);
            chi[d] = wave_max(chi[d]);
            lo[d] = wave_min(lo[d]);
            hi[d] = wave_max(hi[d]);
        }
        if ((threadIdx.x & 63) == 0) {
            part[w][0] = any ? m0 : -1;
            for (int d = 0; d < 3; ++d) {
                part[w][1 + d] = f2ord(clo[d]);
                part[w][4 + d] = f2ord(chi[d]);
                part[w][7 + d] = f2ord(lo[d]);
                part[w][10 + d] = f2ord(hi[d]);
            }
        }
    } else {
        if ((threadIdx.x & 63) == 0) part[w][0] = -1;
    }
    __syncthreads();
    if (threadIdx.x < 12) { // word k of the bounds: min for k % 6 < 3, max otherwise
        const int k = threadIdx.x;
        const bool is_min = (k % 6) < 3;
        int cur = -1;
        int32_t acc = 0;
        for (int ww = 0; ww < TS / 64; ++ww) {
            const int mw = part[ww][0];
            if (mw < 0) continue;
            const int32_t v = part[ww][1 + k];
            if (mw != cur) {
                if (cur >= 0) {
                    if (is_min) atomicMin(boxes + 12 * cur + k, acc);
                    else atomicMax(boxes + 12 * cur + k, acc);
                }
                cur = mw;
                acc = v;
            } else {
                acc = is_min ? min(acc, v) : max(acc, v);
            }
        }
        if (cur >= 0) {
            if (is_min) atomicMin(boxes + 12 * cur + k, acc);
            else atomicMax(boxes + 12 * cur + k, acc);
        }
    }
    if (!same && valid) {
        int32_t* b = boxes + 12 * m;
        for (int d = 0; d < 3; ++d) {
            atomicMin(b + d, f2ord(clo[d]));
            atomicMax(b + 3 + d, f2ord(chi[d]));
            atomicMin(b + 6 + d, f2ord(lo[d]));
            atomicMax(b + 9 + d, f2ord(hi[d]));
        }
    }
}

// per mesh: cinfo = centroid lo[3], inv[3]; minfo = query lo[3], inv[3], tau, 0
__global__ void k_box_final(const int32_t* __restrict__ boxes, int M, float rel, float* __restrict__ cinfo,
                            float* __restrict__ minfo)
{
    int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= M) return;
    const int32_t* b = boxes + 12 * m;
    bool empty = b[0] == INT32_MAX;
    float diag2 = 0.0f;
    for (int d = 0; d < 3; ++d) {
        float clo = empty ? 0.0f : ord2f(b[d]), chi = empty ? 0.0f : ord2f(b[3 + d]);
        float vlo = empty ? 0.0f : ord2f(b[6 + d]), vhi = empty ? 0.0f : ord2f(b[9 + d]);
        float ce = chi - clo, ve = vhi - vlo;
        cinfo[6 * m + d] = clo;
        cinfo[6 * m + 3 + d] = (ce > 0.0f) ? 1.0f / ce : 0.0f;
        minfo[8 * m + d] = vlo;
        minfo[8 * m + 3 + d] = (ve > 0.0f) ? 1.0f / ve : 0.0f;
        diag2 += ve * ve;
    }
    minfo[8 * m + 6] = rel * sqrtf(diag2);
    minfo[8 * m + 7] = 0.0f;
}

__global__ __launch_bounds__(BT) void k_tri_keys(const float* __restrict__ cen, int64_t nF,
                                                 const int64_t* __restrict__ f_off, int M,
                                                 const float* __restrict__ cinfo, uint64_t* __restrict__ keys,
                                                 uint32_t* __restrict__ vals)
{
    int64_t t = (int64_t)blockIdx.x * BT + threadIdx.x;
    if (t >= nF) return;
    int m = mesh_of(f_off, M, t);
    const float* ci = cinfo + 6 * m;
    uint32_t mc = morton30(cen[3 * t], cen[3 * t + 1], cen[3 * t + 2], ci, ci + 3);
    keys[t] = ((uint64_t)(uint32_t)m << 32) | mc;
    vals[t] = (uint32_t)t;
}

__device__ __forceinline__ int delta(const uint64_t* __restrict__ k, int64_t n, int64_t i, int64_t j)
{
    if (j < 0 || j >= n) return -1;
    uint64_t a = k[i], b = k[j];
    if (a == b) return 64 + __clz((uint32_t)(i ^ j));
    return __clzll(a ^ b);
}

// unified node ids: internal i in [0, n-1), leaf j -> (n-1) + j
__global__ __launch_bounds__(BT) void k_karras(const uint64_t* __restrict__ keys, int64_t n,
                                               int32_t* __restrict__ left, int32_t* __restrict__ right,
                                               int32_t* __restrict__ parent, int32_t* __restrict__ first,
                                               int32_t* __restrict__ last)
{
    int64_t i = (int64_t)blockIdx.x * BT + threadIdx.x;
    if (i >= n - 1) return;
    int d = (delta(keys, n, i, i + 1) - delta(keys, n, i, i - 1)) >= 0 ? 1 : -1;
    int dmin = delta(keys, n, i, i - d);
    int64_t lmax = 2;
    while (delta(keys, n, i, i + lmax * d) > dmin) lmax <<= 1;
    int64_t l = 0;
    for (int64_t t = lmax >> 1; t >= 1; t >>= 1)
        if (delta(keys, n, i, i + (l + t) * d) > dmin) l += t;
    int64_t j = i + l * d;
    int dnode = delta(keys, n, i, j);
    int64_t s = 0;
    int64_t t = l;
    do {
        t = (t + 1) >> 1;
        if (delta(keys, n, i, i + (s + t) * d) > dnode) s += t;
    } while (t > 1);
    int64_t gamma = i + s * d + (d < 0 ? -1 : 0);
    int64_t lo = i < j ? i : j, hi = i < j ? j : i;
    int32_t lc = (lo == gamma) ? (int32_t)(n - 1 + gamma) : (int32_t)gamma;
    int32_t rc = (hi == gamma + 1) ? (int32_t)(n - 1 + gamma + 1) : (int32_t)(gamma + 1);
    left[i] = lc;
    right[i] = rc;
    parent[lc] = (int32_t)i;
    parent[rc] = (int32_t)i;
    first[i] = (int32_t)lo;
    last[i] = (int32_t)hi;
}

__global__ void k_fill_i32(int32_t* __restrict__ p, int64_t n, int32_t v)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

__global__ void k_gather_i32(const int32_t* __restrict__ from, const int32_t* __restrict__ at, int32_t n,
                             int32_t* __restrict__ to)
{
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) to[i] = from[at[i]];
}

__global__ __launch_bounds__(BT) void k_find_roots(const int32_t* __restrict__ first, const int32_t* __restrict__ last,
                                                   int64_t n, const uint64_t* __restrict__ keys,
                                                   const int64_t* __restrict__ f_off, int M,
                                                   int32_t* __restrict__ root_bin, uint8_t* __restrict__ is_root)
{
    int64_t i = (int64_t)blockIdx.x * BT + threadIdx.x;
    if (i < n - 1) {
        int m = (int)(keys[first[i]] >> 32);
        if (first[i] == f_off[m] && (int64_t)last[i] == f_off[m + 1] - 1) {
            root_bin[m] = (int32_t)i;
            is_root[i] = 1;
        }
    }
    if (i < M && f_off[i + 1] - f_off[i] == 1) {
        int64_t u = n - 1 + f_off[i];
        root_bin[i] = (int32_t)u;
        is_root[u] = 1;
    }
}

// ---- moments ------------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ void tri_record(const float (&v)[3][3], double* __restrict__ r)
{
    T e1[3], e2[3], c[3];
    for (int d = 0; d < 3; ++d) {
        e1[d] = (T)v[1][d] - (T)v[0][d];
        e2[d] = (T)v[2][d] - (T)v[0][d];
        c[d] = (((T)v[0][d] + (T)v[1][d]) + (T)v[2][d]) * (T)(1.0 / 3.0);
    }
    T N[3] = {(T)0.5 * (e1[1] * e2[2] - e1[2] * e2[1]), (T)0.5 * (e1[2] * e2[0] - e1[0] * e2[2]),
              (T)0.5 * (e1[0] * e2[1] - e1[1] * e2[0])};
    T A = sqrt(N[0] * N[0] + N[1] * N[1] + N[2] * N[2]);
    T C[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
    for (int k = 0; k < 3; ++k) {
        T e[3] = {(T)v[k][0] - c[0], (T)v[k][1] - c[1], (T)v[k][2] - c[2]};
        for (int j = 0; j < 3; ++j)
            for (int jj = 0; jj < 3; ++jj) C[j][jj] += e[j] * e[jj] * (T)(1.0 / 12.0);
    }
    r[R_A] = A;
    for (int d = 0; d < 3; ++d) {
        r[R_P + d] = c[d];
        r[R_N + d] = N[d];
        r[R_LO + d] = fminf(v[0][d], fminf(v[1][d], v[2][d]));
        r[R_HI + d] = fmaxf(v[0][d], fmaxf(v[1][d], v[2][d]));
    }
    for (int k = 0; k < 9; ++k) r[R_M1 + k] = 0.0;
    const int SI[10][3] = {{0, 0, 0}, {1, 1, 1}, {2, 2, 2}, {0, 0, 1}, {0, 0, 2},
                           {1, 1, 0}, {1, 1, 2}, {2, 2, 0}, {2, 2, 1}, {0, 1, 2}};
    for (int s = 0; s < 10; ++s) {
        int a = SI[s][0], b = SI[s][1], cc = SI[s][2];
        r[R_S + s] = (C[a][b] * N[cc] + C[b][cc] * N[a] + C[cc][a] * N[b]) * (T)(1.0 / 3.0);
    }
}

// parent record from two child records, each about its own centroid (parallel-axis shift)
template <typename T>
__device__ void merge2(const double* __restrict__ a, const double* __restrict__ b, double* __restrict__ o)
{
    const double* ch[2] = {a, b};
    T A = (T)a[R_A] + (T)b[R_A];
    T P[3];
    for (int d = 0; d < 3; ++d)
        P[d] = (A > (T)0) ? ((T)a[R_A] * (T)a[R_P + d] + (T)b[R_A] * (T)b[R_P + d]) / A
                          : ((T)a[R_P + d] + (T)b[R_P + d]) * (T)0.5;
    T N[3] = {0, 0, 0}, M1[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0}, S[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    const int SI[10][3] = {{0, 0, 0}, {1, 1, 1}, {2, 2, 2}, {0, 0, 1}, {0, 0, 2},
                           {1, 1, 0}, {1, 1, 2}, {2, 2, 0}, {2, 2, 1}, {0, 1, 2}};
    for (int c = 0; c < 2; ++c) {
        const double* x = ch[c];
        T dl[3] = {(T)x[R_P] - P[0], (T)x[R_P + 1] - P[1], (T)x[R_P + 2] - P[2]};
        T xn[3] = {(T)x[R_N], (T)x[R_N + 1], (T)x[R_N + 2]};
        T xm[9];
        for (int k = 0; k < 9; ++k) xm[k] = (T)x[R_M1 + k];
        for (int i = 0; i < 3; ++i) N[i] += xn[i];
        for (int j = 0; j < 3; ++j)
            for (int i = 0; i < 3; ++i) M1[3 * j + i] += xm[3 * j + i] + dl[j] * xn[i];
        for (int s = 0; s < 10; ++s) {
            int p = SI[s][0], q = SI[s][1], r = SI[s][2];
            // Y_jk,i = d_j M1_ki + d_k M1_ji + d_j d_k N_i ; Sym(Y)_pqr = (Y_pq,r + Y_qr,p + Y_rp,q) / 3
            T y1 = dl[p] * xm[3 * q + r] + dl[q] * xm[3 * p + r] + dl[p] * dl[q] * xn[r];
            T y2 = dl[q] * xm[3 * r + p] + dl[r] * xm[3 * q + p] + dl[q] * dl[r] * xn[p];
            T y3 = dl[r] * xm[3 * p + q] + dl[p] * xm[3 * r + q] + dl[r] * dl[p] * xn[q];
            S[s] += (T)x[R_S + s] + (y1 + y2 + y3) * (T)(1.0 / 3.0);
        }
    }
    o[R_A] = A;
    for (int d = 0; d < 3; ++d) {
        o[R_P + d] = P[d];
        o[R_N + d] = N[d];
        o[R_LO + d] = fmin(a[R_LO + d], b[R_LO + d]);
        o[R_HI + d] = fmax(a[R_HI + d], b[R_HI + d]);
    }
    for (int k = 0; k < 9; ++k) o[R_M1 + k] = M1[k];
    for (int s = 0; s < 10; ++s) o[R_S + s] = S[s];
}

// Records and slots go through LDS on their way out where a thread makes one by itself: 64 lanes writing
// 256 bytes each touch a cache line per lane and store.  101,568 and 940,800 triangles: k_leaf_records 15
// and 99 us, 10 and 64 so; k_write_slots 25 and 216 us, 19 and 166 so (its reads through LDS too: 28 and 252).
constexpr int RT = 128;                  // threads (and records) of such a block
constexpr int kRecPad = kRecWords + 1;   // doubles per record in LDS: the rows start on different banks
__global__ __launch_bounds__(RT) void k_leaf_records(const uint32_t* __restrict__ vals, int64_t n,
                                                     const float* __restrict__ V, const int32_t* __restrict__ F,
                                                     const int64_t* __restrict__ f_off,
                                                     const int64_t* __restrict__ v_off, int M,
                                                     uint32_t* __restrict__ tris, double* __restrict__ rec)
{
    __shared__ double lds[RT * kRecPad];
    const int64_t j0 = (int64_t)blockIdx.x * RT, j = j0 + threadIdx.x;
    int64_t t = vals[min(j, n - 1)];
    int m = mesh_of(f_off, M, t);
    int64_t nv = v_off[m + 1] - v_off[m];
    float v[3][3];
    for (int k = 0; k < 3; ++k) {
        int32_t idx = F[3 * t + k];
        if (idx < 0 || (int64_t)idx >= nv) idx = 0; // reported by k_tri_setup
        int64_t g = v_off[m] + idx;
        for (int d = 0; d < 3; ++d) v[k][d] = (nv > 0) ? V[3 * g + d] : 0.0f;
    }
    if (j < n) {
        float tw[kTriWords] = {}; // a leaf's near-field thresholds are written with the slots
        for (int k = 0; k < 3; ++k)
            for (int d = 0; d < 3; ++d) tw[3 * k + d] = v[k][d];
        tw[FWN_T_FACET] = __uint_as_float((uint32_t)(t - f_off[m]));
        float4* o = reinterpret_cast<float4*>(tris + j * kTriWords);
        for (int k = 0; k < kTriWords; k += 4) o[k / 4] = make_float4(tw[k], tw[k + 1], tw[k + 2], tw[k + 3]);
    }
    tri_record<float>(v, lds + threadIdx.x * kRecPad);
    __syncthreads();
    const int words = (int)min((int64_t)RT, n - j0) * kRecWords;
    for (int k = threadIdx.x; k < words; k += RT) rec[(n - 1 + j0) * kRecWords + k] = lds[k + k / kRecWords];
}

__global__ __launch_bounds__(BT) void k_bottom_up(const int32_t* __restrict__ parent,
                                                  const int32_t* __restrict__ left,
                                                  const int32_t* __restrict__ right,
                                                  const int32_t* __restrict__ first, const int32_t* __restrict__ last,
                                                  const uint8_t* __restrict__ is_root, int64_t n,
                                                  int32_t fp64_min, double* rec, int32_t* visits)
{
    int64_t j = (int64_t)blockIdx.x * BT + threadIdx.x;
    if (j >= n) return;
    int64_t u = n - 1 + j;
    while (!is_root[u]) {
        int32_t p = parent[u];
        if (p < 0) return;
        __threadfence();
        if (atomicAdd(&visits[p], 1) == 0) return; // the sibling's thread finishes this node
        __threadfence();
        const double* a = rec + (int64_t)left[p] * kRecWords;
        const double* b = rec + (int64_t)right[p] * kRecWords;
        if (last[p] - first[p] + 1 >= fp64_min) merge2<double>(a, b, rec + (int64_t)p * kRecWords);
        else merge2<float>(a, b, rec + (int64_t)p * kRecWords);
        u = p;
    }
}

// ---- level-synchronous moments ------------------------------------------------------------------
constexpr int kMaxLevels = 512; // deeper trees (pathological splits) use the arrival-counter walk

// depth of each internal node below its mesh root; -1 for ids outside every mesh tree (unused
// ids, nodes above the mesh roots) and for nodes deeper than kMaxLevels (then *deep is set).
// Per-depth counts are gathered in LDS and added to hist once per block and depth.
__global__ __launch_bounds__(BT) void k_node_depth(const int32_t* __restrict__ parent,
                                                   const uint8_t* __restrict__ is_root, int64_t n_int,
                                                   int32_t* __restrict__ depth, int32_t* __restrict__ hist,
                                                   int32_t* __restrict__ deep)
{
    __shared__ int32_t cnt[kMaxLevels];
    for (int k = threadIdx.x; k < kMaxLevels; k += BT) cnt[k] = 0;
    __syncthreads();
    const int64_t i = (int64_t)blockIdx.x * BT + threadIdx.x;
    if (i < n_int) {
        int d = 0;
        int32_t u = (int32_t)i;
        for (;;) { // at most kMaxLevels steps
            if (is_root[u]) break;
            const int32_t p = parent[u];
            if (p < 0) {
                d = -1;
                break;
            }
            if (++d >= kMaxLevels) {
                atomicOr(deep, 1);
                d = -1;
                break;
            }
            u = p;
        }
        depth[i] = d;
        if (d >= 0) atomicAdd(&cnt[d], 1);
    }
    __syncthreads();
    for (int k = threadIdx.x; k < kMaxLevels; k += BT)
        if (cnt[k] > 0) atomicAdd(&hist[k], cnt[k]);
}

// node ids grouped by depth: level d occupies order[off[d], off[d] + hist[d]); each block
// reserves its range per depth with one atomic on cursor[d] (order within a level is free)
__global__ __launch_bounds__(BT) void k_depth_bucket(const int32_t* __restrict__ depth, int64_t n_int,
                                                     const int32_t* __restrict__ off, int32_t* __restrict__ cursor,
                                                     int32_t* __restrict__ order)
{
    __shared__ int32_t cnt[kMaxLevels];
    __shared__ int32_t base[kMaxLevels];
    for (int k = threadIdx.x; k < kMaxLevels; k += BT) cnt[k] = 0;
    __syncthreads();
    const int64_t i = (int64_t)blockIdx.x * BT + threadIdx.x;
    const int d = (i < n_int) ? depth[i] : -1;
    int r = 0;
    if (d >= 0) r = atomicAdd(&cnt[d], 1);
    __syncthreads();
    for (int k = threadIdx.x; k < kMaxLevels; k += BT)
        if (cnt[k] > 0) base[k] = off[k] + atomicAdd(&cursor[k], cnt[k]);
    __syncthreads();
    if (d >= 0) order[base[d] + r] = (int32_t)i;
}

__global__ __launch_bounds__(BT) void k_merge_level(const int32_t* __restrict__ nodes, int32_t cnt,
                                                    const int32_t* __restrict__ left,
                                                    const int32_t* __restrict__ right,
                                                    const int32_t* __restrict__ first,
                                                    const int32_t* __restrict__ last, int32_t fp64_min,
                                                    double* rec)
{
    const int i = blockIdx.x * BT + threadIdx.x;
    if (i >= cnt) return;
    const int32_t p = nodes[i];
    const double* a = rec + (int64_t)left[p] * kRecWords;
    const double* b = rec + (int64_t)right[p] * kRecWords;
    if (last[p] - first[p] + 1 >= fp64_min) merge2<double>(a, b, rec + (int64_t)p * kRecWords);
    else merge2<float>(a, b, rec + (int64_t)p * kRecWords);
}

// ---- moments of an SAH tree ----------------------------------------------------------------------
// The same merges, a workgroup per mid segment (a subtree of at most kSahMid triangles over
// neighbouring positions, its nodes' ids in [lo, hi - 2]), then one workgroup for the nodes above
// them: threads climb from the leaves (the subtrees' roots) and the second child to arrive at a node
// merges it.  Arrivals and records stay within a workgroup, so block-scope fences order them: two
// launches where the levels took one each and a host round trip for their sizes.  Bound: the 768
// bytes of records a merge reads and writes (101,568 triangles: 0.12 + 0.04 ms; 22 launches and the
// wait before 0.25 ms; 256 threads a workgroup instead of 512: 0.17 ms for the first).
constexpr int kMergeThreads = 512;
__global__ __launch_bounds__(kMergeThreads) void k_merge_mid(
    const int32_t* __restrict__ seg, const int32_t* __restrict__ left, const int32_t* __restrict__ right,
    const int32_t* __restrict__ parent, const int32_t* __restrict__ first, const int32_t* __restrict__ last, int64_t n,
    int32_t fp64_min, double* rec, int32_t* __restrict__ seg_root, int32_t* __restrict__ visits)
{
    __shared__ int32_t cnt[kSahMid];
    const int32_t lo = seg[4 * (int64_t)blockIdx.x], hi = seg[4 * (int64_t)blockIdx.x + 1];
    for (int k = threadIdx.x; k < hi - lo; k += kMergeThreads) cnt[k] = 0;
    if (threadIdx.x == 0) { // the nodes above the subtrees are the splits between them
        if (lo > 0) visits[lo - 1] = 0;
        visits[hi - 1] = 0;
    }
    __syncthreads();
    for (int32_t j = lo + (int32_t)threadIdx.x; j < hi; j += kMergeThreads) {
        int32_t u = (int32_t)(n - 1) + j;
        for (;;) {
            const int32_t p = parent[u];
            if (p < lo || p > hi - 2) { // the subtree's root
                seg_root[blockIdx.x] = u;
                break;
            }
            __threadfence_block();
            if (atomicAdd(&cnt[p - lo], 1) == 0) break; // the sibling's thread finishes this node
            __threadfence_block();
            const double* a = rec + (int64_t)left[p] * kRecWords;
            const double* b = rec + (int64_t)right[p] * kRecWords;
            if (last[p] - first[p] + 1 >= fp64_min) merge2<double>(a, b, rec + (int64_t)p * kRecWords);
            else merge2<float>(a, b, rec + (int64_t)p * kRecWords);
            u = p;
        }
    }
}

constexpr int kTopThreads = 1024;
__global__ __launch_bounds__(kTopThreads) void k_merge_top(const int32_t* __restrict__ seg_root, int64_t n_seg,
                                                           const int32_t* __restrict__ left,
                                                           const int32_t* __restrict__ right,
                                                           const int32_t* __restrict__ parent,
                                                           const int32_t* __restrict__ first,
                                                           const int32_t* __restrict__ last, int32_t fp64_min,
                                                           double* rec, int32_t* visits)
{
    for (int64_t k = threadIdx.x; k < n_seg; k += kTopThreads) {
        int32_t u = seg_root[k];
        for (;;) {
            const int32_t p = parent[u];
            if (p < 0) break;
            __threadfence_block();
            if (atomicAdd(&visits[p], 1) == 0) break;
            __threadfence_block();
            const double* a = rec + (int64_t)left[p] * kRecWords;
            const double* b = rec + (int64_t)right[p] * kRecWords;
            if (last[p] - first[p] + 1 >= fp64_min) merge2<double>(a, b, rec + (int64_t)p * kRecWords);
            else merge2<float>(a, b, rec + (int64_t)p * kRecWords);
            u = p;
        }
    }
}

// ---- collapse into wide nodes -----------------------------------------------------------------
__device__ __forceinline__ int32_t node_count(int32_t u, int64_t n, const int32_t* first, const int32_t* last)
{
    return (u >= n - 1) ? 1 : last[u] - first[u] + 1;
}

struct BinTree {
    const int32_t *left, *right, *first, *last;
    int64_t n;
};

// the slots of binary node b's wide node: binary nodes sl[], their triangle counts sc[]; returns how many
__device__ __forceinline__ int wide_slots(int32_t b, const BinTree& t, int leaf_max, int width, int rounds,
                                          int32_t (&sl)[kWidth], int32_t (&sc)[kWidth])
{
    const int32_t *left = t.left, *right = t.right, *first = t.first, *last = t.last;
    const int64_t n = t.n;
    int ns;
    if (b >= n - 1 || node_count(b, n, first, last) <= leaf_max) {
        sl[0] = b;
        sc[0] = node_count(b, n, first, last);
        ns = 1;
    } else {
        sl[0] = left[b];
        sl[1] = right[b];
        sc[0] = node_count(sl[0], n, first, last);
        sc[1] = node_count(sl[1], n, first, last);
        ns = 2;
        // rounds > 0: take whole binary levels (every non-leaf slot opened, rounds - 1 times)
        for (int r = 1; r < rounds; ++r) {
            int32_t nl[kWidth], nc[kWidth];
            int nn = 0;
            for (int s = 0; s < ns; ++s) {
                int32_t u = sl[s];
                if (u < n - 1 && sc[s] > leaf_max) {
                    nl[nn] = left[u];
                    nc[nn] = node_count(nl[nn], n, first, last);
                    ++nn;
                    nl[nn] = right[u];
                    nc[nn] = node_count(nl[nn], n, first, last);
                    ++nn;
                } else {
                    nl[nn] = u;
                    nc[nn] = sc[s];
                    ++nn;
                }
            }
            for (int s = 0; s < nn; ++s) {
                sl[s] = nl[s];
                sc[s] = nc[s];
            }
            ns = nn;
        }
        // rounds == 0: repeatedly open the largest non-leaf slot until the node has width slots
        while (rounds == 0 && ns < width) {
            int best = -1, bc = leaf_max;
            for (int s = 0; s < ns; ++s)
                if (sc[s] > bc) {
                    bc = sc[s];
                    best = s;
                }
            if (best < 0) break;
            int32_t u = sl[best];
            for (int s = ns; s > best + 1; --s) {
                sl[s] = sl[s - 1];
                sc[s] = sc[s - 1];
            }
            sl[best] = left[u];
            sl[best + 1] = right[u];
            sc[best] = node_count(sl[best], n, first, last);
            sc[best + 1] = node_count(sl[best + 1], n, first, last);
            ++ns;
        }
    }
    return ns;
}

// Wide nodes are numbered level by level, each level in slot order.  The level in work is a list of
// binary nodes; its state (nodes, number of the first one, levels done, list array) stays on the
// device, one entry per level, so that the host enqueues as many levels as it expects and reads the
// state once.  k_collapse_top takes the levels of up to 1,024 nodes in one workgroup; a larger level
// takes two launches: slots and block sums of new nodes, then the numbers of the children (every
// block adds up the sums of the blocks before it).
struct LevelState {
    int32_t cnt, base, depth, cur;
};
struct Wide {
    int32_t *slot_bin, *child; // width entries per wide node
    int32_t* ns;
    int32_t* lvl[2];
};

// exclusive scan over a workgroup of T threads (T / 64 waves); total of all
template <int T>
__device__ __forceinline__ int block_scan(int v, int32_t* part, int& total)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int x = v;
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 63) part[w] = x;
    __syncthreads();
    int before = 0;
    total = 0;
    for (int k = 0; k < T / 64; ++k) {
        if (k < w) before += part[k];
        total += part[k];
    }
    __syncthreads();
    return before + x - v;
}

// writes wide node g's children numbers (from `next` on) and the next level's list
__device__ __forceinline__ void link_children(const Wide& w, int64_t g, int width, int leaf_max, const BinTree& t,
                                              int32_t next_base, int k, int32_t* __restrict__ level_next)
{
    for (int s = 0; s < width; ++s) {
        const int32_t u = w.slot_bin[g * width + s];
        int32_t cw = -1;
        if (u >= 0 && node_count(u, t.n, t.first, t.last) > leaf_max) {
            cw = next_base + k;
            level_next[k] = u;
            ++k;
        }
        w.child[g * width + s] = cw;
    }
}

// writes wide node g's slots; returns its number of children
__device__ __forceinline__ int put_slots(const Wide& w, int64_t g, int32_t b, const BinTree& t, int leaf_max, int width,
                                         int rounds)
{
    int32_t sl[kWidth], sc[kWidth];
    const int ns = b < 0 ? 0 : wide_slots(b, t, leaf_max, width, rounds, sl, sc); // b < 0: no root was found
    int nc = 0;
    for (int s = 0; s < width; ++s) {
        w.slot_bin[g * width + s] = (s < ns) ? sl[s] : -1;
        if (s < ns && sc[s] > leaf_max) ++nc;
    }
    w.ns[g] = ns;
    return nc;
}

constexpr int kTopNodes = 1024;
__global__ __launch_bounds__(kTopNodes) void k_collapse_top(Wide w, BinTree t, int32_t cnt, int leaf_max, int width,
                                                            int rounds, LevelState* __restrict__ state)
{
    __shared__ int32_t part[kTopNodes / 64];
    LevelState st{cnt, 0, 0, 0};
    while (st.cnt > 0 && st.cnt <= kTopNodes) { // uniform
        const int i = threadIdx.x;
        const bool live = i < st.cnt;
        const int nc = live ? put_slots(w, st.base + i, w.lvl[st.cur][i], t, leaf_max, width, rounds) : 0;
        int total;
        const int k = block_scan<kTopNodes>(nc, part, total);
        if (live) link_children(w, st.base + i, width, leaf_max, t, st.base + st.cnt, k, w.lvl[st.cur ^ 1]);
        __syncthreads(); // the next level's list
        st = LevelState{total, st.base + st.cnt, st.depth + 1, st.cur ^ 1};
    }
    if (threadIdx.x == 0) state[0] = st;
}

__global__ __launch_bounds__(BT) void k_collapse_slots(Wide w, BinTree t, int leaf_max, int width, int rounds,
                                                       const LevelState* __restrict__ state,
                                                       int32_t* __restrict__ newcount, int32_t* __restrict__ sums)
{
    __shared__ int32_t part[BT / 64];
    const LevelState st = *state;
    if ((int64_t)blockIdx.x * BT >= st.cnt) return;
    const int i = blockIdx.x * BT + threadIdx.x;
    const int nc = i < st.cnt ? put_slots(w, st.base + i, w.lvl[st.cur][i], t, leaf_max, width, rounds) : 0;
    if (i < st.cnt) newcount[i] = nc;
    int total;
    block_scan<BT>(nc, part, total);
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

__global__ __launch_bounds__(BT) void k_collapse_link(Wide w, BinTree t, int leaf_max, int width,
                                                      LevelState* __restrict__ state,
                                                      const int32_t* __restrict__ newcount,
                                                      const int32_t* __restrict__ sums)
{
    __shared__ int32_t part[BT / 64];
    const LevelState st = state[0];
    if ((int64_t)blockIdx.x * BT >= st.cnt) {
        if (blockIdx.x == 0 && threadIdx.x == 0) state[1] = st; // no level left
        return;
    }
    int before = 0, own;
    for (int k = threadIdx.x; k < blockIdx.x; k += BT) before += sums[k];
    (void)block_scan<BT>(before, part, before);
    const int i = blockIdx.x * BT + threadIdx.x;
    const int k = before + block_scan<BT>(i < st.cnt ? newcount[i] : 0, part, own);
    if (i < st.cnt) link_children(w, st.base + i, width, leaf_max, t, st.base + st.cnt, k, w.lvl[st.cur ^ 1]);
    if ((int64_t)(blockIdx.x + 1) * BT >= st.cnt && threadIdx.x == 0)
        state[1] = LevelState{before + own, st.base + st.cnt, st.depth + 1, st.cur ^ 1};
}

// one slot: its words into w, its box and link into bx, a leaf's near-field rule into its first triangle
__device__ __forceinline__ void write_slot(int64_t idx, int width, const int32_t* __restrict__ wide_slot_bin,
                                           const int32_t* __restrict__ wide_ns, const int32_t* __restrict__ child_wide,
                                           const double* __restrict__ rec, const int32_t* __restrict__ first,
                                           const int32_t* __restrict__ last, int64_t n, float beta2,
                                           const int64_t* __restrict__ f_off, int M, const float* __restrict__ minfo,
                                           uint32_t* w, float* __restrict__ bx, uint32_t* __restrict__ tris)
{
    const int64_t src = idx; // the collapse's tables have width entries per node
    int32_t u = wide_slot_bin[src];
    if ((int)(idx % width) >= wide_ns[idx / width] || u < 0) {
        for (int k = 0; k < FWN_W_LINK; ++k) w[k] = 0u;
        w[FWN_W_LINK] = FWN_LINK_EMPTY;
        for (int k = 0; k < kBoxWords; ++k) bx[k] = 0.0f;
        bx[6] = __uint_as_float(FWN_LINK_EMPTY);
        return;
    }
    const double* r = rec + (int64_t)u * kRecWords;
    // the slot's box for distance queries, rounded outward so it still contains the triangles
    float box[8];
    for (int d = 0; d < 3; ++d) {
        box[d] = __double2float_rd(r[R_LO + d]);
        box[3 + d] = __double2float_ru(r[R_HI + d]);
    }
    float4* b4 = reinterpret_cast<float4*>(bx); // the link here, the disk by k_slot_disks
    b4[0] = make_float4(box[0], box[1], box[2], box[3]);
    double r2 = 0.0;
    for (int d = 0; d < 3; ++d) {
        double a = fabs(r[R_P + d] - r[R_LO + d]), b = fabs(r[R_HI + d] - r[R_P + d]);
        double e = a > b ? a : b;
        r2 += e * e;
    }
    const float r2f = nextafterf((float)r2, INFINITY); // rounded up: still a bound
    float f[FWN_W_LINK];
    f[FWN_W_PX] = (float)r[R_P];
    f[FWN_W_PY] = (float)r[R_P + 1];
    f[FWN_W_PZ] = (float)r[R_P + 2];
    f[FWN_W_THR] = beta2 * r2f; // the query's far-field threshold
    f[FWN_W_NX] = (float)r[R_N];
    f[FWN_W_NY] = (float)r[R_N + 1];
    f[FWN_W_NZ] = (float)r[R_N + 2];
    // tr and C are folded into the homogeneous quadratic and cubic: tr = tr |d|^2 / |d|^2 adds
    // tr to the diagonal of A, (C.d) = (C.d) |d|^2 / |d|^2 adds C_i to the cubic monomials
    // d_i d_j d_j; the far field then needs no constant terms
    const double* M1 = r + R_M1;
    const double tr = M1[0] + M1[4] + M1[8];
    float* A = f + FWN_W_A;
    A[0] = (float)(-3.0 * M1[0] + tr);
    A[1] = (float)(-3.0 * M1[4] + tr);
    A[2] = (float)(-3.0 * M1[8] + tr);
    A[3] = (float)(-3.0 * (M1[1] + M1[3]));
    A[4] = (float)(-3.0 * (M1[5] + M1[7]));
    A[5] = (float)(-3.0 * (M1[6] + M1[2]));
    const double* S = r + R_S;
    const double sc[10] = {7.5, 7.5, 7.5, 22.5, 22.5, 22.5, 22.5, 22.5, 22.5, 45.0};
    const double cx = -4.5 * (S[0] + S[5] + S[7]);
    const double cy = -4.5 * (S[3] + S[1] + S[8]);
    const double cz = -4.5 * (S[4] + S[6] + S[2]);
    // monomials: xxx yyy zzz xxy xxz yyx yyz zzx zzy xyz
    const double fold[10] = {cx, cy, cz, cy, cz, cx, cz, cx, cy, 0.0};
    for (int k = 0; k < 10; ++k) f[FWN_W_B + k] = (float)(sc[k] * S[k] + fold[k]);
    for (int k = 0; k < FWN_W_LINK; ++k) w[k] = __float_as_uint(f[k]);
    // a leaf slot is any slot without a wide child: a single triangle or a bucket of at most
    // leaf_max triangles (an internal binary node); both cover a contiguous sorted range
    const int32_t cw = child_wide[src];
    if (cw >= 0) {
        w[FWN_W_LINK] = ((uint32_t)cw << 4) | (uint32_t)wide_ns[cw];
        b4[1] = make_float4(box[4], box[5], __uint_as_float(w[FWN_W_LINK]), 0.0f);
        return;
    }
    const bool bin_leaf = u >= n - 1;
    const int64_t tf = bin_leaf ? (u - (n - 1)) : first[u];
    const int32_t tc = bin_leaf ? 1 : last[u] - first[u] + 1;
    w[FWN_W_LINK] = FWN_LINK_LEAF | ((uint32_t)tf << 3) | (uint32_t)(tc - 1);
    b4[1] = make_float4(box[4], box[5], __uint_as_float(w[FWN_W_LINK]), 0.0f);
    // the leaf's FP64 near-field rule, in its first triangle: q is within tau of the leaf's
    // bounding sphere when |d|^2 < (sqrt(r2) + tau)^2 and, for a single triangle, within tau of
    // its plane when (d.N)^2 < tau^2 |N|^2
    const float tau = minfo[8 * mesh_of(f_off, M, tf) + 6];
    const float rr = sqrtf(r2f) + tau;
    const float nn = fmaf(f[FWN_W_NX], f[FWN_W_NX], fmaf(f[FWN_W_NY], f[FWN_W_NY], f[FWN_W_NZ] * f[FWN_W_NZ]));
    uint32_t* tw = tris + tf * kTriWords;
    tw[FWN_T_NEAR2] = __float_as_uint(rr * rr);
    tw[FWN_T_PLANE] = __float_as_uint((tau * tau) * nn);
}

__global__ __launch_bounds__(RT) void k_write_slots(int64_t W, int width, const int32_t* __restrict__ wide_slot_bin,
                                                    const int32_t* __restrict__ wide_ns,
                                                    const int32_t* __restrict__ child_wide,
                                                    const double* __restrict__ rec,
                                                    const int32_t* __restrict__ first,
                                                    const int32_t* __restrict__ last, int64_t n, float beta2,
                                                    const int64_t* __restrict__ f_off, int M,
                                                    const float* __restrict__ minfo, uint32_t* __restrict__ slots,
                                                    float* __restrict__ boxes, uint32_t* __restrict__ tris)
{
    // the block's slots, written together below
    __shared__ uint32_t lds[RT * (kSlotWords + 1)];
    const int64_t idx0 = (int64_t)blockIdx.x * RT, idx = idx0 + threadIdx.x;
    if (idx < W * width)
        write_slot(idx, width, wide_slot_bin, wide_ns, child_wide, rec, first, last, n, beta2, f_off, M, minfo,
                   lds + threadIdx.x * (kSlotWords + 1), boxes + idx * kBoxWords, tris);
    __syncthreads();
    const int words = (int)min((int64_t)RT, W * width - idx0) * kSlotWords;
    for (int k = threadIdx.x; k < words; k += RT) slots[idx0 * kSlotWords + k] = lds[k + k / kSlotWords];
}

// Each slot's disk, from its triangles' vertices in double.  A thread takes a slot of one triangle by
// itself (three in four); the block's other slots are listed and taken by rows of 16 lanes, those above
// kDiskRow triangles by waves.  A block's slots are spread over the array, as the large ones come first.
// Bound: the chain of loads of a slot's triangles; 101,568 and 940,800 triangles 48 and 395 us with a row
// for every slot, 41 and 182 so.  A slot of more than kDiskTris triangles (nearly always entered, and a
// serial loop here) or with a sliver (sine below 1e-4: its evaluated distance may be off by more than
// the bound allows for) gets no bound (400k closest points, F = 199,692: limit 128 4.33 ms, 512 4.07,
// 1,024 3.98).
constexpr int64_t kDiskTris = 1024, kDiskRow = 64;

struct DiskSpan { // of a slot's triangles about a point and a normal; rounded outward
    float lo = INFINITY, hi = -INFINITY, rr = 0.0f;
    bool none = false;
};

__device__ __forceinline__ void disk_triangle(const float* __restrict__ tw, const double (&c0)[3],
                                              const double (&nn)[3], DiskSpan& S)
{
    double w[3][3];
    for (int k = 0; k < 3; ++k)
        for (int d = 0; d < 3; ++d) w[k][d] = (double)tw[3 * k + d] - c0[d];
    double e1[3], e2[3];
    for (int d = 0; d < 3; ++d) {
        e1[d] = w[1][d] - w[0][d];
        e2[d] = w[2][d] - w[0][d];
    }
    const double N[3] = {e1[1] * e2[2] - e1[2] * e2[1], e1[2] * e2[0] - e1[0] * e2[2],
                         e1[0] * e2[1] - e1[1] * e2[0]};
    S.none |= !(N[0] * N[0] + N[1] * N[1] + N[2] * N[2] >
                1e-8 * (e1[0] * e1[0] + e1[1] * e1[1] + e1[2] * e1[2]) *
                    (e2[0] * e2[0] + e2[1] * e2[1] + e2[2] * e2[2]));
    for (int k = 0; k < 3; ++k) {
        const double h = w[k][0] * nn[0] + w[k][1] * nn[1] + w[k][2] * nn[2];
        double q = 0.0;
        for (int d = 0; d < 3; ++d) q += (w[k][d] - h * nn[d]) * (w[k][d] - h * nn[d]);
        S.lo = fminf(S.lo, __double2float_rd(h));
        S.hi = fmaxf(S.hi, __double2float_ru(h));
        S.rr = fmaxf(S.rr, __double2float_ru(q));
    }
}

__device__ __forceinline__ void write_disk(float* __restrict__ o, const double (&c0)[3], const double (&nn)[3],
                                           const DiskSpan& S)
{
    float c[3];
    double margin = 0.0; // the rounding of c and n
    for (int d = 0; d < 3; ++d) {
        c[d] = (float)(c0[d] + nn[d] * 0.5 * ((double)S.lo + (double)S.hi));
        margin += 1e-7 * fabs((double)c[d]);
    }
    const double t = 0.5 * ((double)S.hi - (double)S.lo), R = sqrt((double)S.rr);
    margin += 3e-7 * (t + R);
    o[7] = S.none ? INFINITY : __double2float_ru(t + margin);
    o[11] = S.none ? INFINITY : __double2float_ru(R + margin);
    for (int d = 0; d < 3; ++d) {
        o[8 + d] = S.none ? 0.0f : c[d];
        o[12 + d] = S.none ? 0.0f : (float)nn[d];
    }
    o[15] = 0.0f;
}

// the point and unit normal that a slot's disk is about; false: no normal
__device__ __forceinline__ bool disk_frame(const double* __restrict__ r, double (&c0)[3], double (&nn)[3])
{
    for (int d = 0; d < 3; ++d) {
        c0[d] = r[R_P + d];
        nn[d] = r[R_N + d];
    }
    const double A = sqrt(nn[0] * nn[0] + nn[1] * nn[1] + nn[2] * nn[2]);
    for (int d = 0; d < 3; ++d) nn[d] /= A;
    return A > 0.0;
}

__global__ __launch_bounds__(BT) void k_slot_disks(int64_t nslots, const int32_t* __restrict__ slot_bin,
                                                   const double* __restrict__ rec, const int32_t* __restrict__ first,
                                                   const int32_t* __restrict__ last, int64_t n,
                                                   const uint32_t* __restrict__ tris, float* __restrict__ boxes)
{
    __shared__ int32_t list[BT], large[BT];
    __shared__ int32_t count[2];
    if (threadIdx.x < 2) count[threadIdx.x] = 0;
    __syncthreads();
    // slot of the block's thread t: runs of 16
    auto slot_of = [&](int t) { return ((int64_t)(t >> 4) * gridDim.x + blockIdx.x) * 16 + (t & 15); };
    const int64_t idx = slot_of(threadIdx.x);
    if (idx < nslots && __float_as_uint(boxes[idx * kBoxWords + 6]) != FWN_LINK_EMPTY) {
        const int64_t u = slot_bin[idx];
        if (u >= n - 1) {
            double c0[3], nn[3];
            DiskSpan S;
            S.none = !disk_frame(rec + u * kRecWords, c0, nn);
            disk_triangle(reinterpret_cast<const float*>(tris + (u - (n - 1)) * kTriWords), c0, nn, S);
            write_disk(boxes + idx * kBoxWords, c0, nn, S);
        } else if (last[u] - first[u] < kDiskRow) {
            list[atomicAdd(&count[0], 1)] = threadIdx.x;
        } else {
            large[atomicAdd(&count[1], 1)] = threadIdx.x;
        }
    }
    __syncthreads();
    // a group of g lanes takes a slot
    auto take = [&](int t, int g) {
        const int64_t at = slot_of(t);
        const int64_t u = slot_bin[at], t0 = first[u], t1 = last[u];
        double c0[3], nn[3];
        DiskSpan S;
        S.none = !disk_frame(rec + u * kRecWords, c0, nn) || t1 - t0 >= kDiskTris;
        if (!S.none)
            for (int64_t k = t0 + (threadIdx.x & (g - 1)); k <= t1; k += g)
                disk_triangle(reinterpret_cast<const float*>(tris + k * kTriWords), c0, nn, S);
        for (int m = g / 2; m > 0; m >>= 1) {
            S.lo = fminf(S.lo, __shfl_xor(S.lo, m));
            S.hi = fmaxf(S.hi, __shfl_xor(S.hi, m));
            S.rr = fmaxf(S.rr, __shfl_xor(S.rr, m));
            S.none |= __shfl_xor((int)S.none, m) != 0;
        }
        if ((threadIdx.x & (g - 1)) == 0) write_disk(boxes + at * kBoxWords, c0, nn, S);
    };
    for (int k = threadIdx.x >> 6; k < count[1]; k += BT / 64) take(large[k], 64);
    for (int k = threadIdx.x >> 4; k < count[0]; k += BT / 16) take(list[k], 16);
}

} // namespace

int grid_blocks(int64_t n, int threads)
{
    int64_t b = (n + threads - 1) / threads;
    if (b < 1) b = 1;
    if (b > INT32_MAX) fail(FWN_LIMIT_EXCEEDED, "grid too large");
    return (int)b;
}

void build_engine(Engine& e, int32_t M, const float* V_host, const int64_t* v_off, const int32_t* F_host,
                  const int64_t* f_off)
{
    hipStream_t s = e.stream;
    const int64_t nV = v_off[M];
    const int64_t nF = f_off[M];
    // a leaf slot's link holds its first triangle in 28 bits
    if (nF >= ((int64_t)1 << 28) - 1) fail(FWN_LIMIT_EXCEEDED, "2^28 - 1 or more triangles");
    e.n_meshes = M;
    e.n_tris = nF;
    e.h_f_off.assign(f_off, f_off + M + 1);
    int64_t largest = 0;
    for (int m = 0; m < M; ++m) largest = std::max(largest, f_off[m + 1] - f_off[m]);
    e.uneven = M > 1 && 2 * largest * M >= 3 * nF;
    const int leaf_max = e.opt.leaf_max;
    const int width = e.opt.tree_width;
    e.width = width;

    hipEvent_t b0, b1;
    FWN_HIP(hipEventCreate(&b0));
    FWN_HIP(hipEventCreate(&b1));
    struct Events {
        hipEvent_t a, b;
        ~Events()
        {
            (void)hipEventDestroy(a);
            (void)hipEventDestroy(b);
        }
    } events{b0, b1};
    FWN_HIP(hipEventRecord(b0, s));

    const bool sah = e.opt.tree_builder == FWN_TREE_SAH;
    const int64_t n = nF;
    // scratch bytes per triangle: mesh 24, centroid and box 36, orders 8, binary tree 32, the SAH lists
    // 24, moment records 512, collapse 8 width + 16
    Arena ar((size_t)(12 * nV + (660 + 8 * width) * nF + 256 * (int64_t)M + (1 << 16)));
    float* dV = ar.take<float>(3 * nV);
    int32_t* dF = ar.take<int32_t>(3 * nF);
    int64_t* dvo = ar.take<int64_t>(M + 1);
    int64_t* dfo = ar.take<int64_t>(M + 1);
    if (nV) FWN_HIP(hipMemcpyAsync(dV, V_host, sizeof(float) * 3 * nV, hipMemcpyHostToDevice, s));
    if (nF) FWN_HIP(hipMemcpyAsync(dF, F_host, sizeof(int32_t) * 3 * nF, hipMemcpyHostToDevice, s));
    FWN_HIP(hipMemcpyAsync(dvo, v_off, sizeof(int64_t) * (M + 1), hipMemcpyHostToDevice, s));
    FWN_HIP(hipMemcpyAsync(dfo, f_off, sizeof(int64_t) * (M + 1), hipMemcpyHostToDevice, s));

    int32_t* boxes = ar.take<int32_t>(12 * (int64_t)M);
    int32_t* err = ar.take<int32_t>(1);
    float* cinfo = ar.take<float>(6 * (int64_t)M);
    e.mesh_info.alloc(sizeof(float) * 8 * M);
    hipLaunchKernelGGL(k_init, dim3(grid_blocks(12 * M, 256)), dim3(256), 0, s, boxes, M, err);
    FWN_LAUNCH_CHECK("k_init");
    float* cen = ar.take<float>(3 * nF);
    float* tbox = sah ? ar.take<float>(6 * nF) : nullptr;
    if (nF) {
        hipLaunchKernelGGL(k_tri_setup, dim3(grid_blocks(nF, TS)), dim3(TS), 0, s, dV, dF, nF, dfo, dvo, M, cen, boxes,
                           tbox, err);
        FWN_LAUNCH_CHECK("k_tri_setup");
    }
    hipLaunchKernelGGL(k_box_final, dim3(grid_blocks(M, 64)), dim3(64), 0, s, boxes, M, e.opt.near_fp64_rel, cinfo,
                       e.mesh_info.as<float>());
    FWN_LAUNCH_CHECK("k_box_final");

    e.tris.alloc(sizeof(uint32_t) * kTriWords * (size_t)std::max<int64_t>(nF, 1));
    e.roots.alloc(sizeof(int32_t) * 2 * M);
    e.h_roots.assign(2 * (size_t)M, -1);
    for (int m = 0; m < M; ++m) e.h_roots[2 * m + 1] = 0;
    e.h_tau.assign(M, 0.0f);
    // what the host reads at the end: input errors and each mesh's tau (the tree of a mesh with
    // input errors is built from clamped indices and thrown away)
    auto read_setup = [&](char* to) {
        FWN_HIP(hipMemcpyAsync(to, err, sizeof(int32_t), hipMemcpyDeviceToHost, s));
        FWN_HIP(hipMemcpyAsync(to + 16, e.mesh_info.p, sizeof(float) * 8 * M, hipMemcpyDeviceToHost, s));
    };
    auto check_setup = [&](const char* from) {
        const int32_t h_err = *reinterpret_cast<const int32_t*>(from);
        if (h_err & 1) fail(FWN_INVALID_ARGUMENT, "facet index out of range of its mesh's vertices");
        if (h_err & 2) fail(FWN_INVALID_ARGUMENT, "non-finite vertex position");
        const float* mi = reinterpret_cast<const float*>(from + 16);
        for (int m = 0; m < M; ++m) e.h_tau[m] = mi[8 * m + 6];
        e.h_info.assign(mi, mi + 8 * (size_t)M);
    };
    const size_t setup_b = 16 + sizeof(float) * 8 * (size_t)M;

    if (nF == 0) {
        char* hs = host_stage(e, setup_b);
        read_setup(hs);
        e.slots.alloc(sizeof(uint32_t) * width * kSlotWords);
        e.boxes.alloc(sizeof(float) * width * kBoxWords);
        e.n_nodes = 0;
        e.max_depth = 0;
        FWN_HIP(hipMemcpyAsync(e.roots.p, e.h_roots.data(), sizeof(int32_t) * 2 * M, hipMemcpyHostToDevice, s));
        FWN_HIP(hipStreamSynchronize(s));
        check_setup(hs);
        return;
    }

    // ---- binary tree topology: Morton-order radix tree, or top-down SAH splits ----
    const int64_t nnodes = 2 * n - 1;
    int32_t* left = ar.take<int32_t>(n - 1);
    int32_t* right = ar.take<int32_t>(n - 1);
    int32_t* first = ar.take<int32_t>(n - 1);
    int32_t* last = ar.take<int32_t>(n - 1);
    int32_t* parent = ar.take<int32_t>(nnodes);
    uint8_t* isroot = ar.take<uint8_t>((nnodes + 3) & ~(int64_t)3);
    int32_t* rootbin = ar.take<int32_t>(M);
    hipLaunchKernelGGL(k_fill_i32, dim3(grid_blocks((nnodes + 3) / 4, 256)), dim3(256), 0, s,
                       reinterpret_cast<int32_t*>(isroot), (nnodes + 3) / 4, 0);
    hipLaunchKernelGGL(k_fill_i32, dim3(grid_blocks(M, 256)), dim3(256), 0, s, rootbin, (int64_t)M, -1);
    FWN_LAUNCH_CHECK("k_fill_i32");
    uint32_t* vp = ar.take<uint32_t>(nF);
    SahMids mids{nullptr, 0};
    if (sah) {
        mids = build_topology_sah(e, ar, cen, tbox, boxes, nF, f_off, M, reinterpret_cast<int32_t*>(vp), left, right,
                                  parent, first, last, isroot, rootbin);
    } else {
        hipLaunchKernelGGL(k_fill_i32, dim3(grid_blocks(nnodes, 256)), dim3(256), 0, s, parent, nnodes, -1);
        FWN_LAUNCH_CHECK("k_fill_i32");
        DBuf hist, rowsum;
        uint64_t* kp = ar.take<uint64_t>(nF);
        uint64_t* kp2 = ar.take<uint64_t>(nF);
        uint32_t* vp2 = ar.take<uint32_t>(nF);
        hipLaunchKernelGGL(k_tri_keys, dim3(grid_blocks(nF, BT)), dim3(BT), 0, s, cen, nF, dfo, M, cinfo, kp, vp);
        FWN_LAUNCH_CHECK("k_tri_keys");
        int mesh_bits = 0;
        while ((1 << mesh_bits) < M) ++mesh_bits;
        int nbits = (M > 1) ? 32 + mesh_bits : 30;
        radix_sort_pairs(kp, vp, kp2, vp2, nF, nbits, hist, rowsum, s);
        if (n > 1) {
            hipLaunchKernelGGL(k_karras, dim3(grid_blocks(n - 1, BT)), dim3(BT), 0, s, kp, n, left, right, parent,
                               first, last);
            FWN_LAUNCH_CHECK("k_karras");
        }
        hipLaunchKernelGGL(k_find_roots, dim3(grid_blocks(std::max<int64_t>(n - 1, M), BT)), dim3(BT), 0, s, first,
                           last, n, kp, dfo, M, rootbin, isroot);
        FWN_LAUNCH_CHECK("k_find_roots");
        FWN_HIP(hipStreamSynchronize(s)); // the sort's own scratch is freed here
    }

    // ---- moments ----
    double* rec = ar.take<double>(kRecWords * nnodes);
    hipLaunchKernelGGL(k_leaf_records, dim3(grid_blocks(n, RT)), dim3(RT), 0, s, vp, n, dV, dF, dfo, dvo, M,
                       e.tris.as<uint32_t>(), rec);
    FWN_LAUNCH_CHECK("k_leaf_records");
    if (n > 1 && sah && e.opt.moment_pass == FWN_MOMENTS_LEVELS) {
        int32_t* seg_root = ar.take<int32_t>(mids.count);
        int32_t* visits = ar.take<int32_t>(n);
        hipLaunchKernelGGL(k_merge_mid, dim3((unsigned)mids.count), dim3(kMergeThreads), 0, s, mids.seg, left, right, parent, first,
                           last, n, e.opt.fp64_moment_min, rec, seg_root, visits);
        FWN_LAUNCH_CHECK("k_merge_mid");
        if (mids.count > 1) {
            hipLaunchKernelGGL(k_merge_top, dim3(1), dim3(kTopThreads), 0, s, seg_root, mids.count, left, right, parent,
                               first, last, e.opt.fp64_moment_min, rec, visits);
            FWN_LAUNCH_CHECK("k_merge_top");
        }
    } else if (n > 1) {
        const int64_t n_int = n - 1;
        int32_t* depth = ar.take<int32_t>(n_int);
        int32_t* hist_d = ar.take<int32_t>(2 * kMaxLevels + 1); // hist[kMaxLevels], cursor[kMaxLevels], deep
        int32_t* lvl_off = ar.take<int32_t>(kMaxLevels);
        int32_t* order = ar.take<int32_t>(n_int);
        std::vector<int32_t> hh(kMaxLevels + 1, 0);
        if (e.opt.moment_pass == FWN_MOMENTS_LEVELS) {
            hipLaunchKernelGGL(k_fill_i32, dim3(grid_blocks(2 * kMaxLevels + 1, 256)), dim3(256), 0, s, hist_d,
                               (int64_t)(2 * kMaxLevels + 1), 0);
            hipLaunchKernelGGL(k_node_depth, dim3(grid_blocks(n_int, BT)), dim3(BT), 0, s, parent, isroot, n_int, depth,
                               hist_d, hist_d + 2 * kMaxLevels);
            FWN_LAUNCH_CHECK("k_node_depth");
            FWN_HIP(hipMemcpyAsync(hh.data(), hist_d, sizeof(int32_t) * kMaxLevels, hipMemcpyDeviceToHost, s));
            FWN_HIP(hipMemcpyAsync(&hh[kMaxLevels], hist_d + 2 * kMaxLevels, sizeof(int32_t), hipMemcpyDeviceToHost, s));
            FWN_HIP(hipStreamSynchronize(s));
        }
        if (hh[kMaxLevels] == 0 && e.opt.moment_pass == FWN_MOMENTS_LEVELS) {
            std::vector<int32_t> off(kMaxLevels, 0);
            int levels = 0;
            for (int d = 0, acc = 0; d < kMaxLevels; ++d) {
                off[d] = acc;
                acc += hh[d];
                if (hh[d] > 0) levels = d + 1;
            }
            FWN_HIP(hipMemcpyAsync(lvl_off, off.data(), sizeof(int32_t) * kMaxLevels, hipMemcpyHostToDevice, s));
            hipLaunchKernelGGL(k_depth_bucket, dim3(grid_blocks(n_int, BT)), dim3(BT), 0, s, depth, n_int, lvl_off,
                               hist_d + kMaxLevels, order);
            FWN_LAUNCH_CHECK("k_depth_bucket");
            for (int d = levels - 1; d >= 0; --d) {
                if (hh[d] == 0) continue;
                hipLaunchKernelGGL(k_merge_level, dim3(grid_blocks(hh[d], BT)), dim3(BT), 0, s, order + off[d], hh[d],
                                   left, right, first, last, e.opt.fp64_moment_min, rec);
                FWN_LAUNCH_CHECK("k_merge_level");
            }
            // off is read by the bucket kernel's upload
            FWN_HIP(hipStreamSynchronize(s));
        } else {
            int32_t* visits = ar.take<int32_t>(n_int);
            hipLaunchKernelGGL(k_fill_i32, dim3(grid_blocks(n_int, 256)), dim3(256), 0, s, visits, n_int, 0);
            hipLaunchKernelGGL(k_bottom_up, dim3(grid_blocks(n, BT)), dim3(BT), 0, s, parent, left, right, first, last,
                               isroot, n, e.opt.fp64_moment_min, rec, visits);
            FWN_LAUNCH_CHECK("k_bottom_up");
        }
    }

    // ---- collapse ----
    // the first level: the roots of the meshes that have facets, in mesh order (gathered on the device)
    std::vector<int32_t> mesh_wide(M, -1), level0_mesh;
    for (int m = 0; m < M; ++m)
        if (f_off[m + 1] > f_off[m]) {
            mesh_wide[m] = (int32_t)level0_mesh.size();
            level0_mesh.push_back(m);
        }
    const int32_t cnt0 = (int32_t)level0_mesh.size();
    // every wide node is a distinct binary node with more than leaf_max triangles, or a mesh root
    const int64_t wcap = n + M;
    Wide w;
    w.slot_bin = ar.take<int32_t>(width * wcap);
    w.child = ar.take<int32_t>(width * wcap);
    w.ns = ar.take<int32_t>(wcap);
    w.lvl[0] = ar.take<int32_t>(wcap);
    w.lvl[1] = ar.take<int32_t>(wcap);
    int32_t* newc = ar.take<int32_t>(wcap);
    int32_t* sums = ar.take<int32_t>((wcap + BT - 1) / BT);
    const BinTree bt{left, right, first, last, n};
    int rounds = 0; // binary levels per wide node for the SAH layout: log2(width)
    while ((1 << rounds) < width) ++rounds;
    if (!sah) rounds = 0;
    // levels a balanced tree needs after the first workgroup's, and a few for uneven ones; more are
    // enqueued while there are nodes
    int group = 3;
    for (int64_t c = n / leaf_max / kTopNodes; c > 0; c /= width) ++group;
    LevelState* state = ar.take<LevelState>(group + 1);
    char* hs = host_stage(e, setup_b + sizeof(LevelState) + sizeof(int32_t) * 2 * (size_t)M);
    LevelState* h_state = reinterpret_cast<LevelState*>(hs + setup_b);
    int32_t* h_small = reinterpret_cast<int32_t*>(hs + setup_b + sizeof(LevelState)); // M ints, twice
    if (cnt0 == M) { // the list is the roots array itself
        FWN_HIP(hipMemcpyAsync(w.lvl[0], rootbin, sizeof(int32_t) * M, hipMemcpyDeviceToDevice, s));
    } else {
        std::copy(level0_mesh.begin(), level0_mesh.end(), h_small);
        FWN_HIP(hipMemcpyAsync(w.lvl[1], h_small, sizeof(int32_t) * cnt0, hipMemcpyHostToDevice, s));
        hipLaunchKernelGGL(k_gather_i32, dim3(grid_blocks(cnt0, 256)), dim3(256), 0, s, rootbin, w.lvl[1], cnt0,
                           w.lvl[0]);
        FWN_LAUNCH_CHECK("k_gather_i32");
    }
    hipLaunchKernelGGL(k_collapse_top, dim3(1), dim3(kTopNodes), 0, s, w, bt, cnt0, leaf_max, width, rounds, state);
    FWN_LAUNCH_CHECK("k_collapse_top");
    int64_t bound = std::max<int64_t>((int64_t)kTopNodes * width, cnt0); // nodes of the level in work
    for (;;) {
        for (int k = 0; k < group; ++k) {
            const int blocks = grid_blocks(std::min(bound, wcap), BT);
            hipLaunchKernelGGL(k_collapse_slots, dim3(blocks), dim3(BT), 0, s, w, bt, leaf_max, width, rounds, state + k,
                               newc, sums);
            FWN_LAUNCH_CHECK("k_collapse_slots");
            hipLaunchKernelGGL(k_collapse_link, dim3(blocks), dim3(BT), 0, s, w, bt, leaf_max, width, state + k, newc,
                               sums);
            FWN_LAUNCH_CHECK("k_collapse_link");
            bound = std::min(bound * width, wcap);
        }
        FWN_HIP(hipMemcpyAsync(h_state, state + group, sizeof(LevelState), hipMemcpyDeviceToHost, s));
        read_setup(hs);
        FWN_HIP(hipMemcpyAsync(h_small, rootbin, sizeof(int32_t) * M, hipMemcpyDeviceToHost, s));
        FWN_HIP(hipMemcpyAsync(h_small + M, w.ns, sizeof(int32_t) * cnt0, hipMemcpyDeviceToHost, s));
        FWN_HIP(hipStreamSynchronize(s));
        if (h_state->cnt == 0) break;
        FWN_HIP(hipMemcpyAsync(state, state + group, sizeof(LevelState), hipMemcpyDeviceToDevice, s));
    }
    check_setup(hs);
    for (int m = 0; m < M; ++m)
        if (mesh_wide[m] >= 0 && h_small[m] < 0) fail(FWN_HIP_ERROR, "tree build: mesh root not found");
    const int64_t W = h_state->base;
    if (W < 1 || W > wcap) fail(FWN_HIP_ERROR, "tree build: wide node bound exceeded");
    if (W >= ((int64_t)1 << 27)) fail(FWN_LIMIT_EXCEEDED, "more than 2^27 tree nodes");
    e.n_nodes = W;
    e.max_depth = h_state->depth;
    for (int m = 0; m < M; ++m) {
        if (mesh_wide[m] >= 0) {
            e.h_roots[2 * m] = mesh_wide[m];
            e.h_roots[2 * m + 1] = h_small[M + mesh_wide[m]];
        }
    }
    e.slots.alloc(sizeof(uint32_t) * width * kSlotWords * (size_t)W);
    e.boxes.alloc(sizeof(float) * width * kBoxWords * (size_t)W);
    hipLaunchKernelGGL(k_write_slots, dim3(grid_blocks(W * width, RT)), dim3(RT), 0, s, W, width, w.slot_bin, w.ns,
                       w.child, rec, first, last, n, e.opt.accuracy_scale * e.opt.accuracy_scale, dfo, M,
                       e.mesh_info.as<float>(), e.slots.as<uint32_t>(), e.boxes.as<float>(), e.tris.as<uint32_t>());
    FWN_LAUNCH_CHECK("k_write_slots");
    hipLaunchKernelGGL(k_slot_disks, dim3(grid_blocks(W * width, BT)), dim3(BT), 0, s, W * width, w.slot_bin, rec,
                       first, last, n, e.tris.as<uint32_t>(), e.boxes.as<float>());
    FWN_LAUNCH_CHECK("k_slot_disks");
    std::copy(e.h_roots.begin(), e.h_roots.end(), h_small);
    FWN_HIP(hipMemcpyAsync(e.roots.p, h_small, sizeof(int32_t) * 2 * M, hipMemcpyHostToDevice, s));
    FWN_HIP(hipEventRecord(b1, s));
    FWN_HIP(hipStreamSynchronize(s));
    float ms = 0.0f;
    FWN_HIP(hipEventElapsedTime(&ms, b0, b1));
    e.build_ms = ms;
}

} // namespace fwn
