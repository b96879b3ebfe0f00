// Top-down SAH topology for the tree build (FWN_TREE_SAH).
//
// Every binary split follows one rule, the binned box-area split of the CPU restatement of the
// reference's 4-ary tree build (the tree the reference builds comes from the dependency's
// UT_SolidAngle::init, called at modules/winding/src/FastWindingNumber.cpp:57):
//   * centroid bounds of the segment's triangles; the axis of the longest extent (x before y
//     before z on ties); a segment whose centroids coincide splits at its middle position;
//   * 16 equal bins along that axis (bin = int((c - lo) * (16 / extent)), clamped), each
//     accumulating its triangle count and the union of its triangles' boxes;
//   * a sweep over the 15 bin boundaries minimising area(left) * n_left + area(right) * n_right,
//     with area = dx*dy + dy*dz + dz*dx of float extents, in double (first minimum wins; a
//     segment with no boundary that has triangles on both sides splits at its middle);
//   * a stable partition: triangles of bins <= best first, each side in its previous order.
// Segments are split down to single triangles.  Centroid and box bounds are exact min/max, so
// they do not depend on the order in which threads combine partial results, and the arithmetic
// is the sequential rule's, operation for operation (no contraction into FMAs): the tree equals
// that of a sequential top-down build.
//
// An internal node's id is the position of the last triangle of its left child: every pair of
// neighbouring positions is separated by exactly one split, so the ids are distinct and need no
// counter.  A node learns its id when it is split and then enters itself into its parent.
//
// Three stages, by segment size:
//   * more than kSahMid triangles: level by level over the whole chip, the segments of a level cut into
//     chunks of kChunk triangles (one workgroup each).  Three launches a level: k_sah_bins (bins and
//     per-chunk bin counts), k_sah_next (one workgroup: splits, nodes, the next level's segments and
//     chunks), k_sah_scatter (stable partition between two item arrays, centroid bounds of the
//     children).  The lists stay on the device; the host waits once, after as many levels as a
//     balanced tree needs;
//   * 17 .. kSahMid: k_sah_mid, one workgroup per segment with its centroids, boxes and order in LDS,
//     round by round, a wave per segment;
//   * 2 .. 16: the same workgroup, 16 lanes per segment with the triangles in registers, all
//     sub-segments of a row split in parallel.
// Bound: latency of the split rounds and launches up to some 100k triangles, LDS atomics and scattered
// 36-byte reads above.  Measured on 101,568 triangles: 27 launches, 0.39 ms of kernels and one wait
// (k_sah_mid 0.13 ms), where a wave per segment of up to 128 triangles with its lanes sweeping the
// bins one after the other took 1.01 ms and the segments above that 11 launches and a host round
// trip a level, 0.66 ms of kernels.  Whole build 3.56 -> 0.98 ms; 940,800 triangles 10.3 -> 3.1 ms.
//
// Output: the binary tree layout of the LBVH path (internal nodes [0, n-1), leaf j -> n-1+j for
// the triangle at sorted position j; first/last = the sorted range an internal node covers).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "fwn_internal.h"

#pragma clang fp contract(off)

namespace fwn {

namespace {

constexpr int kSahBins = 16;
constexpr int kChunk = 1024;   // triangles per workgroup in the level-synchronous stage
constexpr int kThreads = 256;  // its threads
constexpr int kMidThreads = 512;
constexpr int kMidWaves = kMidThreads / 64;
constexpr int kRow = 16;       // largest segment of the row stage
// per-segment accumulator (ints): centroid lo[3] hi[3] (order-preserving), bin counts[16],
// bin boxes [16][lo3 hi3] (order-preserving)
constexpr int kAccCb = 0, kAccCnt = 6, kAccBox = 6 + kSahBins, kAccWords = 6 + kSahBins + 6 * kSahBins;

__device__ __forceinline__ double sah_area(const float lo[3], const float hi[3])
{
    double dx = (double)(hi[0] - lo[0]), dy = (double)(hi[1] - lo[1]), dz = (double)(hi[2] - lo[2]);
    if (dx < 0.0) return 0.0;
    return (dx * dy + dy * dz) + dz * dx;
}

// axis of the longest centroid extent (first on ties) and that extent
__device__ __forceinline__ int sah_axis(const float clo[3], const float chi[3], float* ext)
{
    int a = 0;
    float e = chi[0] - clo[0];
    if (chi[1] - clo[1] > e) {
        a = 1;
        e = chi[1] - clo[1];
    }
    if (chi[2] - clo[2] > e) {
        a = 2;
        e = chi[2] - clo[2];
    }
    *ext = e;
    return a;
}

__device__ __forceinline__ int sah_bin(float c, float clo, float sc)
{
    int b = (int)((c - clo) * sc);
    return b < 0 ? 0 : (b >= kSahBins ? kSahBins - 1 : b);
}

__device__ __forceinline__ float pick3(const float v[3], int a) { return a == 0 ? v[0] : (a == 1 ? v[1] : v[2]); }

// value of the lane D places below (shr) or above (shl) within the 16-lane row; id where there is none
template <int D>
__device__ __forceinline__ float row_shr(float v, float id)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(id), __float_as_int(v), 0x110 + D, 0xF, 0xF, false));
}
template <int D>
__device__ __forceinline__ float row_shl(float v, float id)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(id), __float_as_int(v), 0x100 + D, 0xF, 0xF, false));
}
template <int D>
__device__ __forceinline__ int row_shr(int v, int id)
{
    return __builtin_amdgcn_update_dpp(id, v, 0x110 + D, 0xF, 0xF, false);
}
template <int D>
__device__ __forceinline__ int row_shl(int v, int id)
{
    return __builtin_amdgcn_update_dpp(id, v, 0x100 + D, 0xF, 0xF, false);
}

// Best bin boundary of the row's segment (bins <= result go left) or -1, and the triangles in bins
// <= result; lane b of the row brings bin b's count and box (+inf / -inf when empty).  All lanes
// active; every lane of the row gets the result.
__device__ __forceinline__ int row_sweep(int lane, int cnt, const float blo[3], const float bhi[3], int* nleft)
{
    float ll[3], lh[3], rl[3], rh[3]; // inclusive prefixes and suffixes
    int ln = cnt, rn = cnt;
#define FWN_SCAN(D)                                                                                                 \
    ln += row_shr<D>(ln, 0);                                                                                        \
    rn += row_shl<D>(rn, 0);                                                                                        \
    for (int d = 0; d < 3; ++d) {                                                                                   \
        ll[d] = fminf(ll[d], row_shr<D>(ll[d], INFINITY));                                                          \
        lh[d] = fmaxf(lh[d], row_shr<D>(lh[d], -INFINITY));                                                         \
        rl[d] = fminf(rl[d], row_shl<D>(rl[d], INFINITY));                                                          \
        rh[d] = fmaxf(rh[d], row_shl<D>(rh[d], -INFINITY));                                                         \
    }
    for (int d = 0; d < 3; ++d) {
        ll[d] = rl[d] = blo[d];
        lh[d] = rh[d] = bhi[d];
    }
    FWN_SCAN(1)
    FWN_SCAN(2)
    FWN_SCAN(4)
    FWN_SCAN(8)
#undef FWN_SCAN
    // boundary b: bins <= b against bins > b
    float xl[3], xh[3];
    for (int d = 0; d < 3; ++d) {
        xl[d] = row_shl<1>(rl[d], INFINITY);
        xh[d] = row_shl<1>(rh[d], -INFINITY);
    }
    const int xn = row_shl<1>(rn, 0);
    double cost = INFINITY;
    if (ln != 0 && xn != 0) cost = sah_area(ll, lh) * (double)ln + sah_area(xl, xh) * (double)xn;
    if (!(cost < INFINITY)) cost = INFINITY;
    // the row's least cost, then the first lane that has it
    double best = cost;
    for (int o = 1; o < 16; o <<= 1) best = fmin(best, __shfl_xor(best, o));
    const uint32_t m = (uint32_t)(__ballot(cost == best && best < INFINITY) >> (lane & 48)) & 0xFFFFu;
    const int b = m ? __ffs(m) - 1 : -1;
    *nleft = __shfl(ln, (lane & 48) + max(b, 0));
    return b;
}

__device__ __forceinline__ float wmin(float v)
{
    for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o));
    return v;
}
__device__ __forceinline__ float wmax(float v)
{
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    return v;
}

// A segment [lo, hi) of the item array and the place it hangs in: the child `side` of internal node
// `parent`, or the root of mesh -1 - parent.
struct Seg {
    int32_t lo, hi, parent, side;
};

// The binary tree being built.
struct Tree {
    int32_t *left, *right, *parent, *first, *last, *root_bin;
    uint8_t* is_root;
    int32_t n;
};

// enters node `id` (an internal id or n - 1 + position) into its parent
__device__ __forceinline__ void hang(const Tree& t, int32_t id, int32_t parent, int32_t side)
{
    if (parent >= 0) {
        (side ? t.right : t.left)[parent] = id;
        t.parent[id] = parent;
    } else {
        t.root_bin[-1 - parent] = id;
        t.is_root[id] = 1;
        t.parent[id] = -1;
    }
}

// the internal node of a segment split at mid
__device__ __forceinline__ int32_t make_node(const Tree& t, int32_t lo, int32_t hi, int32_t mid, int32_t parent,
                                             int32_t side)
{
    const int32_t id = mid - 1;
    hang(t, id, parent, side);
    t.first[id] = lo;
    t.last[id] = hi - 1;
    return id;
}

// ---- level-synchronous stage -------------------------------------------------------------------
// Device lists of one level; two of them alternate.
struct Level {
    Seg* seg;
    int32_t* seg_fc;  // first chunk
    int32_t* acc;     // kAccWords per segment
    int32_t* ch;      // seg, lo, hi per chunk
};
// counters: segments and chunks of the level in work, [2 * parity + {0, 1}]; mid segments
enum { H_SEG = 0, H_CHUNK = 1, H_MID = 4, H_WORDS = 8 };

__global__ void k_iota(int32_t* __restrict__ p, int64_t n)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = (int32_t)i;
}

__device__ __forceinline__ int32_t acc_empty(int k)
{
    if (k < kAccCnt) return (k < 3) ? f2ord(INFINITY) : f2ord(-INFINITY);
    if (k < kAccBox) return 0;
    return ((k - kAccBox) % 6 < 3) ? f2ord(INFINITY) : f2ord(-INFINITY);
}

// first level: whole meshes, whose centroid bounds the triangle setup has (12 ints per mesh, the
// centroids' first)
__global__ void k_sah_init(Level L, int64_t nseg, const int32_t* __restrict__ boxes)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nseg * kAccWords) return;
    const int64_t s = i / kAccWords;
    const int k = (int)(i % kAccWords);
    L.acc[i] = k < kAccCnt ? boxes[12 * (int64_t)(-1 - L.seg[s].parent) + k] : acc_empty(k);
}

// the split axis (-1: middle split), bin origin and scale of an accumulator's centroid bounds
__device__ __forceinline__ int acc_axis(const int32_t* __restrict__ g, float* clo, float* sc)
{
    float lo[3], hi[3], ext;
    for (int d = 0; d < 3; ++d) {
        lo[d] = ord2f(g[kAccCb + d]);
        hi[d] = ord2f(g[kAccCb + 3 + d]);
    }
    const int ax = sah_axis(lo, hi, &ext);
    *clo = pick3(lo, ax);
    *sc = ext > 0.0f ? __fdiv_rn((float)kSahBins, ext) : 0.0f;
    return ext > 0.0f ? ax : -1;
}

__global__ __launch_bounds__(kThreads) void k_sah_bins(Level L, const int32_t* __restrict__ hdr, int par,
                                                       const int32_t* __restrict__ items,
                                                       const float* __restrict__ cen, const float* __restrict__ tbox,
                                                       int32_t* __restrict__ ch_cnt)
{
    __shared__ int32_t lcnt[kSahBins];
    __shared__ int32_t lbox[6 * kSahBins];
    const int c = blockIdx.x;
    if (c >= hdr[2 * par + H_CHUNK]) return;
    const int sg = L.ch[3 * c], a = L.ch[3 * c + 1], b = L.ch[3 * c + 2];
    int32_t* g = L.acc + (int64_t)sg * kAccWords;
    float clo, sc;
    const int ax = acc_axis(g, &clo, &sc);
    if (ax < 0) return; // uniform over the block
    const int tid = threadIdx.x;
    if (tid < kSahBins) lcnt[tid] = 0;
    if (tid < 6 * kSahBins) lbox[tid] = acc_empty(kAccBox + tid);
    __syncthreads();
    for (int i = a + tid; i < b; i += kThreads) {
        const int64_t t = items[i];
        const int bin = sah_bin(cen[3 * t + ax], clo, sc);
        atomicAdd(&lcnt[bin], 1);
        for (int d = 0; d < 3; ++d) {
            atomicMin(&lbox[6 * bin + d], f2ord(tbox[6 * t + d]));
            atomicMax(&lbox[6 * bin + 3 + d], f2ord(tbox[6 * t + 3 + d]));
        }
    }
    __syncthreads();
    if (tid < kSahBins) {
        ch_cnt[c * kSahBins + tid] = lcnt[tid];
        if (lcnt[tid] > 0) atomicAdd(g + kAccCnt + tid, lcnt[tid]);
    }
    if (tid < 6 * kSahBins && lcnt[tid / 6] > 0) {
        if ((tid % 6) < 3) atomicMin(g + kAccBox + tid, lbox[tid]);
        else atomicMax(g + kAccBox + tid, lbox[tid]);
    }
}

// One workgroup: the split of every segment of the level (16 lanes each), its node, and its children:
// segments of the next level with their chunks, or (up to kSahMid triangles) entries of the mid list,
// whose items are in array `mid_par` after the scatter.  seg_split: best boundary (-1: middle),
// split position, next-level segment of each child (-1: none).
constexpr int kNextThreads = 1024;
constexpr int kNextSegs = kNextThreads / 16;
__global__ __launch_bounds__(kNextThreads) void k_sah_next(Level L, Level N, int32_t* __restrict__ hdr, int par,
                                                           int kmid, Tree tree, int4* __restrict__ seg_split,
                                                           Seg* __restrict__ mid, int32_t* __restrict__ mid_buf)
{
    __shared__ int32_t off[3][2 * kNextSegs]; // per child: its large segment, first chunk, mid entry
    __shared__ int32_t base[3];               // of the segments before
    __shared__ int32_t tot[3];
    const int nseg = hdr[2 * par + H_SEG];
    if (nseg == 0) {
        if (threadIdx.x == 0) hdr[2 * (par ^ 1) + H_SEG] = hdr[2 * (par ^ 1) + H_CHUNK] = 0;
        return;
    }
    const int tid = threadIdx.x, lane = tid & 63, row = tid >> 4, bin = tid & 15;
    if (tid == 0) {
        base[0] = base[1] = 0;
        base[2] = hdr[H_MID];
    }
    __syncthreads();
    for (int s0 = 0; s0 < nseg; s0 += kNextSegs) {
        const int s = s0 + row;
        const bool live = s < nseg;
        const int32_t* g = L.acc + (int64_t)(live ? s : 0) * kAccWords;
        const Seg sg = L.seg[live ? s : 0];
        float clo, sc, blo[3], bhi[3];
        const int ax = acc_axis(g, &clo, &sc);
        for (int d = 0; d < 3; ++d) {
            blo[d] = ord2f(g[kAccBox + 6 * bin + d]);
            bhi[d] = ord2f(g[kAccBox + 6 * bin + 3 + d]);
        }
        int nl = 0;
        int best = row_sweep(lane, g[kAccCnt + bin], blo, bhi, &nl);
        if (ax < 0) best = -1;
        const int mid_at = best >= 0 ? sg.lo + nl : sg.lo + (sg.hi - sg.lo) / 2;
        // children: counts, then their places by an exclusive scan in segment order
        if (bin < 2) {
            const int sz = !live ? 0 : (bin == 0 ? mid_at - sg.lo : sg.hi - mid_at);
            off[0][2 * row + bin] = sz > kmid ? 1 : 0;
            off[1][2 * row + bin] = sz > kmid ? (sz + kChunk - 1) / kChunk : 0;
            off[2][2 * row + bin] = (sz > 0 && sz <= kmid) ? 1 : 0;
        }
        __syncthreads();
        if (tid < 192) { // one wave per list: 128 counts, two a lane
            const int l = tid >> 6;
            const int a = off[l][2 * lane], b = off[l][2 * lane + 1];
            int x = a + b;
            for (int o = 1; o < 64; o <<= 1) {
                const int y = __shfl_up(x, o);
                if (lane >= o) x += y;
            }
            off[l][2 * lane] = base[l] + x - a - b;
            off[l][2 * lane + 1] = base[l] + x - b;
            if (lane == 63) tot[l] = x;
        }
        __syncthreads();
        if (live && bin == 0) {
            const int32_t id = make_node(tree, sg.lo, sg.hi, mid_at, sg.parent, sg.side);
            int32_t kid[2];
            for (int h = 0; h < 2; ++h) {
                const int32_t lo = h ? mid_at : sg.lo, hi = h ? sg.hi : mid_at;
                kid[h] = -1;
                if (hi - lo > kmid) {
                    kid[h] = off[0][2 * row + h];
                    N.seg[kid[h]] = Seg{lo, hi, id, h};
                    N.seg_fc[kid[h]] = off[1][2 * row + h];
                } else {
                    mid[off[2][2 * row + h]] = Seg{lo, hi, id, h};
                    mid_buf[off[2][2 * row + h]] = par ^ 1;
                }
            }
            seg_split[s] = make_int4(best, mid_at, kid[0], kid[1]);
        }
        // the children's accumulators and chunks, 16 lanes per segment
        if (live) {
            for (int h = 0; h < 2; ++h) {
                const int32_t lo = h ? mid_at : sg.lo, hi = h ? sg.hi : mid_at;
                if (hi - lo <= kmid) continue;
                const int k = off[0][2 * row + h], c0 = off[1][2 * row + h];
                for (int w = bin; w < kAccWords; w += 16) N.acc[(int64_t)k * kAccWords + w] = acc_empty(w);
                for (int c = bin; lo + (int64_t)c * kChunk < hi; c += 16) {
                    N.ch[3 * (c0 + c)] = k;
                    N.ch[3 * (c0 + c) + 1] = lo + c * kChunk;
                    N.ch[3 * (c0 + c) + 2] = min(lo + c * kChunk + kChunk, hi);
                }
            }
        }
        __syncthreads();
        if (tid < 3) base[tid] += tot[tid];
        __syncthreads();
    }
    if (tid == 0) {
        hdr[2 * (par ^ 1) + H_SEG] = base[0];
        hdr[2 * (par ^ 1) + H_CHUNK] = base[1];
        hdr[H_MID] = base[2];
    }
}

__global__ __launch_bounds__(kThreads) void k_sah_scatter(Level L, Level N, const int32_t* __restrict__ hdr, int par,
                                                          const int4* __restrict__ seg_split,
                                                          const int32_t* __restrict__ ch_cnt,
                                                          const int32_t* __restrict__ items, int32_t* __restrict__ out,
                                                          const float* __restrict__ cen)
{
    __shared__ int32_t wl[kThreads / 64];
    __shared__ int32_t red[kThreads / 64];
    __shared__ float bnd[kThreads / 64][12];
    const int c = blockIdx.x;
    if (c >= hdr[2 * par + H_CHUNK]) return;
    const int sg = L.ch[3 * c], a = L.ch[3 * c + 1], b = L.ch[3 * c + 2];
    const int4 sp = seg_split[sg];
    const int best = sp.x;
    const int32_t mid = sp.y, lo = L.seg[sg].lo;
    float clo, sc;
    const int ax = acc_axis(L.acc + (int64_t)sg * kAccWords, &clo, &sc);
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const unsigned long long lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    int32_t relL = 0;
    if (best >= 0) { // triangles of the segment's earlier chunks that go left
        int32_t x = 0;
        for (int k = L.seg_fc[sg] + tid; k < c; k += kThreads)
            for (int q = 0; q <= best; ++q) x += ch_cnt[k * kSahBins + q];
        for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
        if (lane == 0) red[w] = x;
        __syncthreads();
        for (int k = 0; k < kThreads / 64; ++k) relL += red[k];
    }
    const int32_t relR = (a - lo) - relL;
    float cl[2][3], chh[2][3]; // centroid bounds of this thread's left and right triangles
    for (int h = 0; h < 2; ++h)
        for (int d = 0; d < 3; ++d) {
            cl[h][d] = INFINITY;
            chh[h][d] = -INFINITY;
        }
    int32_t runL = 0, runR = 0;
    for (int i0 = a; i0 < b; i0 += kThreads) {
        const int i = i0 + tid;
        const bool valid = i < b;
        const int32_t t = valid ? items[i] : 0;
        float x[3] = {0.0f, 0.0f, 0.0f};
        if (valid)
            for (int d = 0; d < 3; ++d) x[d] = cen[3 * (int64_t)t + d];
        const bool f = valid && (best >= 0 ? sah_bin(pick3(x, ax), clo, sc) <= best : i < mid);
        if (valid)
            for (int d = 0; d < 3; ++d) {
                if (f) {
                    cl[0][d] = fminf(cl[0][d], x[d]);
                    chh[0][d] = fmaxf(chh[0][d], x[d]);
                } else {
                    cl[1][d] = fminf(cl[1][d], x[d]);
                    chh[1][d] = fmaxf(chh[1][d], x[d]);
                }
            }
        if (best < 0) { // middle split: the order stays (uniform over the block)
            if (valid) out[i] = t;
            continue;
        }
        const unsigned long long m = __ballot(f);
        if (lane == 0) wl[w] = __popcll(m);
        __syncthreads();
        int woff = 0, all = 0;
        for (int k = 0; k < kThreads / 64; ++k) {
            if (k < w) woff += wl[k];
            all += wl[k];
        }
        __syncthreads();
        const int pre = woff + __popcll(m & lt); // left triangles before this one in the round
        if (valid) out[f ? lo + relL + runL + pre : mid + relR + runR + (tid - pre)] = t;
        const int nv = min(kThreads, b - i0);
        runL += all;
        runR += nv - all;
    }
    // centroid bounds of the children that are split at the next level
    if (sp.z < 0 && sp.w < 0) return;
    for (int h = 0; h < 2; ++h)
        for (int d = 0; d < 3; ++d) {
            const float mn = wmin(cl[h][d]), mx = wmax(chh[h][d]);
            if (lane == 0) {
                bnd[w][6 * h + d] = mn;
                bnd[w][6 * h + 3 + d] = mx;
            }
        }
    __syncthreads();
    if (tid < 12) {
        const int kid = tid < 6 ? sp.z : sp.w;
        const bool is_min = (tid % 6) < 3;
        if (kid >= 0) {
            float v = bnd[0][tid];
            for (int k = 1; k < kThreads / 64; ++k) v = is_min ? fminf(v, bnd[k][tid]) : fmaxf(v, bnd[k][tid]);
            int32_t* g = N.acc + (int64_t)kid * kAccWords + kAccCb + tid % 6;
            if (is_min) atomicMin(g, f2ord(v));
            else atomicMax(g, f2ord(v));
        }
    }
}

// ---- one workgroup per mid segment -----------------------------------------------------------------
struct MidEntry {
    int32_t range; // local lo | hi << 16
    int32_t parent, side;
};

__device__ __forceinline__ float perm_f(float v, int src) // value of lane `src`
{
    return __int_as_float(__builtin_amdgcn_ds_bpermute(src << 2, __float_as_int(v)));
}
__device__ __forceinline__ int perm_i(int v, int src) { return __builtin_amdgcn_ds_bpermute(src << 2, v); }
__device__ __forceinline__ float push_f(float v, int dst) // v to lane `dst`
{
    return __int_as_float(__builtin_amdgcn_ds_permute(dst << 2, __float_as_int(v)));
}

// out: the sorted triangles; one of the two item arrays (a workgroup reads its own range before it
// writes it)
__global__ __launch_bounds__(kMidThreads) void k_sah_mid(const Seg* __restrict__ mids,
                                                         const int32_t* __restrict__ mid_buf, const int32_t* items0,
                                                         const int32_t* items1, int32_t* out,
                                                         const float* __restrict__ cen, const float* __restrict__ tbox,
                                                         Tree tree)
{
    __shared__ int32_t tri[kSahMid];
    __shared__ float c3[3][kSahMid];
    __shared__ float bl[3][kSahMid];
    __shared__ float bh[3][kSahMid];
    __shared__ uint16_t perm[kSahMid];
    __shared__ uint16_t perm2[kSahMid];
    __shared__ MidEntry big[2][kSahMid / (kRow + 1) + 1];
    __shared__ MidEntry small[kSahMid / 2];
    __shared__ int32_t nbig[2], nsmall;
    __shared__ int32_t wcnt[kMidWaves][kSahBins];
    __shared__ int32_t wbox[kMidWaves][6 * kSahBins];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const Seg sg = mids[blockIdx.x];
    const int32_t* src = mid_buf[blockIdx.x] ? items1 : items0;
    const int s = sg.hi - sg.lo;
    if (s == 1) {
        if (tid == 0) {
            out[sg.lo] = src[sg.lo];
            hang(tree, tree.n - 1 + sg.lo, sg.parent, sg.side);
        }
        return;
    }
    for (int k = tid; k < s; k += kMidThreads) {
        const int64_t t = src[sg.lo + k];
        tri[k] = (int32_t)t;
        for (int d = 0; d < 3; ++d) {
            c3[d][k] = cen[3 * t + d];
            bl[d][k] = tbox[6 * t + d];
            bh[d][k] = tbox[6 * t + 3 + d];
        }
        perm[k] = (uint16_t)k;
    }
    if (tid == 0) {
        const MidEntry e{s << 16, sg.parent, sg.side};
        nbig[0] = s > kRow ? 1 : 0;
        nbig[1] = 0;
        nsmall = s > kRow ? 0 : 1;
        if (s > kRow) big[0][0] = e;
        else small[0] = e;
    }
    __syncthreads();
    // segments above 16: rounds, a wave per segment
    const unsigned long long lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (int cur = 0;; cur ^= 1) {
        const int nb = nbig[cur];
        if (nb == 0) break; // uniform: read after a barrier
        for (int q = wave; q < nb; q += kMidWaves) {
            const MidEntry en = big[cur][q];
            const int a = en.range & 0xFFFF, b = en.range >> 16;
            float clo[3] = {INFINITY, INFINITY, INFINITY}, chi[3] = {-INFINITY, -INFINITY, -INFINITY};
            for (int p = a + lane; p < b; p += 64) {
                const int k = perm[p];
                for (int d = 0; d < 3; ++d) {
                    clo[d] = fminf(clo[d], c3[d][k]);
                    chi[d] = fmaxf(chi[d], c3[d][k]);
                }
            }
            for (int d = 0; d < 3; ++d) {
                clo[d] = wmin(clo[d]);
                chi[d] = wmax(chi[d]);
            }
            float ext;
            const int ax = sah_axis(clo, chi, &ext);
            int mid = a + (b - a) / 2;
            if (ext > 0.0f) {
                const float sc = __fdiv_rn((float)kSahBins, ext), cl = pick3(clo, ax);
                if (lane < kSahBins) wcnt[wave][lane] = 0;
                for (int k = lane; k < 6 * kSahBins; k += 64) wbox[wave][k] = acc_empty(kAccBox + k);
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                for (int p = a + lane; p < b; p += 64) {
                    const int k = perm[p];
                    const int bin = sah_bin(c3[ax][k], cl, sc);
                    atomicAdd(&wcnt[wave][bin], 1);
                    for (int d = 0; d < 3; ++d) {
                        atomicMin(&wbox[wave][6 * bin + d], f2ord(bl[d][k]));
                        atomicMax(&wbox[wave][6 * bin + 3 + d], f2ord(bh[d][k]));
                    }
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                float blo[3], bhi[3];
                for (int d = 0; d < 3; ++d) {
                    blo[d] = ord2f(wbox[wave][6 * (lane & 15) + d]);
                    bhi[d] = ord2f(wbox[wave][6 * (lane & 15) + 3 + d]);
                }
                int nl = 0;
                const int best = row_sweep(lane, wcnt[wave][lane & 15], blo, bhi, &nl);
                if (best >= 0) { // the same in every row of the wave
                    mid = a + nl;
                    int runL = 0, runR = 0;
                    for (int i0 = a; i0 < b; i0 += 64) {
                        const int p = i0 + lane;
                        const bool valid = p < b;
                        const int k = valid ? perm[p] : 0;
                        const bool f = valid && sah_bin(c3[ax][k], cl, sc) <= best;
                        const unsigned long long m = __ballot(f);
                        const int pre = __popcll(m & lt);
                        if (valid) perm2[f ? a + runL + pre : mid + runR + (lane - pre)] = (uint16_t)k;
                        const int all = __popcll(m), nv = min(64, b - i0);
                        runL += all;
                        runR += nv - all;
                    }
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    for (int p = a + lane; p < b; p += 64) perm[p] = perm2[p];
                }
            }
            if (lane == 0) {
                const int32_t id = make_node(tree, sg.lo + a, sg.lo + b, sg.lo + mid, en.parent, en.side);
                for (int h = 0; h < 2; ++h) {
                    const int lo = h ? mid : a, hi = h ? b : mid;
                    const MidEntry e{lo | (hi << 16), id, h};
                    if (hi - lo == 1) hang(tree, tree.n - 1 + sg.lo + lo, id, h);
                    else if (hi - lo <= kRow) small[atomicAdd(&nsmall, 1)] = e;
                    else big[cur ^ 1][atomicAdd(&nbig[cur ^ 1], 1)] = e;
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
        __syncthreads();
        if (tid == 0) nbig[cur] = 0;
        __syncthreads();
    }
    // segments of 2 .. 16: a 16-lane row each, all its sub-segments split in parallel
    const int ns = nsmall;
    const int rbase = lane & 48, j = lane & 15;
    for (int q0 = 0; q0 < ns; q0 += kMidThreads / kRow) {
        const int q = q0 + (tid >> 4);
        const bool live = q < ns;
        const MidEntry en = small[live ? q : 0];
        const int r0 = live ? en.range & 0xFFFF : 0, m = live ? (en.range >> 16) - r0 : 0;
        const bool mine = j < m;
        int k = mine ? perm[r0 + j] : 0;
        float c[3], lo[3], hi[3];
        for (int d = 0; d < 3; ++d) {
            c[d] = c3[d][k];
            lo[d] = bl[d][k];
            hi[d] = bh[d][k];
        }
        // this lane's sub-segment [a, b) of the row and where it hangs
        int a = mine ? 0 : j, b = mine ? m : j + 1;
        int32_t par = en.parent, side = en.side;
        for (;;) {
            const int len = b - a;
            if (__ballot(len > 1) == 0ull) break;
            int mx = len; // the wave's longest sub-segment
            for (int o = 32; o > 0; o >>= 1) mx = max(mx, __shfl_xor(mx, o));
            const int maxlen = __builtin_amdgcn_readfirstlane(mx);
            float clo[3] = {c[0], c[1], c[2]}, chi[3] = {c[0], c[1], c[2]};
            for (int t = 0; t < maxlen; ++t) {
                const int from = rbase + (a + t < b ? a + t : a);
                for (int d = 0; d < 3; ++d) {
                    const float x = perm_f(c[d], from);
                    clo[d] = fminf(clo[d], x);
                    chi[d] = fmaxf(chi[d], x);
                }
            }
            float ext;
            const int ax = sah_axis(clo, chi, &ext);
            const bool split = ext > 0.0f;
            const int bin = split ? sah_bin(pick3(c, ax), pick3(clo, ax), __fdiv_rn((float)kSahBins, ext)) : 0;
            // the boundary after this lane's bin: the first minimum over all boundaries is at a
            // triangle's bin, since the ones between two bins part the triangles the same way
            float ll[3], lh[3], rl[3], rh[3];
            for (int d = 0; d < 3; ++d) {
                ll[d] = rl[d] = INFINITY;
                lh[d] = rh[d] = -INFINITY;
            }
            int ln = 0, rn = 0;
            for (int t = 0; t < maxlen; ++t) {
                const bool in = a + t < b;
                const int from = rbase + (in ? a + t : a);
                const int ob = perm_i(bin, from);
                const bool l = in && ob <= bin, r = in && ob > bin;
                ln += l ? 1 : 0;
                rn += r ? 1 : 0;
                for (int d = 0; d < 3; ++d) {
                    const float x = perm_f(lo[d], from), y = perm_f(hi[d], from);
                    if (l) {
                        ll[d] = fminf(ll[d], x);
                        lh[d] = fmaxf(lh[d], y);
                    }
                    if (r) {
                        rl[d] = fminf(rl[d], x);
                        rh[d] = fmaxf(rh[d], y);
                    }
                }
            }
            double cost = INFINITY;
            if (split && rn != 0) cost = sah_area(ll, lh) * (double)ln + sah_area(rl, rh) * (double)rn;
            if (!(cost < INFINITY)) cost = INFINITY;
            double bc = INFINITY; // the sub-segment's least cost and the first bin that has it
            int best = kSahBins;
            for (int t = 0; t < maxlen; ++t) {
                const int from = rbase + (a + t < b ? a + t : a);
                const double x = __shfl(cost, from);
                const int ob = perm_i(bin, from);
                if (x < bc || (x == bc && x < INFINITY && ob < best)) {
                    bc = x;
                    best = ob;
                }
            }
            const bool has = bc < INFINITY;
            const bool f = len > 1 && (has ? bin <= best : j < a + len / 2);
            const uint32_t seg = ((1u << b) - 1u) & ~((1u << a) - 1u);
            const uint32_t lm = (uint32_t)(__ballot(f) >> rbase) & seg;
            const uint32_t under = (1u << j) - 1u;
            const int nl = __popc(lm), mid = a + nl;
            int to = j;
            if (len > 1) to = f ? a + __popc(lm & under) : mid + __popc(seg & ~lm & under);
            // triangles to their new lanes
            k = __builtin_amdgcn_ds_permute((rbase + to) << 2, k);
            for (int d = 0; d < 3; ++d) {
                c[d] = push_f(c[d], rbase + to);
                lo[d] = push_f(lo[d], rbase + to);
                hi[d] = push_f(hi[d], rbase + to);
            }
            if (len > 1) {
                const int32_t g0 = sg.lo + r0;
                const int32_t id = g0 + mid - 1;
                if (j == a) {
                    make_node(tree, g0 + a, g0 + b, g0 + mid, par, side);
                    if (mid - a == 1) hang(tree, tree.n - 1 + g0 + a, id, 0);
                    if (b - mid == 1) hang(tree, tree.n - 1 + g0 + mid, id, 1);
                }
                side = j < mid ? 0 : 1;
                if (j < mid) b = mid;
                else a = mid;
                par = id;
            }
        }
        if (mine) perm[r0 + j] = (uint16_t)k;
    }
    __syncthreads();
    for (int p = tid; p < s; p += kMidThreads) out[sg.lo + p] = tri[perm[p]];
}

int blocks_for(int64_t n, int threads)
{
    int64_t b = (n + threads - 1) / threads;
    return (int)std::max<int64_t>(b, 1);
}

} // namespace

SahMids build_topology_sah(Engine& e, Arena& ar, const float* cen, const float* tbox, const int32_t* boxes, int64_t nF,
                           const int64_t* f_off, int M, int32_t* items, int32_t* left, int32_t* right, int32_t* parent,
                           int32_t* first, int32_t* last, uint8_t* is_root, int32_t* root_bin)
{
    hipStream_t s = e.stream;
    const int64_t n = nF;
    const Tree tree{left, right, parent, first, last, root_bin, is_root, (int32_t)n};
    // segments of a level have more than kSahMid triangles each
    const int64_t max_seg = n / (kSahMid + 1) + 1;
    const int64_t max_ch = n / kChunk + max_seg + 1;
    std::vector<Seg> large, mid0;
    std::vector<int32_t> fc, ch;
    for (int m = 0; m < M; ++m) {
        const int64_t lo = f_off[m], hi = f_off[m + 1];
        if (hi == lo) continue;
        const Seg sg{(int32_t)lo, (int32_t)hi, -1 - m, 0};
        if (hi - lo <= kSahMid) {
            mid0.push_back(sg);
            continue;
        }
        fc.push_back((int32_t)(ch.size() / 3));
        for (int64_t a = lo; a < hi; a += kChunk)
            ch.insert(ch.end(), {(int32_t)large.size(), (int32_t)a, (int32_t)std::min<int64_t>(a + kChunk, hi)});
        large.push_back(sg);
    }
    // every mid segment has at least one triangle; with no large segment they are the meshes
    const int64_t max_mid = large.empty() ? (int64_t)mid0.size() : n;
    Level lv[2];
    for (Level& L : lv) {
        L.seg = ar.take<Seg>(max_seg);
        L.seg_fc = ar.take<int32_t>(max_seg);
        L.acc = ar.take<int32_t>(max_seg * kAccWords);
        L.ch = ar.take<int32_t>(3 * max_ch);
    }
    int32_t* hdr = ar.take<int32_t>(H_WORDS);
    int4* seg_split = ar.take<int4>(max_seg);
    int32_t* ch_cnt = ar.take<int32_t>(max_ch * kSahBins);
    Seg* mid = ar.take<Seg>(max_mid);
    int32_t* mid_buf = ar.take<int32_t>(max_mid);
    int32_t* items2 = ar.take<int32_t>(n);

    // the first level's lists in one staged upload each (the stage is not touched before the sync)
    const size_t b_seg = sizeof(Seg) * large.size(), b_fc = sizeof(int32_t) * fc.size(), b_ch = sizeof(int32_t) * ch.size(),
                 b_mid = sizeof(Seg) * mid0.size(), b_buf = sizeof(int32_t) * mid0.size();
    char* hs = host_stage(e, 2 * H_WORDS * sizeof(int32_t) + b_seg + b_fc + b_ch + b_mid + b_buf);
    int32_t* hh = reinterpret_cast<int32_t*>(hs); // counters up, then down
    std::fill(hh, hh + 2 * H_WORDS, 0);
    hh[H_SEG] = (int32_t)large.size();
    hh[H_CHUNK] = (int32_t)(ch.size() / 3);
    hh[H_MID] = (int32_t)mid0.size();
    char* at = hs + 2 * H_WORDS * sizeof(int32_t);
    auto up = [&](void* dst, const void* from, size_t bytes) {
        if (bytes == 0) return;
        std::copy((const char*)from, (const char*)from + bytes, at);
        FWN_HIP(hipMemcpyAsync(dst, at, bytes, hipMemcpyHostToDevice, s));
        at += bytes;
    };
    FWN_HIP(hipMemcpyAsync(hdr, hh, H_WORDS * sizeof(int32_t), hipMemcpyHostToDevice, s));
    up(lv[0].seg, large.data(), b_seg);
    up(lv[0].seg_fc, fc.data(), b_fc);
    up(lv[0].ch, ch.data(), b_ch);
    up(mid, mid0.data(), b_mid);
    std::vector<int32_t> zero(mid0.size(), 0);
    up(mid_buf, zero.data(), b_buf);
    hipLaunchKernelGGL(k_iota, dim3(blocks_for(n, 256)), dim3(256), 0, s, items, n);
    FWN_LAUNCH_CHECK("k_iota");
    if (!large.empty()) {
        hipLaunchKernelGGL(k_sah_init, dim3(blocks_for((int64_t)large.size() * kAccWords, 256)), dim3(256), 0, s, lv[0],
                           (int64_t)large.size(), boxes);
        FWN_LAUNCH_CHECK("k_sah_init");
    }
    int64_t largest = 0;
    for (const Seg& sg : large) largest = std::max<int64_t>(largest, sg.hi - sg.lo);
    int levels = 0; // of a balanced tree, and one for uneven splits
    if (largest > 0)
        for (levels = 1; (largest >> (levels - 1)) > kSahMid; ++levels) {}
    int32_t* buf[2] = {items, items2};
    int par = 0;
    for (;;) {
        for (int k = 0; k < levels; ++k, par ^= 1) {
            hipLaunchKernelGGL(k_sah_bins, dim3((unsigned)max_ch), dim3(kThreads), 0, s, lv[par], hdr, par, buf[par],
                               cen, tbox, ch_cnt);
            FWN_LAUNCH_CHECK("k_sah_bins");
            hipLaunchKernelGGL(k_sah_next, dim3(1), dim3(kNextThreads), 0, s, lv[par], lv[par ^ 1], hdr, par,
                               (int)kSahMid, tree, seg_split, mid, mid_buf);
            FWN_LAUNCH_CHECK("k_sah_next");
            hipLaunchKernelGGL(k_sah_scatter, dim3((unsigned)max_ch), dim3(kThreads), 0, s, lv[par], lv[par ^ 1], hdr,
                               par, seg_split, ch_cnt, buf[par], buf[par ^ 1], cen);
            FWN_LAUNCH_CHECK("k_sah_scatter");
        }
        FWN_HIP(hipMemcpyAsync(hh + H_WORDS, hdr, H_WORDS * sizeof(int32_t), hipMemcpyDeviceToHost, s));
        FWN_HIP(hipStreamSynchronize(s));
        if (hh[H_WORDS + 2 * par + H_SEG] == 0) break;
        levels = 2; // uneven splits
    }
    const int64_t n_mid = hh[H_WORDS + H_MID];
    if (n_mid < 1 || n_mid > max_mid) fail(FWN_HIP_ERROR, "tree build: SAH segment count out of range");
    hipLaunchKernelGGL(k_sah_mid, dim3((unsigned)n_mid), dim3(kMidThreads), 0, s, mid, mid_buf, items, items2, items, cen,
                       tbox, tree);
    FWN_LAUNCH_CHECK("k_sah_mid");
    return SahMids{reinterpret_cast<const int32_t*>(mid), n_mid};
}

} // namespace fwn
