// Calls of few points (gfx950): the per-point API and batches of up to a few thousand points of one
// mesh, one wave per point (the batched traversals need more points to fill the chip, and a
// Morton sort first).  Compiled without machine LICM, which would hoist the FP64 constants of the
// near-field evaluation in front of every point's walk.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>

#include "fwn_eval.h"
#include "fwn_internal.h"

namespace fwn {

namespace {

__device__ __forceinline__ float readlane_f(float v, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// calls of up to kPointArgs points pass them in the kernel arguments (no read of host memory
// across the bus before the first node)
constexpr int kPointArgs = 16;
struct PointArgs {
    float q[kPointArgs][3];
};

// Depth-first walk of one point, the lanes of the wave taking the slots of a node in parallel, for
// the points whose breadth-first walk does not fit in its LDS records.  The point walks the same
// tree in the same order as in the batched traversal (children pushed in slot order, popped
// last-in-first-out), so the walk is a chain of dependent node loads; every pushed child's node is
// fetched at push time straight into the LDS buffer of its stack position (global_load_lds; the
// positions past the last buffer are read when popped).  The terms are added in the batched
// traversal's order, the FP64 near leaves (acc) in 2^-40 fixed point.  nodebuf: lds_nodes nodes.
template <int NB>
__device__ __forceinline__ float point_dfs(const uint32_t* __restrict__ slots, int width,
                                           const uint32_t* __restrict__ tris, int32_t root, int32_t root_ns, float tau,
                                           float qx, float qy, float qz, uint4* nodebuf, int lds_nodes, int lane,
                                           int32_t* __restrict__ flag, unsigned long long& acc)
{
    const int nwords = width * (kSlotWords / 4); // uint4 per node
    float om = 0.0f;
    acc = 0ull; // FP64 near leaves, 2^-40 fixed point
    if (root >= 0) {
        WaveStack<NB> S;
        S.push(0, lane, ((uint32_t)root << 4) | (uint32_t)root_ns, 0ull);
        fetch_node(slots + (size_t)root * (size_t)width * kSlotWords, nodebuf, width, lane);
        int sp = 1;
        bool overflow = false;
        while (sp > 0) {
            --sp;
            uint32_t e;
            uint64_t unused;
            S.pop(sp, e, unused);
            const int ns = (int)(e & 15u);
            if (ns == 0) continue;
            // parallel phase: lane s < ns reads, tests and (when far) expands slot s
            float w[FWN_W_LINK];
            uint32_t link = FWN_LINK_EMPTY;
            float dx = 0.0f, dy = 0.0f, dz = 0.0f, d2 = 0.0f, t = 0.0f, inv3 = 0.0f;
            bool far = false;
            const bool buffered = sp < lds_nodes;
            if (buffered) asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // this node's fetch has landed
            if (lane < ns) {
                const uint4* src = buffered ? nodebuf + (size_t)sp * nwords + lane * (kSlotWords / 4)
                                            : reinterpret_cast<const uint4*>(
                                                  slots + ((size_t)(e >> 4) * (size_t)width + lane) * kSlotWords);
                uint32_t u[kSlotWords];
#pragma unroll
                for (int k = 0; k < kSlotWords / 4; ++k) {
                    const uint4 v = src[k];
                    u[4 * k] = v.x;
                    u[4 * k + 1] = v.y;
                    u[4 * k + 2] = v.z;
                    u[4 * k + 3] = v.w;
                }
#pragma unroll
                for (int k = 0; k < FWN_W_LINK; ++k) w[k] = __uint_as_float(u[k]);
                link = u[FWN_W_LINK];
                dx = w[FWN_W_PX] - qx;
                dy = w[FWN_W_PY] - qy;
                dz = w[FWN_W_PZ] - qz;
                d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
                far = d2 > w[FWN_W_THR];
                // evaluated on every lane (used only where far): the lanes run in parallel, and
                // an unconditional use keeps all six loads of the slot in one round trip
                far_field_terms(LaneWords{w}, dx, dy, dz, d2, t, inv3);
            }
            const uint64_t farm = __ballot(far);
            // near leaves: the FP64 rule's thresholds from the leaf's first triangle (loaded before the
            // children's fetches, so that its wait does not include them)
            const bool nleaf = lane < ns && !far && (link & FWN_LINK_LEAF) != 0u;
            bool use64 = false;
            if (nleaf && tau > 0.0f) {
                const int32_t first = (int32_t)((link & ~FWN_LINK_LEAF) >> 3);
                const int32_t tcnt = (int32_t)(link & 7u) + 1;
                // words 10-11 of a 48-byte record: one 8-byte load
                const float2 np2 = *reinterpret_cast<const float2*>(tris + (size_t)first * kTriWords + FWN_T_NEAR2);
                const float nd = fmaf(dx, w[FWN_W_NX], fmaf(dy, w[FWN_W_NY], dz * w[FWN_W_NZ]));
                use64 = (d2 < np2.x) & ((tcnt > 1) | (nd * nd < np2.y)); // no short circuit: one load
            }
            const uint64_t m64 = __ballot(use64);
            // children first, in slot order, each fetched as it is pushed (before the serial sums)
            const uint64_t pushm = __ballot(lane < ns && !far && (link & FWN_LINK_LEAF) == 0u);
            for (int s2 = 0; s2 < ns; ++s2) {
                if (!((pushm >> s2) & 1ull)) continue;
                const uint32_t ls = (uint32_t)__builtin_amdgcn_readlane((int)link, s2);
                overflow |= sp >= WaveStack<NB>::kCap;
                S.push(sp, lane, ls, 0ull);
                if (sp < lds_nodes)
                    fetch_node(slots + (size_t)(ls >> 4) * (size_t)width * kSlotWords, nodebuf + (size_t)sp * nwords,
                               width, lane);
                ++sp;
            }
            // serial phase: the terms in slot order
            for (int s2 = 0; s2 < ns; ++s2) {
                if ((farm >> s2) & 1ull) {
                    om = fmaf(readlane_f(t, s2), readlane_f(inv3, s2), om);
                } else if (!((pushm >> s2) & 1ull)) {
                    const uint32_t ls = (uint32_t)__builtin_amdgcn_readlane((int)link, s2);
                    const int32_t first = (int32_t)((ls & ~FWN_LINK_LEAF) >> 3);
                    const int32_t tcnt = (int32_t)(ls & 7u) + 1;
                    if ((m64 >> s2) & 1ull) {
                        double s64 = 0.0;
                        for (int32_t k = first; k < first + tcnt; ++k)
                            s64 += tri_f64(reinterpret_cast<const float*>(tris + (size_t)k * kTriWords), qx, qy, qz);
                        acc += (unsigned long long)__double2ll_rn(s64 * kFixScale);
                    } else {
                        for (int32_t k = first; k < first + tcnt; ++k)
                            om += tri_f32(reinterpret_cast<const float*>(tris + (size_t)k * kTriWords), qx, qy, qz);
                    }
                }
            }
        }
        if (overflow && lane == 0) *flag = 1;
    }
    return om;
}

// Breadth-first single-point walk (calls of a few thousand points; the per-point API).  A depth-first
// walk is a chain of dependent node loads; here one wave per point takes the tree a level at
// a time, every slot of up to 64 / width of the level's nodes in its own lane, so the point waits
// for one load round trip per level step instead of one per node.  Each visited node gets a
// record in LDS: per slot its kind (far, near internal, near FP32 leaf, near FP64 leaf), the far
// term's t and inv3, the child's record or the FP32 leaf's triangle values.  FP64 near leaves
// are evaluated on the way and summed in 2^-40 fixed point (integer addition: any order).
//
// The FP32 terms must then be added in the batched traversal's order: a node's own terms in slot
// order (far terms, then the triangles of near leaves), followed by the subtrees of its near
// children in reverse slot order (they were pushed in slot order and are popped last first).  So
// two more level-parallel passes over the records compute, bottom up, every record's number of
// terms T (kept in its parent's slot entry, beside the other slots' own term counts, so that a
// pass reads one word per slot) and, top down, where its terms start in that order (a slot's own terms after the
// node's earlier own terms; a child's subtree after the node's own terms and the subtrees of the
// children in later slots), writing each term's pair (a, b) to that position of a list.  One
// chain of fmaf over the list gives the sum: far terms as fmaf(t, inv3, omega) and triangle
// values as fmaf(1, v, omega) = omega + v (exact product, one rounding), the same operations on
// the same values as the batched traversal, so a point gets bit for bit the value a batched call
// gives it.  A walk that needs more than max_rec records, max_tv triangle values or kBfsLevels
// levels is done again by the same wave, depth first (point_dfs, in the same LDS).
//
// Points and results: Q and done NULL for points in the kernel arguments; done (host memory): a byte
// the kernel writes after a point's results, for a few points whose results the host waits for
// directly; without it the results go to device memory and k_publish follows.
constexpr uint32_t kRecLeaf64 = 0u, kRecFar = 1u, kRecInner = 2u, kRecLeaf32 = 3u;
constexpr int kBfsLevels = 63; // level bounds live in the lanes of one register (lane L: first record of level L)
// slot entry: kind in bits 0-1; a near internal slot: child record << 2; an FP32 leaf:
// (triangles - 1) << 2 | first value << 5

// sums over aligned groups of w lanes (w = 2, 4 or 8, all lanes active; ls = lane % w): inclusive
// prefix and inclusive suffix by DPP row shifts (a group lies inside one 16-lane row, and the
// lanes a shift brings in from outside the group are masked off)
template <int D>
__device__ __forceinline__ int dpp_shr(int x) { return __builtin_amdgcn_update_dpp(0, x, 0x110 + D, 0xF, 0xF, true); }
template <int D>
__device__ __forceinline__ int dpp_shl(int x) { return __builtin_amdgcn_update_dpp(0, x, 0x100 + D, 0xF, 0xF, true); }
__device__ __forceinline__ int seg_prefix(int x, int ls, int w)
{
    int y = dpp_shr<1>(x);
    x += ls >= 1 ? y : 0;
    if (w > 2) {
        y = dpp_shr<2>(x);
        x += ls >= 2 ? y : 0;
    }
    if (w > 4) {
        y = dpp_shr<4>(x);
        x += ls >= 4 ? y : 0;
    }
    return x;
}
__device__ __forceinline__ int seg_suffix(int x, int ls, int w)
{
    int y = dpp_shl<1>(x);
    x += ls + 1 < w ? y : 0;
    if (w > 2) {
        y = dpp_shl<2>(x);
        x += ls + 2 < w ? y : 0;
    }
    if (w > 4) {
        y = dpp_shl<4>(x);
        x += ls + 4 < w ? y : 0;
    }
    return x;
}

template <int NB>
__global__ __launch_bounds__(64) void k_point_bfs(const uint32_t* __restrict__ slots, int width,
                                                  const uint32_t* __restrict__ tris, int32_t root, int32_t root_ns,
                                                  float tau, const float* __restrict__ Q, PointArgs pa, int max_rec,
                                                  int max_tv, int lds_nodes, float* __restrict__ omega,
                                                  uint8_t* __restrict__ inside, int32_t* __restrict__ flag,
                                                  uint8_t* __restrict__ done)
{
    // LDS: the list of term pairs (at most one per slot entry and FP32 value); per record its
    // node link, its parent's slot entry and its start; per slot entry its kind word (kind 0 for
    // a node's unused slots), t, inv3 and its term count (own terms; T of the child for a near
    // internal slot); the FP32 triangle values
    extern __shared__ float2 terms[];
    const int nsl = max_rec * width; // slot entries
    uint32_t* rec_node = reinterpret_cast<uint32_t*>(terms + nsl + max_tv);
    int* rec_par = reinterpret_cast<int*>(rec_node + max_rec);
    int* rec_S = rec_par + max_rec;
    uint32_t* rec_k = reinterpret_cast<uint32_t*>(rec_S + max_rec);
    float* rec_a = reinterpret_cast<float*>(rec_k + nsl);
    float* rec_b = rec_a + nsl;
    int* slot_n = reinterpret_cast<int*>(rec_b + nsl);
    float* trival = reinterpret_cast<float*>(slot_n + nsl);
    const int i = blockIdx.x;
    const int lane = threadIdx.x;
    float qx, qy, qz;
    if (Q) { // one load for the point's 12 bytes (they may lie in host memory)
        const float c = lane < 3 ? Q[3 * (size_t)i + lane] : 0.0f;
        qx = readlane_f(c, 0);
        qy = readlane_f(c, 1);
        qz = readlane_f(c, 2);
    } else {
        qx = pa.q[i][0];
        qy = pa.q[i][1];
        qz = pa.q[i][2];
    }
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const int per = 64 / width;       // nodes per step
    const int ln = lane / width;      // this lane's node within the step
    const int ls = lane - ln * width; // and slot
    float om = 0.0f;
    unsigned long long acc_lane = 0ull; // this lane's FP64 near leaves, 2^-40 fixed point
    bool redo = false;
    int lvl = 0; // lane L: the first record of level L (level L holds records [lvl_L, lvl_L+1))
    if (root >= 0) {
        if (lane == 0) {
            rec_node[0] = ((uint32_t)root << 4) | (uint32_t)root_ns;
            rec_S[0] = 0;
            rec_par[0] = -1;
        }
        __syncthreads();
        // pass 1: the walk, a level at a time
        int b = 0, e = 1, nfree = 1, tvfree = 0, nlev = 0;
        while (b < e) {
            if (nlev == kBfsLevels) {
                redo = true;
                break;
            }
            for (int c = b; c < e; c += per) {
                const int r = c + ln;
                const bool in_r = ln < per && r < e;
                const uint32_t ne = in_r ? rec_node[r] : 0u;
                const bool act = in_r && ls < (int)(ne & 15u);
                float w[FWN_W_LINK];
                uint32_t link = FWN_LINK_EMPTY;
                float dx = 0.0f, dy = 0.0f, dz = 0.0f, d2 = 0.0f, t = 0.0f, inv3 = 0.0f;
                bool far = false;
                if (act) {
                    const uint4* src =
                        reinterpret_cast<const uint4*>(slots + ((size_t)(ne >> 4) * (size_t)width + ls) * kSlotWords);
                    uint32_t u[kSlotWords];
#pragma unroll
                    for (int k = 0; k < kSlotWords / 4; ++k) {
                        const uint4 v = src[k];
                        u[4 * k] = v.x;
                        u[4 * k + 1] = v.y;
                        u[4 * k + 2] = v.z;
                        u[4 * k + 3] = v.w;
                    }
#pragma unroll
                    for (int k = 0; k < FWN_W_LINK; ++k) w[k] = __uint_as_float(u[k]);
                    link = u[FWN_W_LINK];
                    dx = w[FWN_W_PX] - qx;
                    dy = w[FWN_W_PY] - qy;
                    dz = w[FWN_W_PZ] - qz;
                    d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
                    far = d2 > w[FWN_W_THR];
                    far_field_terms(LaneWords{w}, dx, dy, dz, d2, t, inv3);
                }
                const bool inner = act && !far && (int32_t)link >= 0;
                const bool nleaf = act && !far && (int32_t)link < 0;
                // a near leaf: its first triangle's record (vertices and the FP64 rule's
                // thresholds) in one round trip
                int32_t first = 0, tcnt = 0;
                float tw[kTriWords];
                bool use64 = false;
                if (nleaf) {
                    first = (int32_t)((link & ~FWN_LINK_LEAF) >> 3);
                    tcnt = (int32_t)(link & 7u) + 1;
                    const uint4* tp = reinterpret_cast<const uint4*>(tris + (size_t)first * kTriWords);
#pragma unroll
                    for (int k = 0; k < kTriWords / 4; ++k) {
                        const uint4 v = tp[k];
                        tw[4 * k] = __uint_as_float(v.x);
                        tw[4 * k + 1] = __uint_as_float(v.y);
                        tw[4 * k + 2] = __uint_as_float(v.z);
                        tw[4 * k + 3] = __uint_as_float(v.w);
                    }
                    const float nd = fmaf(dx, w[FWN_W_NX], fmaf(dy, w[FWN_W_NY], dz * w[FWN_W_NZ]));
                    use64 = tau > 0.0f && d2 < tw[FWN_T_NEAR2] && (tcnt > 1 || nd * nd < tw[FWN_T_PLANE]);
                }
                const bool use32 = nleaf && !use64;
                // records of the near children and places for the FP32 values, in lane order
                const uint64_t im = __ballot(inner);
                const int cnt = __popcll(im);
                const int c32 = use32 ? tcnt : 0; // 1..8: four bits
                int pre = 0, tot = 0;
#pragma unroll
                for (int bit = 0; bit < 4; ++bit) {
                    const uint64_t bm = __ballot((c32 >> bit) & 1);
                    pre += __popcll(bm & lt_mask) << bit;
                    tot += __popcll(bm) << bit;
                }
                if (nfree + cnt > max_rec || tvfree + tot > max_tv) {
                    redo = true;
                    break;
                }
                const int child = nfree + __popcll(im & lt_mask);
                if (inner) {
                    rec_node[child] = link;
                    rec_par[child] = r * width + ls;
                }
                if (use32) {
                    float* tv = trival + tvfree + pre;
                    tv[0] = tri_f32(tw, qx, qy, qz);
                    for (int32_t k = 1; k < tcnt; ++k)
                        tv[k] = tri_f32(reinterpret_cast<const float*>(tris + (size_t)(first + k) * kTriWords), qx, qy, qz);
                }
                if (use64) {
                    double s64 = tri_f64(tw, qx, qy, qz);
                    for (int32_t k = 1; k < tcnt; ++k)
                        s64 += tri_f64(reinterpret_cast<const float*>(tris + (size_t)(first + k) * kTriWords), qx, qy, qz);
                    acc_lane += (unsigned long long)__double2ll_rn(s64 * kFixScale);
                }
                if (in_r) {
                    const int k = r * width + ls;
                    rec_k[k] = !act ? kRecLeaf64 : far ? kRecFar
                                   : (inner ? (kRecInner | ((uint32_t)child << 2))
                                            : (use32 ? (kRecLeaf32 | ((uint32_t)(tcnt - 1) << 2) |
                                                        ((uint32_t)(tvfree + pre) << 5))
                                                     : kRecLeaf64));
                    rec_a[k] = t;
                    rec_b[k] = inv3;
                    slot_n[k] = (act && far) ? 1 : (use32 ? (int)tcnt : 0); // internal: set by pass 2
                }
                nfree += cnt;
                tvfree += tot;
            }
            if (redo) break;
            ++nlev;
            if (lane == nlev) lvl = e; // the level just walked is [b, e); the next, [e, nfree)
            __syncthreads(); // the level's records before the next level reads them
            b = e;
            e = nfree;
        }
        if (!redo) {
            // pass 2, bottom up: T, the terms of a record's subtree, into its parent's slot entry
            int t_root = 0;
            for (int L = nlev - 1; L >= 0; --L) {
                const int lb = __builtin_amdgcn_readlane(lvl, L), le = __builtin_amdgcn_readlane(lvl, L + 1);
                for (int c = lb; c < le; c += per) {
                    const int r = c + ln;
                    const bool in_r = ln < per && r < le;
                    int n = 0, par = -1;
                    if (in_r) {
                        n = slot_n[r * width + ls];
                        par = rec_par[r];
                    }
                    n = seg_prefix(n, ls, width) + seg_suffix(n, ls, width) - n; // the group's total
                    if (in_r && ls == 0) {
                        if (par >= 0) slot_n[par] = n;
                        else t_root = n;
                    }
                }
                __syncthreads();
            }
            t_root = __builtin_amdgcn_readfirstlane(t_root); // lane 0 holds the root's record
            // pass 3, top down: where each record's terms start; each term's location in the list
            for (int L = 0; L < nlev; ++L) {
                const int lb = __builtin_amdgcn_readlane(lvl, L), le = __builtin_amdgcn_readlane(lvl, L + 1);
                for (int c = lb; c < le; c += per) {
                    const int r = c + ln;
                    const bool in_r = ln < per && r < le;
                    const int k = r * width + ls;
                    uint32_t kk = 0u;
                    int sr = 0, nk = 0;
                    float ta = 0.0f, tb = 0.0f;
                    if (in_r) { // one round trip: every word of the slot and the record's start
                        kk = rec_k[k];
                        sr = rec_S[r];
                        ta = rec_a[k];
                        tb = rec_b[k];
                        nk = slot_n[k];
                    }
                    const uint32_t kind = kk & 3u;
                    const int own = kind == kRecInner ? 0 : nk;
                    const int sub = kind == kRecInner ? nk : 0;
                    const int own_incl = seg_prefix(own, ls, width);
                    const int own_all = own_incl + seg_suffix(own, ls, width) - own; // the node's own terms
                    const int sub_incl = seg_suffix(sub, ls, width);
                    if (kind == kRecFar) {
                        terms[sr + own_incl - 1] = make_float2(ta, tb);
                    } else if (kind == kRecLeaf32) {
                        const int p0 = sr + own_incl - own;
                        const float* tv = trival + (kk >> 5);
                        for (int j = 0; j < own; ++j) terms[p0 + j] = make_float2(1.0f, tv[j]);
                    } else if (kind == kRecInner) {
                        rec_S[kk >> 2] = sr + own_all + sub_incl - sub;
                    }
                }
                __syncthreads();
            }
            // the sum, in list order: one fmaf per term (every lane runs the chain on broadcast
            // reads, 16 reads in flight ahead of their fmaf)
            const int nt = min(t_root, nsl + max_tv); // at most one term per slot entry and value
            int j = 0;
            for (; j + 16 <= nt; j += 16) {
                float2 v[16];
#pragma unroll
                for (int u = 0; u < 16; ++u) v[u] = terms[j + u];
#pragma unroll
                for (int u = 0; u < 16; ++u) om = fmaf(v[u].x, v[u].y, om);
            }
            for (; j < nt; ++j) {
                const float2 v = terms[j];
                om = fmaf(v.x, v.y, om);
            }
        }
    }
    unsigned long long acc = 0ull;
    if (redo) { // more records than the LDS holds: the same point depth first
        __syncthreads();
        om = point_dfs<NB>(slots, width, tris, root, root_ns, tau, qx, qy, qz, reinterpret_cast<uint4*>(terms),
                           lds_nodes, lane, flag, acc);
    } else { // the wave's FP64 sum
        for (uint64_t m = __ballot(acc_lane != 0ull); m != 0ull; m &= m - 1ull) {
            const int l = (int)__builtin_ctzll(m);
            const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)acc_lane, l);
            const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(acc_lane >> 32), l);
            acc += ((unsigned long long)hi << 32) | lo;
        }
    }
    const long long v = (long long)acc;
    if (v != 0) om = (float)((double)om + (double)v * (1.0 / kFixScale));
    if (lane == 0) {
        omega[i] = om;
        if (inside) inside[i] = ((double)om / (4.0 * 3.14159265358979323846) > 0.5) ? 1 : 0;
        if (done) { // the host waits on this byte: the results and the overflow flag go first
            __threadfence_system();
            *(volatile uint8_t*)(done + i) = 1;
        }
    }
}

// End of a host call whose results were collected in device memory: copies them to the pinned stage,
// reports and clears the overflow flag, then writes the word the host waits for.  One workgroup,
// 16 bytes a thread and step over the bus.
__global__ __launch_bounds__(1024) void k_publish(const uint4* __restrict__ om, int64_t om16,
                                                  const uint4* __restrict__ in, int64_t in16, uint4* __restrict__ hom,
                                                  uint4* __restrict__ hin, int32_t* __restrict__ flag,
                                                  int32_t* __restrict__ hflag, volatile uint32_t* __restrict__ hdone,
                                                  uint32_t token)
{
    for (int64_t k = threadIdx.x; k < om16; k += 1024) hom[k] = om[k];
    for (int64_t k = threadIdx.x; k < in16; k += 1024) hin[k] = in[k];
    if (threadIdx.x == 0) {
        *hflag = *flag;
        *flag = 0;
    }
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) *hdone = token;
}

__global__ void k_clear(int32_t* p) { *p = 0; }

// results of up to this many points go straight to host memory, each wave writing its own and a
// done byte (three bus writes a point); more are collected in device memory first
constexpr int64_t kPointDirect = 128;
// LDS of a k_point_bfs wave: as much as lets all waves of the call be resident, within these bounds
// (a point's walk takes 108 bytes a visited 4-wide node and 12 an FP32 triangle)
constexpr size_t kPointLdsMax = 65536, kPointLdsMin = 20480;

} // namespace

// Few points of a single-mesh engine.  Host calls of up to 2,048 points record no device time.
void run_points(Engine& e, const float* Q, int64_t nQ, float* omega, uint8_t* inside, int banks, bool dev)
{
    hipStream_t s = e.stream;
    const bool direct = !dev && nQ <= kPointDirect;
    const bool timed = dev || nQ > 2048;
    auto up16 = [](size_t b) { return (b + 15) & ~(size_t)15; };
    const size_t done_b = up16(direct ? (size_t)nQ : 4);
    const size_t pts_b = dev ? 0 : up16(sizeof(float) * 3 * (size_t)nQ);
    const size_t om_b = dev ? 0 : up16(sizeof(float) * (size_t)nQ), in_b = dev ? 0 : up16((size_t)nQ);
    // stage: overflow flag (16 B), done bytes or word, points, omega, inside
    char* hs = host_stage(e, 16 + done_b + pts_b + om_b + in_b);
    int32_t* hflag = reinterpret_cast<int32_t*>(hs);
    uint8_t* hdone = reinterpret_cast<uint8_t*>(hs + 16);
    float* hq = reinterpret_cast<float*>(hs + 16 + done_b);
    float* hom = reinterpret_cast<float*>(hs + 16 + done_b + pts_b);
    uint8_t* hin = reinterpret_cast<uint8_t*>(hs + 16 + done_b + pts_b + om_b);
    *hflag = 0;
    std::memset(hdone, 0, done_b);
    PointArgs pa;
    std::memset(&pa, 0, sizeof(pa));
    const float* dq = Q; // device points, points in the pinned stage, or in the arguments (nullptr)
    if (!dev) {
        dq = nullptr;
        if (nQ <= kPointArgs) {
            std::memcpy(pa.q, Q, sizeof(float) * 3 * (size_t)nQ);
        } else {
            std::memcpy(hq, Q, sizeof(float) * 3 * (size_t)nQ);
            dq = hq;
        }
    }
    float* dom = omega;
    uint8_t* din = inside;
    int32_t* dflag = hflag;
    if (direct) {
        dom = hom;
        din = hin;
    } else if (!dev) {
        if (!e.q_ptflag.p) { // kept zero between calls
            e.q_ptflag.alloc(sizeof(int32_t));
            hipLaunchKernelGGL(k_clear, dim3(1), dim3(1), 0, s, e.q_ptflag.as<int32_t>());
            FWN_LAUNCH_CHECK("k_clear");
        }
        dflag = e.q_ptflag.as<int32_t>();
        e.q_om.reserve(om_b);
        dom = e.q_om.as<float>();
        e.q_in8.reserve(in_b);
        din = inside ? e.q_in8.as<uint8_t>() : nullptr;
    }
    if (timed) {
        if (!e.ev[0])
            for (int k = 0; k < 4; ++k) FWN_HIP(hipEventCreate(&e.ev[k]));
        FWN_HIP(hipEventRecord(e.ev[0], s));
    }
    const int32_t root = e.h_roots[0], root_ns = e.h_roots[1];
    const float tau = e.h_tau[0];
    const size_t per_cu = (size_t)((nQ + 255) / 256);
    const size_t lds = std::min(kPointLdsMax, std::max(kPointLdsMin, (size_t)163840 / per_cu & ~(size_t)1023));
    const int max_tv = (int)(lds / 64);
    const int max_rec = (int)((lds / sizeof(uint32_t) - 3 * (size_t)max_tv) / (size_t)(3 + 6 * e.width));
    const int lds_nodes = (int)(lds / ((size_t)e.width * kSlotWords * sizeof(uint32_t)));
#define FWN_POINT(NB)                                                                                               \
    hipLaunchKernelGGL(k_point_bfs<NB>, dim3((unsigned)nQ), dim3(64), lds, s, e.slots.as<uint32_t>(), e.width,     \
                       e.tris.as<uint32_t>(), root, root_ns, tau, dq, pa, max_rec, max_tv, lds_nodes, dom, din,    \
                       dflag, direct ? hdone : nullptr)
    if (banks == 1) FWN_POINT(1);
    else FWN_POINT(3);
#undef FWN_POINT
    FWN_LAUNCH_CHECK("k_point_bfs");
    if (timed) FWN_HIP(hipEventRecord(e.ev[3], s));
    if (!dev && !direct) {
        hipLaunchKernelGGL(k_publish, dim3(1), dim3(1024), 0, s, e.q_om.as<uint4>(), (int64_t)(om_b / 16),
                           e.q_in8.as<uint4>(), (int64_t)(inside ? in_b / 16 : 0), reinterpret_cast<uint4*>(hom),
                           reinterpret_cast<uint4*>(hin), dflag, hflag, reinterpret_cast<uint32_t*>(hdone), 1u);
        FWN_LAUNCH_CHECK("k_publish");
    }
    // host results are waited for by polling the bytes (or word) written after them: no stream
    // synchronisation in the round trip.  Every 256 polls the stream is asked whether it has
    // finished, so a failed launch ends the wait.
    if (dev) {
        FWN_HIP(hipStreamSynchronize(s));
    } else {
        const volatile uint8_t* vd = hdone;
        const int64_t n = direct ? nQ : 1;
        bool polled = false;
        int64_t k = 0;
        for (uint32_t spin = 1;; ++spin) {
            while (k < n && vd[k] != 0) ++k;
            if (k == n) {
                polled = true;
                break;
            }
            if ((spin & 255u) == 0u && hipStreamQuery(s) != hipErrorNotReady) break;
        }
        std::atomic_thread_fence(std::memory_order_acquire);
        if (!polled) FWN_HIP(hipStreamSynchronize(s));
    }
    if (*hflag) fail(FWN_LIMIT_EXCEEDED, "traversal stack overflow");
    if (!dev) {
        std::memcpy(omega, hom, sizeof(float) * (size_t)nQ);
        if (inside) std::memcpy(inside, hin, (size_t)nQ);
    }
    e.last_traverse_ms = 0.0;
    e.last_total_ms = 0.0;
    if (timed) {
        float t = 0.0f;
        FWN_HIP(hipEventSynchronize(e.ev[3]));
        FWN_HIP(hipEventElapsedTime(&t, e.ev[0], e.ev[3]));
        e.last_traverse_ms = t;
        e.last_total_ms = t;
    }
}

} // namespace fwn
