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
        if (overflow && lane == 0) { // never with the host's stack bound
            *flag = 1;
            __threadfence_system(); // before the mark of a packed result
        }
    }
    return om;
}

// Breadth-first single-point walk (calls of a few thousand points; the per-point API).  A depth-first
// walk is a chain of dependent node loads; here one wave per point takes the waiting nodes 64 / W at
// a time, every slot in its own lane (W = tree width), so the point waits for one load round trip
// per step (about one per tree level) instead of one per node.  Each visited node gets a record in
// LDS, in visiting order: its link, its number of FP32 terms and of near children (whose records are
// consecutive, in slot order), and per slot the pair (a, b) that the term adds as fmaf(a, b, omega)
// (far terms (t, inv3); a near FP32 triangle (1, value); the values of a larger bucket are kept
// apart).  FP64 near leaves are evaluated on the way and summed in 2^-40 fixed point (integer
// addition: any order).
//
// The FP32 terms must then be added in the batched traversal's order: a node's own terms in slot
// order, followed by the subtrees of its near children in reverse slot order (they were pushed in
// slot order and are popped last first).  Two passes over the levels, a lane per record, count each
// subtree's terms bottom up and hand out the records' places top down; the terms are moved to their
// places in a list, 64 / W records a step, and one chain of fmaf over the list gives the sum: the
// same operations on the same values as the batched traversal, so a point gets bit for bit the value
// a batched call gives it.  A walk that needs more than max_rec records, max_tv bucket values or 63
// levels is done again by the same wave, depth first (point_dfs, in the same LDS).
//
// Points: Q, or the kernel arguments (Q NULL).  Results: packed (host memory): one 8-byte store a
// point with omega, the inside flag and a mark the host waits for; otherwise omega and inside.
//
// Bound: latency of one wave's dependent steps for a call of few points (8.8 us of kernel for a random
// point of 199,692 triangles, 10.3 with slot-wise counting passes and a system fence before a done
// byte), VALU issue and LDS space for thousands.  Fetching the top three levels into LDS at the start
// (one round trip instead of three) was measured and not kept: 9.0 us.

// sums over aligned groups of W lanes (2, 4 or 8; all lanes active; ls = lane % W): inclusive prefix
// by DPP row shifts (a group lies inside one 16-lane row, and the lanes a shift brings in from
// outside the group are masked off)
template <int D>
__device__ __forceinline__ int dpp_shr(int x) { return __builtin_amdgcn_update_dpp(0, x, 0x110 + D, 0xF, 0xF, true); }
template <int W>
__device__ __forceinline__ int seg_prefix(int x, int ls)
{
    int y = dpp_shr<1>(x);
    x += ls >= 1 ? y : 0;
    if (W > 2) {
        y = dpp_shr<2>(x);
        x += ls >= 2 ? y : 0;
    }
    if (W > 4) {
        y = dpp_shr<4>(x);
        x += ls >= 4 ? y : 0;
    }
    return x;
}

// LDS bytes of a record (list places and pairs of its slots, their words, link, info, place, count) and
// of a bucket value (its place in the list and itself)
constexpr size_t point_rec_bytes(int W) { return (size_t)W * 20 + 16; }
constexpr size_t kPointValueBytes = 12;

template <int W, int NB>
__global__ __launch_bounds__(64) void k_point_bfs(const uint32_t* __restrict__ slots,
                                                  const uint32_t* __restrict__ tris, int32_t root, int32_t root_ns,
                                                  float tau, const float* __restrict__ Q, PointArgs pa, int max_rec,
                                                  int max_tv, int lds_nodes, float* __restrict__ omega,
                                                  uint8_t* __restrict__ inside, int32_t* __restrict__ flag,
                                                  uint64_t* __restrict__ packed)
{
    constexpr int kPer = 64 / W;                     // nodes per step
    constexpr uint32_t kGroup = (1u << W) - 1u;
    extern __shared__ uint4 lds[];
    const int nsl = max_rec * W; // slot entries
    float2* terms = reinterpret_cast<float2*>(lds);                // the list
    float2* slot_ab = terms + nsl + max_tv;                        // per slot its pair
    uint32_t* slot_w = reinterpret_cast<uint32_t*>(slot_ab + nsl); // terms | offset in the record << 4 | value << 12
    uint32_t* rec_node = slot_w + nsl;
    uint32_t* rec_info = rec_node + max_rec; // own terms | near children << 8 | first child's record << 16
    int* rec_S = reinterpret_cast<int*>(rec_info + max_rec);
    int* rec_T = rec_S + max_rec;
    float* trival = reinterpret_cast<float*>(rec_T + max_rec);
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
    const int ln = lane / W;      // this lane's node within the step
    const int ls = lane - ln * W; // and slot
    float om = 0.0f;
    unsigned long long acc_lane = 0ull; // this lane's FP64 near leaves, 2^-40 fixed point
    bool redo = false;
    uint32_t lvl = 0u; // lane L: the first record of level L
    const uint64_t before = (1ull << (ln * W)) - 1ull; // lanes of the step's earlier nodes
    if (root >= 0) {
        if (lane == 0) rec_node[0] = ((uint32_t)root << 4) | (uint32_t)root_ns;
        __syncthreads();
        int nrec = 1, ntv = 0; // records and bucket values so far
        int nlev = 0, next = 1; // levels finished, first record of the level after this one
        for (int c = 0; c < nrec;) {
            const int took = min(kPer, next - c); // of the level's nodes
            const int r = c + ln;
            const bool in_r = ln < took;
            const uint32_t ne = in_r ? rec_node[r] : 0u;
            const bool act = in_r && ls < (int)(ne & 15u);
            uint4 x[kSlotWords / 4];
            if (act) {
                const uint4* src =
                    reinterpret_cast<const uint4*>(slots + ((size_t)(ne >> 4) * (size_t)W + ls) * kSlotWords);
#pragma unroll
                for (int k = 0; k < kSlotWords / 4; ++k) x[k] = src[k];
            }
            float w[FWN_W_LINK];
#pragma unroll
            for (int k = 0; k < FWN_W_LINK; ++k) w[k] = __uint_as_float(reinterpret_cast<const uint32_t*>(x)[k]);
            const uint32_t link = x[5].w;
            const float dx = w[FWN_W_PX] - qx, dy = w[FWN_W_PY] - qy, dz = w[FWN_W_PZ] - qz;
            const float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
            const bool far = act && d2 > w[FWN_W_THR];
            const bool inner = act && !far && (int32_t)link >= 0;
            const bool nleaf = act && !far && (int32_t)link < 0;
            float ta = 0.0f, tb = 0.0f;
            if (far) far_field_terms(LaneWords{w}, dx, dy, dz, d2, ta, tb);
            // records of the near children, in lane order
            const uint64_t im = __ballot(inner);
            const int cnt = __popcll(im);
            int n = far ? 1 : 0; // FP32 terms of the slot
            int32_t first = 0;
            bool use64 = false;
            float v0 = 0.0f;
            const uint64_t leafm = __ballot(nleaf);
            if (leafm != 0ull) {
                if (nleaf) {
                    // the first triangle's record (vertices, the FP64 rule's thresholds) in one round trip
                    first = (int32_t)((link & ~FWN_LINK_LEAF) >> 3);
                    const int32_t tcnt = (int32_t)(link & 7u) + 1;
                    const uint4* tp = reinterpret_cast<const uint4*>(tris + (size_t)first * kTriWords);
                    float tw[kTriWords];
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
                    if (use64) {
                        double s64 = tri_f64(tw, qx, qy, qz);
                        for (int32_t k = 1; k < tcnt; ++k)
                            s64 += tri_f64(reinterpret_cast<const float*>(tris + (size_t)(first + k) * kTriWords), qx,
                                           qy, qz);
                        acc_lane += (unsigned long long)__double2ll_rn(s64 * kFixScale);
                    } else {
                        n = tcnt;
                        v0 = tri_f32(tw, qx, qy, qz);
                        ta = 1.0f;
                        tb = v0;
                    }
                }
            }
            // the slot's terms within its record
            const uint64_t big = __ballot(n > 1);
            int off, own, tv = 0, tot = 0;
            if (big == 0ull) {
                const uint32_t g = (uint32_t)(__ballot(n == 1) >> (ln * W)) & kGroup;
                off = __popc(g & ((1u << ls) - 1u));
                own = __popc(g);
            } else { // buckets: their values get places in the value array, in lane order
                const int incl = seg_prefix<W>(n, ls);
                off = incl - n;
                own = __shfl(incl, ln * W + W - 1);
                const int nb = n > 1 ? n : 0; // 2..8: four bits
#pragma unroll
                for (int bit = 0; bit < 4; ++bit) {
                    const uint64_t bm = __ballot((nb >> bit) & 1);
                    tv += __popcll(bm & lt_mask) << bit;
                    tot += __popcll(bm) << bit;
                }
                tv += ntv;
            }
            if (nrec + cnt > max_rec || ntv + tot > max_tv) {
                redo = true;
                break;
            }
            if (n > 1) {
                trival[tv] = v0;
                for (int32_t k = 1; k < n; ++k)
                    trival[tv + k] = tri_f32(reinterpret_cast<const float*>(tris + (size_t)(first + k) * kTriWords), qx,
                                             qy, qz);
            }
            if (inner) rec_node[nrec + __popcll(im & lt_mask)] = link;
            if (in_r) {
                slot_ab[r * W + ls] = make_float2(ta, tb);
                slot_w[r * W + ls] = (uint32_t)n | ((uint32_t)off << 4) | ((uint32_t)tv << 12);
                if (ls == 0)
                    rec_info[r] = (uint32_t)own | ((uint32_t)__popc((uint32_t)(im >> (ln * W)) & kGroup) << 8) |
                                  ((uint32_t)(nrec + __popcll(im & before)) << 16);
            }
            __syncthreads(); // the step's records before the next step reads them
            nrec += cnt;
            ntv += tot;
            c += took;
            if (c == next) { // the level is done
                ++nlev;
                lvl = wave_writelane((uint32_t)c, nlev, lvl);
                next = nrec;
                if (nlev == 63 && c < nrec) {
                    redo = true;
                    break;
                }
            }
        }
        if (!redo) {
            // bottom up, a lane per record: the terms T of a record's subtree
            for (int L = nlev - 1; L >= 0; --L) {
                const int lb = __builtin_amdgcn_readlane(lvl, L), le = __builtin_amdgcn_readlane(lvl, L + 1);
                for (int r = lb + lane; r < le; r += 64) {
                    const uint32_t in = rec_info[r];
                    const int kids = (int)(in >> 8) & 15, f = (int)(in >> 16);
                    int T = (int)(in & 255u);
#pragma unroll
                    for (int k = 0; k < W; ++k) T += k < kids ? rec_T[f + k] : 0;
                    rec_T[r] = T;
                }
                __syncthreads();
            }
            const int nt = rec_T[0]; // at most one term per slot entry and bucket value
            // top down: where a record's terms start; its children's follow its own, last child first
            if (lane == 0) rec_S[0] = 0;
            for (int L = 0; L < nlev; ++L) {
                const int lb = __builtin_amdgcn_readlane(lvl, L), le = __builtin_amdgcn_readlane(lvl, L + 1);
                for (int r = lb + lane; r < le; r += 64) {
                    const uint32_t in = rec_info[r];
                    const int kids = (int)(in >> 8) & 15, f = (int)(in >> 16);
                    int S = rec_S[r] + (int)(in & 255u);
#pragma unroll
                    for (int k = W - 1; k >= 0; --k)
                        if (k < kids) {
                            rec_S[f + k] = S;
                            S += rec_T[f + k];
                        }
                }
                __syncthreads();
            }
            // the terms to their places
            for (int c = 0; c < nrec; c += kPer) {
                const int r = c + ln;
                if (r < nrec) {
                    const uint32_t sw = slot_w[r * W + ls];
                    const float2 ab = slot_ab[r * W + ls];
                    const int n = (int)(sw & 15u), p0 = rec_S[r] + (int)((sw >> 4) & 255u);
                    if (n == 1) {
                        terms[p0] = ab;
                    } else if (n > 1) {
                        const float* tv = trival + (sw >> 12);
                        for (int j = 0; j < n; ++j) terms[p0 + j] = make_float2(1.0f, tv[j]);
                    }
                }
            }
            __syncthreads();
            // the sum, in list order: one fmaf per term (every lane runs the chain on broadcast
            // reads, 16 terms in flight ahead of their fmaf)
            const float4* two = reinterpret_cast<const float4*>(terms);
            int j = 0;
            for (; j + 16 <= nt; j += 16) {
                float4 v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = two[j / 2 + u];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    om = fmaf(v[u].x, v[u].y, om);
                    om = fmaf(v[u].z, v[u].w, om);
                }
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
        om = point_dfs<NB>(slots, W, tris, root, root_ns, tau, qx, qy, qz, lds, lds_nodes, lane, flag, acc);
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
    const uint32_t in = ((double)om / (4.0 * 3.14159265358979323846) > 0.5) ? 1u : 0u;
    if (lane == 0) {
        if (packed) { // omega, the flag and the mark in one store, the wave's last access to the pinned stage
            __hip_atomic_store(packed + i, (uint64_t)__float_as_uint(om) | ((uint64_t)(2u | in) << 32),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        } else {
            omega[i] = om;
            if (inside) inside[i] = (uint8_t)in;
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
    if (threadIdx.x == 0) *hdone = token; // the last access to the pinned stage
}

__global__ void k_clear(int32_t* p) { *p = 0; }

// Results of up to this many points go straight to host memory, one 8-byte store each; more are
// collected in device memory first.  Host calls in us, stored / collected: 129 points 30.0 / 35.3 (F =
// 20,172) and 32.6 / 37.6 (F = 874,800), 512 33.0 / 38.0 and 35.6 / 39.9, 2,048 37.0 / 40.4 and 39.7 / 44.0
constexpr int64_t kPointDirect = 2048;
// LDS of a k_point_bfs wave: as much as lets all waves of the call be resident, within these bounds
constexpr size_t kPointLdsMax = 65536, kPointLdsMin = 20480;

template <int W>
void launch_points(Engine& e, int banks, int64_t nQ, const float* dq, const PointArgs& pa, float* omega,
                   uint8_t* inside, int32_t* flag, uint64_t* packed, hipStream_t s)
{
    const size_t per_cu = (size_t)((nQ + 255) / 256);
    const size_t lds = std::min(kPointLdsMax, std::max(kPointLdsMin, (size_t)163840 / per_cu & ~(size_t)1023));
    const int lds_nodes = (int)(lds / ((size_t)W * kSlotWords * 4));
    const int max_tv = e.opt.leaf_max > 1 ? (int)(lds / 64) : 0;
    const int max_rec = (int)((lds - max_tv * kPointValueBytes) / point_rec_bytes(W));
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)nQ), dim3(64), lds, s, e.slots.as<uint32_t>(), e.tris.as<uint32_t>(),
                           e.h_roots[0], e.h_roots[1], e.h_tau[0], dq, pa, max_rec, max_tv, lds_nodes, omega,
                           inside, flag, packed);
        FWN_LAUNCH_CHECK("k_point_bfs");
    };
    if (banks == 1) go(k_point_bfs<W, 1>);
    else go(k_point_bfs<W, 3>);
}

} // namespace

// Few points of a single-mesh engine.  Host calls of up to 2,048 points record no device time.
void run_points(Engine& e, const float* Q, int64_t nQ, float* omega, uint8_t* inside, int banks, bool dev)
{
    hipStream_t s = e.stream;
    const bool direct = !dev && nQ <= kPointDirect;
    const bool timed = dev || nQ > 2048;
    auto up16 = [](size_t b) { return (b + 15) & ~(size_t)15; };
    const size_t pts_b = dev ? 0 : up16(sizeof(float) * 3 * (size_t)nQ);
    const size_t om_b = dev || direct ? 0 : up16(sizeof(float) * (size_t)nQ), in_b = dev || direct ? 0 : up16((size_t)nQ);
    const size_t done_b = direct ? sizeof(uint64_t) * (size_t)kPointDirect : 16;
    // stage: overflow flag (16 B), packed results or the done word, points, omega, inside
    char* hs = host_stage(e, 16 + done_b + pts_b + om_b + in_b);
    int32_t* hflag = reinterpret_cast<int32_t*>(hs);
    uint64_t* hdone = reinterpret_cast<uint64_t*>(hs + 16);
    float* hq = reinterpret_cast<float*>(hs + 16 + done_b);
    float* hom = reinterpret_cast<float*>(hs + 16 + done_b + pts_b);
    uint8_t* hin = reinterpret_cast<uint8_t*>(hs + 16 + done_b + pts_b + om_b);
    *hflag = 0;
    std::memset(hdone, 0, direct ? sizeof(uint64_t) * (size_t)nQ : 8);
    PointArgs pa;
    const float* dq = Q; // device points, points in the pinned stage, or in the arguments (nullptr)
    if (!dev) {
        if (nQ <= kPointArgs) {
            std::memset(&pa, 0, sizeof(pa));
            std::memcpy(pa.q, Q, sizeof(float) * 3 * (size_t)nQ);
            dq = nullptr;
        } else {
            std::memcpy(hq, Q, sizeof(float) * 3 * (size_t)nQ);
            dq = hq;
        }
    }
    float* dom = omega;
    uint8_t* din = inside;
    int32_t* dflag = hflag;
    if (!dev && !direct) {
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
    uint64_t* packed = direct ? hdone : nullptr;
    if (e.width == 4) launch_points<4>(e, banks, nQ, dq, pa, dom, din, dflag, packed, s);
    else if (e.width == 2) launch_points<2>(e, banks, nQ, dq, pa, dom, din, dflag, packed, s);
    else launch_points<8>(e, banks, nQ, dq, pa, dom, din, dflag, packed, s);
    if (timed) FWN_HIP(hipEventRecord(e.ev[3], s));
    if (!dev && !direct) {
        hipLaunchKernelGGL(k_publish, dim3(1), dim3(1024), 0, s, e.q_om.as<uint4>(), (int64_t)(om_b / 16),
                           e.q_in8.as<uint4>(), (int64_t)(inside ? in_b / 16 : 0), reinterpret_cast<uint4*>(hom),
                           reinterpret_cast<uint4*>(hin), dflag, hflag, reinterpret_cast<uint32_t*>(hdone), 1u);
        FWN_LAUNCH_CHECK("k_publish");
    }
    // host results are waited for by polling the marks (or the word) that arrive with them: no stream
    // synchronisation in the round trip.  Every 256 polls the stream is asked whether it has
    // finished, so a failed launch ends the wait.
    if (dev) {
        FWN_HIP(hipStreamSynchronize(s));
    } else {
        const volatile uint64_t* vd = hdone;
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
    if (direct) {
        for (int64_t k = 0; k < nQ; ++k) {
            const uint32_t w = (uint32_t)hdone[k];
            std::memcpy(omega + k, &w, sizeof(w));
            if (inside) inside[k] = (uint8_t)((hdone[k] >> 32) & 1u);
        }
    } else if (!dev) {
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
