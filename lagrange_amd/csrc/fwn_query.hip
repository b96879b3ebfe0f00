// Winding number queries on gfx950.
//
// Replaces UT_SolidAngle<float,float>::computeSolidAngle, called per point by the reference at
// modules/winding/src/FastWindingNumber.cpp:66 (is_inside) and :75 (solid_angle), and the
// per-voxel loop of modules/volume/src/mesh_to_volume.cpp:167-183 that issues those calls.
//
// Points are sorted by mesh and 30-bit Morton code, then each wave64 takes 64 consecutive
// points (one per lane) and walks its mesh's wide tree once for all of them:
//  * the wave pops a (node, lane mask) pair from a wave-private stack held in three VGPRs
//    (entry i lives in lane i%64 of bank i/64; pushes are v_writelane, pops v_readlane), so
//    node ids and masks stay scalar and slot/triangle loads are scalar (s_load) broadcasts;
//  * for every slot each active lane tests |q - p|^2 > beta^2 r2: far lanes add the order-2
//    expansion, near lanes either take the exact triangle solid angles (leaf slot) or stay
//    active in the child pushed with their mask;
//  * a lane's own sequence of tests, far terms and triangles is exactly the single-point
//    traversal (children pushed in slot order, popped last-in-first-out), so each point gets
//    the same result the per-point reference loop would give on this tree.
// Triangles closer than tau (near_fp64_rel x bbox diagonal) to the leaf's bounding sphere
// use the FP64 van Oosterom-Strackee formula, 64 leaves at a time from a queue in LDS.
//
// Bound: VALU issue for points close together (16.7M grid points, F = 940,800: 98 % of the issue
// slots).  Compiled without machine LICM, which would hold the FP64 constants in 45 vector registers
// through the walk (112 registers, 4 waves per SIMD, instead of 61 and 8).  Before the queue, FP64
// leaves went to a work list in memory for two more kernels, its slots claimed 64 at a time from one
// counter, which points near the surface saturated: 4M of them, F = 199,692, 4.30 -> 2.29 ms (the
// three kernels 3.44 + 0.30 + 0.27 -> 2.05 ms), the grid 3.54 -> 3.52 ms.
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstring>
#include <thread>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "fwn_eval.h"
#include "fwn_internal.h"
#include "fwn_order.h"

namespace fwn {

namespace {

constexpr int QT = 256; // key kernel threads

// a value equal in every lane of the wave, made visibly uniform (scalar registers)
__device__ __forceinline__ int64_t wave_uniform64(int64_t v)
{
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
}

// The key of point i.  Only leading bits of the keys are sorted: a wave needs its points close together,
// not in exact curve order, and every point's result is independent of which points share its wave.
__device__ __forceinline__ uint32_t point_key(const float* __restrict__ Q, int64_t nQ, int64_t i,
                                              const int64_t* __restrict__ q_off, int M, int mesh_bits, int first,
                                              const float* __restrict__ minfo)
{
    int m = 0;
    if (M > 1) {
        // the wave's first and last points (wave-uniform: scalar loads); only a wave that spans a
        // mesh boundary searches per lane
        const int64_t w0 = wave_uniform64(i - (threadIdx.x & 63));
        const int m0 = mesh_of64(q_off, M, w0), m1 = mesh_of64(q_off, M, wave_uniform64(min(w0 + 63, nQ - 1)));
        m = (m0 == m1) ? m0 : mesh_of64(q_off, M, i);
    }
    const float* mi = minfo + 8 * m;
    // the sort's first pass takes the values to be the positions i
    return point_key_of(morton30(Q[3 * i], Q[3 * i + 1], Q[3 * i + 2], mi, mi + 3), (uint32_t)m, mesh_bits, first);
}

// A look at the n points of one mesh, Q[0..n), by the first blocks of the kernel that makes the keys: how many of
// 2^kLookBits cells of the mesh's box hold one of as many of them, and for kLookWalks points (depth > 0) the
// threshold of the last slot of a walk from the root of a 4-wide tree, each time into the slot nearest in terms
// of its threshold (0: the walk ended in a leaf; infinity: the root's slots are far).  Each result is one store
// to host memory, which holds kLookUnset there before.  A block of 1,024 threads and one more for the walks, or
// one and four of 256.  Bound: latency of its rounds of loads; the keys' kernel takes 13.7 us with it, 6.5
// (499,000 points) and 4.8 (600,000) without.  (On a stream of its own beside the sort, 12 us, the calls for it
// cost the host 10 us, and the stream 300 in an engine's first such call.)
struct Look {
    const float* Q = nullptr;
    int64_t n = 0;
    const float* minfo = nullptr;
    const uint32_t* slots = nullptr;
    int32_t root = -1, root_ns = 0, depth = 0;
    uint32_t* result = nullptr; // cells, then kLookWalks thresholds
    int blocks = 0;             // 0: no look
};
constexpr uint32_t kLookUnset = 0xFFFFFFFFu;
__host__ __device__ constexpr int look_blocks(int threads, bool walks) { return 1 + (walks ? 4 * kLookWalks / threads : 0); }

typedef float point3 __attribute__((ext_vector_type(3), aligned(4)));
__device__ __forceinline__ point3 look_point(const Look& look, uint32_t part)
{
    return *reinterpret_cast<const point3*>(look.Q + 3 * look_index(part, kLookBits, look.n));
}

template <int THREADS>
__device__ __forceinline__ void look_at_points(const Look& look)
{
    const int tid = threadIdx.x, lane = tid & 63;
    if (blockIdx.x == 0) {
        __shared__ uint32_t filled[(1 << kLookBits) / 32];
        __shared__ int32_t part[THREADS / 64];
        for (int k = tid; k < (1 << kLookBits) / 32; k += THREADS) filled[k] = 0u;
        __syncthreads();
        constexpr int kAhead = 4; // points in flight; 8 would take the keys' blocks to 80 registers
        for (int r = 0; r < (1 << kLookBits) / THREADS; r += kAhead) {
            point3 q[kAhead];
#pragma unroll
            for (int k = 0; k < kAhead; ++k) q[k] = look_point(look, (uint32_t)((r + k) * THREADS + tid));
#pragma unroll
            for (int k = 0; k < kAhead; ++k) {
                const uint32_t c = morton30(q[k].x, q[k].y, q[k].z, look.minfo, look.minfo + 3) >> (30 - kLookBits);
                atomicOr(&filled[c >> 5], 1u << (c & 31u));
            }
        }
        __syncthreads();
        int32_t cells = 0;
        for (int k = tid; k < (1 << kLookBits) / 32; k += THREADS) cells += __popc(filled[k]);
        for (int o = 32; o > 0; o >>= 1) cells += __shfl_xor(cells, o);
        if (lane == 0) part[tid >> 6] = cells;
        __syncthreads();
        if (tid == 0) {
            cells = 0;
            for (int k = 0; k < THREADS / 64; ++k) cells += part[k];
            __hip_atomic_store(look.result, (uint32_t)cells, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        return;
    }
    // a walk in four lanes, a slot in each
    const int walk = ((int)blockIdx.x - 1) * (THREADS / 4) + (tid >> 2), s = tid & 3;
    const point3 w = look_point(look, (uint32_t)walk * ((1u << kLookBits) / kLookWalks));
    uint32_t e = (uint32_t)look.root << 4 | (uint32_t)look.root_ns; // the same in the walk's four lanes
    bool on = look.root >= 0;
    float last = INFINITY;
    for (int level = 0; level < look.depth && __ballot(on) != 0ull; ++level) {
        float near = INFINITY, thr = 0.0f; // distance over threshold
        uint32_t link = FWN_LINK_EMPTY;
        if (on && s < (int)(e & 15u)) {
            const uint32_t* slot = look.slots + ((size_t)(e >> 4) * 4 + s) * kSlotWords;
            const float4 p = *reinterpret_cast<const float4*>(slot); // centre, threshold
            link = slot[FWN_W_LINK];
            const float dx = p.x - w.x, dy = p.y - w.y, dz = p.z - w.z;
            const float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
            if (d2 <= p.w && p.w > 0.0f) near = d2 / p.w;
            thr = p.w;
        }
        // the nearest of the four lanes' slots, the lower one of equals
        float least = INFINITY, best = 0.0f;
        e = 0u;
        auto take = [&](auto lane_of_quad) __attribute__((always_inline)) {
            constexpr int kPerm = lane_of_quad.value * 0x55; // quad_perm: that lane in all four
            const float d = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(near), kPerm, 0xF, 0xF, true));
            const uint32_t l = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)link, kPerm, 0xF, 0xF, true);
            const float t = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(thr), kPerm, 0xF, 0xF, true));
            const bool nearer = d < least;
            least = nearer ? d : least;
            e = nearer ? l : e;
            best = nearer ? t : best;
        };
        take(std::integral_constant<int, 0>{});
        take(std::integral_constant<int, 1>{});
        take(std::integral_constant<int, 2>{});
        take(std::integral_constant<int, 3>{});
        on = on && least < INFINITY;
        if (on) last = (int32_t)e < 0 ? 0.0f : best;
        on = on && (int32_t)e >= 0;
    }
    if (s == 0)
        __hip_atomic_store(look.result + 1 + walk, __float_as_uint(last), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// flags (nullptr: none): the traversal's overflow flag and work counter, cleared on the way
__global__ __launch_bounds__(QT) void k_query_keys(const float* __restrict__ Q, int64_t nQ,
                                                   const int64_t* __restrict__ q_off, int M, int mesh_bits,
                                                   const float* __restrict__ minfo, uint32_t* __restrict__ keys,
                                                   int32_t* __restrict__ flags, Look look)
{
    if ((int)blockIdx.x < look.blocks) {
        look_at_points<QT>(look);
        return;
    }
    const int64_t i = (int64_t)((int)blockIdx.x - look.blocks) * QT + threadIdx.x;
    if (i < 2 && flags) flags[i] = 0;
    if (i < nQ) keys[i] = point_key(Q, nQ, i, q_off, M, mesh_bits, sort24_first(mesh_bits), minfo);
}

// the same in tiles of kFewTile points, with the tile's counts of the sort's first digit
__global__ __launch_bounds__(1024) void k_query_keys_few(const float* __restrict__ Q, int64_t nQ,
                                                         const int64_t* __restrict__ q_off, int M, int mesh_bits,
                                                         const float* __restrict__ minfo, uint32_t* __restrict__ keys,
                                                         int32_t* __restrict__ hist, int32_t* __restrict__ flags,
                                                         Look look)
{
    if ((int)blockIdx.x < look.blocks) {
        look_at_points<1024>(look);
        return;
    }
    __shared__ int32_t cnt[1024];
    const int tile = (int)blockIdx.x - look.blocks;
    if (tile == 0 && threadIdx.x < 2) flags[threadIdx.x] = 0;
    cnt[threadIdx.x] = 0;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kFewTile / 1024; ++r) {
        const int64_t i = (int64_t)tile * kFewTile + r * 1024 + threadIdx.x;
        const bool valid = i < nQ;
        const uint32_t key = valid ? point_key(Q, nQ, i, q_off, M, mesh_bits, 0, minfo) : 0u;
        if (valid) keys[i] = key;
        count_digit(cnt, key >> 12 & 1023u, valid);
    }
    __syncthreads();
    hist[(int64_t)tile * 1024 + threadIdx.x] = cnt[threadIdx.x];
}

// One slot's 24 words held in SGPRs (a 16-dword and an 8-dword scalar load issued together at
// the top of the slot).  The other waves of the SIMD (8 resident) hide the load latency.
typedef uint32_t v16u __attribute__((ext_vector_type(16)));
typedef uint32_t v8u __attribute__((ext_vector_type(8)));
typedef v16u v16u_a4 __attribute__((aligned(4))); // slots are 96-byte records: 4-byte alignment
typedef v8u v8u_a4 __attribute__((aligned(4)));
struct SlotRegs {
    v16u a;
    v8u b;
};

__device__ __forceinline__ SlotRegs load_slot(const uint32_t* __restrict__ p)
{
    return SlotRegs{*reinterpret_cast<const v16u_a4*>(p), *reinterpret_cast<const v8u_a4*>(p + 16)};
}

__device__ __forceinline__ uint32_t su(const SlotRegs& r, int k) { return k < 16 ? r.a[k] : r.b[k - 16]; }
__device__ __forceinline__ float sw(const SlotRegs& r, int k) { return __uint_as_float(su(r, k)); }

// a triangle's record in SGPRs: two scalar loads issued together
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef v4u v4u_a4 __attribute__((aligned(4)));
__device__ __forceinline__ void load_tri(const uint32_t* __restrict__ p, float (&t)[kTriWords])
{
    const v8u a = *reinterpret_cast<const v8u_a4*>(p);
    const v4u b = *reinterpret_cast<const v4u_a4*>(p + 8);
#pragma unroll
    for (int k = 0; k < kTriWords; ++k) t[k] = __uint_as_float(k < 8 ? a[k] : b[k - 8]);
}

struct SlotWords {
    const SlotRegs& r;
    __device__ __forceinline__ float operator()(int k) const { return sw(r, k); }
};

__device__ __forceinline__ float far_field_acc(const SlotRegs& r, float dx, float dy, float dz, float d2, float om)
{
    float t, inv3;
    far_field_terms(SlotWords{r}, dx, dy, dz, d2, t, inv3);
    return fmaf(t, inv3, om);
}

// LDS of a traversal wave: the queue of FP64 near leaves (link without its leaf bit, lane), at most 63
// left over and a node's 64 per slot, and the lanes' FP64 sums in 2^-40 fixed point
__host__ __device__ __forceinline__ constexpr int queue_entries(int width) { return 64 + 64 * width; }
__host__ __device__ __forceinline__ constexpr size_t traverse_lds_bytes(int width)
{
    return sizeof(uint2) * (size_t)queue_entries(width) + sizeof(unsigned long long) * 64;
}

// One batch of up to bpts <= 64 points (one per lane) of one mesh, walked through that mesh's
// tree (bpts is 64 except in small calls, which spread their points over more waves).  FP64 near
// leaves are queued in LDS and evaluated 64 at a time, one leaf per lane whichever point it
// belongs to; a leaf's sum goes to its point's accumulator in 2^-40 fixed point (integer addition
// is associative: the total does not depend on the order) and the total is added once at the end.
template <bool STATS, int NB>
__device__ __forceinline__ void traverse_batch(
    int64_t batch, const uint32_t* __restrict__ slots, int width, const uint32_t* __restrict__ tris,
    const int32_t* __restrict__ roots, const float* __restrict__ minfo, const float* __restrict__ Q,
    const uint32_t* __restrict__ perm, const int64_t* __restrict__ q_off, const int64_t* __restrict__ b_off,
    const int32_t* __restrict__ mesh_order, int M, int bpts, float beta2, float* __restrict__ omega,
    uint8_t* __restrict__ inside, int32_t* __restrict__ stats, int32_t* __restrict__ flag, uint2* queue,
    unsigned long long* acc)
{
    const int lane = threadIdx.x & 63;
    // batches are numbered over the meshes in mesh_order; b_off is the prefix over that order
    const int pos = mesh_of64(b_off, M, batch);
    const int m = mesh_order[pos];
    const int64_t start = q_off[m] + (batch - b_off[pos]) * bpts;
    const int64_t cnt64 = q_off[m + 1] - start;
    const int cnt = cnt64 < bpts ? (int)cnt64 : bpts;
    const bool valid = lane < cnt;
    const uint32_t orig = valid ? (perm ? perm[start + lane] : (uint32_t)(start + lane)) : 0u;
    const float qx = valid ? Q[3 * (int64_t)orig] : 0.0f;
    const float qy = valid ? Q[3 * (int64_t)orig + 1] : 0.0f;
    const float qz = valid ? Q[3 * (int64_t)orig + 2] : 0.0f;
    const int32_t root = roots[2 * m];
    const int32_t root_ns = roots[2 * m + 1];
    const uint64_t tau_mask = __ballot(minfo[8 * m + 6] > 0.0f); // all lanes or none

    const uint32_t node_words = (uint32_t)width * kSlotWords;
    float om = 0.0f;
    int nq = 0;  // queued FP64 leaves
    int n64 = 0; // all that were queued
    int32_t n_test = 0, n_far = 0, n_t32 = 0, n_t64 = 0;
    if (root >= 0 && root_ns > 0) { // an inner node has a slot at least
        WaveStack<NB> S;
        S.push(0, lane, ((uint32_t)root << 4) | (uint32_t)root_ns, __ballot(valid));
        int sp = 1;
        int sp_max = 1;
        do {
            while (((sp - 1) | (63 - nq)) >= 0) { // sp > 0 and nq < 64
                --sp;
                uint32_t e;
                uint64_t mk;
                S.pop(sp, e, mk);
                const bool act = __builtin_amdgcn_inverse_ballot_w64(mk); // this lane's bit of mk, as a mask
                const uint32_t* nb = slots + (size_t)(e >> 4) * node_words;
                const int ns = (int)(e & 15u);
                // one slot: test, far term, leaf triangles or push of the child
                auto slot = [&](const SlotRegs& cur) __attribute__((always_inline)) {
                    const float dx = sw(cur, FWN_W_PX) - qx, dy = sw(cur, FWN_W_PY) - qy, dz = sw(cur, FWN_W_PZ) - qz;
                    const float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
                    const bool far = d2 > sw(cur, FWN_W_THR); // beta^2 r^2, written by the build
                    // near lanes: active and not far (scalar mask arithmetic on the compare's ballot,
                    // taken before the divergent far-field branch)
                    const uint64_t nearm = mk & ~__ballot(far);
                    if (STATS) n_test += act ? 1 : 0;
                    if (act && far) {
                        om = far_field_acc(cur, dx, dy, dz, d2, om);
                        if (STATS) ++n_far;
                    }
                    const uint32_t link = su(cur, FWN_W_LINK);
                    if (nearm == 0ull) return;
                    // written above the stack top for every slot with near lanes, kept (sp advanced)
                    // only for an internal slot: the writelanes then sit in a branch-free block and
                    // the stack registers need no copies.  The position written is below the
                    // capacity (the host keeps a one-entry margin for it), so the entries below stay
                    // intact; an overflow is checked once per node.  The link of an internal slot is
                    // the stack entry: (child << 4) | its slot count
                    S.push(sp, lane, link, nearm);
                    const bool leaf = (int32_t)link < 0; // FWN_LINK_LEAF is the sign bit
                    sp += leaf ? 0 : 1;
                    if (leaf) {
                        const int32_t first = (int32_t)((link & ~FWN_LINK_LEAF) >> 3);
                        const int32_t tcnt = (int32_t)(link & 7u) + 1;
                        // FP64 for points within tau of the leaf's bounding sphere and, for a single
                        // triangle, within tau of its plane (p lies on that plane); both thresholds are
                        // stored in the leaf's first triangle
                        float t0[kTriWords]; // the whole first triangle at once
                        load_tri(tris + (size_t)first * kTriWords, t0);
                        const float nd =
                            fmaf(dx, sw(cur, FWN_W_NX), fmaf(dy, sw(cur, FWN_W_NY), dz * sw(cur, FWN_W_NZ)));
                        uint64_t m64 = nearm & tau_mask & __ballot(d2 < t0[FWN_T_NEAR2]);
                        if (tcnt == 1) m64 &= __ballot(nd * nd < t0[FWN_T_PLANE]);
                        const uint64_t m32 = nearm & ~m64;
                        if (m32 != 0ull) {
                            const bool use32 = __builtin_amdgcn_inverse_ballot_w64(m32);
                            for (int32_t t = first;;) {
                                if (use32) {
                                    om += tri_f32(t0, qx, qy, qz);
                                    if (STATS) ++n_t32;
                                }
                                if (++t == first + tcnt) break;
                                load_tri(tris + (size_t)t * kTriWords, t0);
                            }
                        }
                        if (m64 != 0ull) {
                            if (n64 == 0) acc[lane] = 0ull;
                            if (__builtin_amdgcn_inverse_ballot_w64(m64)) {
                                const uint32_t below = __builtin_amdgcn_mbcnt_hi(
                                    (uint32_t)(m64 >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m64, 0u));
                                queue[nq + (int)below] = make_uint2(link & ~FWN_LINK_LEAF, (uint32_t)lane);
                                if (STATS) n_t64 += tcnt;
                            }
                            nq += (int)__popcll(m64);
                            n64 += (int)__popcll(m64);
                        }
                    }
                };
                const uint32_t* sl = nb;
                int s = 0;
                do {
                    slot(load_slot(sl));
                    sl += kSlotWords;
                } while (++s < ns);
                // the host only launches trees whose stack bound 1 + (width - 1) depth fits; a push
                // past the capacity is reported
                sp_max = max(sp_max, sp);
            }
            // 64 queued leaves, or what is left at the end
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            while (nq >= 64 || (sp == 0 && nq > 0)) {
                const int take = min(nq, 64);
                nq -= take;
                const uint2 it = queue[nq + (lane < take ? lane : 0)];
                // the leaf's point, from its own lane's registers
                const float x = __shfl(qx, (int)it.y), y = __shfl(qy, (int)it.y), z = __shfl(qz, (int)it.y);
                if (lane < take) {
                    const uint32_t first = it.x >> 3, n = (it.x & 7u) + 1u;
                    double s64 = 0.0;
                    for (uint32_t t = first; t < first + n; ++t)
                        s64 += tri_f64(reinterpret_cast<const float*>(tris + (size_t)t * kTriWords), x, y, z);
                    atomicAdd(&acc[it.y], (unsigned long long)__double2ll_rn(s64 * kFixScale));
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        } while (sp > 0);
        if (sp_max > WaveStack<NB>::kCap && lane == 0) atomicOr(flag, 1);
    }
    if (n64 > 0) {
        const long long v = (long long)acc[lane];
        if (v != 0) om = (float)((double)om + (double)v * (1.0 / kFixScale));
    }
    if (valid) {
        omega[orig] = om;
        if (inside) inside[orig] = ((double)om / (4.0 * 3.14159265358979323846) > 0.5) ? 1 : 0;
        if (STATS) {
            stats[4 * (int64_t)orig + 0] = n_test;
            stats[4 * (int64_t)orig + 1] = n_far;
            stats[4 * (int64_t)orig + 2] = n_t32;
            stats[4 * (int64_t)orig + 3] = n_t64;
        }
    }
}

// Grid launch: one wave per batch, XCD-aware block order.  Persistent launch: a grid sized to
// the device's resident waves; each wave takes batches from a work counter until none is left
// (the batch numbering puts the meshes with the most triangles first).
template <bool STATS, int WAVES, bool PERSIST, int NB>
__global__ __launch_bounds__(WAVES * 64) void k_traverse(
    const uint32_t* __restrict__ slots, int width, const uint32_t* __restrict__ tris,
    const int32_t* __restrict__ roots, const float* __restrict__ minfo, const float* __restrict__ Q,
    const uint32_t* __restrict__ perm, const int64_t* __restrict__ q_off, const int64_t* __restrict__ b_off,
    const int32_t* __restrict__ mesh_order, int M, int64_t n_batches, int bpts, int run, float beta2,
    float* __restrict__ omega, uint8_t* __restrict__ inside, int32_t* __restrict__ stats, int32_t* __restrict__ flag,
    uint32_t* __restrict__ work)
{
    extern __shared__ uint4 traverse_lds[];
    char* lds = reinterpret_cast<char*>(traverse_lds) + (size_t)(threadIdx.x >> 6) * traverse_lds_bytes(width);
    unsigned long long* acc = reinterpret_cast<unsigned long long*>(lds);
    uint2* queue = reinterpret_cast<uint2*>(acc + 64);
    if (!PERSIST) {
        const int64_t batch = (int64_t)xcd_batch(blockIdx.x, gridDim.x, run) * WAVES + (threadIdx.x >> 6);
        if (batch >= n_batches) return; // whole wave
        traverse_batch<STATS, NB>(batch, slots, width, tris, roots, minfo, Q, perm, q_off, b_off, mesh_order, M, bpts,
                                  beta2, omega, inside, stats, flag, queue, acc);
    } else {
        for (;;) {
            uint32_t b = 0u;
            if ((threadIdx.x & 63) == 0) b = atomicAdd(work, 1u);
            b = __builtin_amdgcn_readfirstlane(b);
            if ((int64_t)b >= n_batches) break; // every wave leaves once the counter passes the end
            traverse_batch<STATS, NB>((int64_t)b, slots, width, tris, roots, minfo, Q, perm, q_off, b_off, mesh_order, M,
                                      bpts, beta2, omega, inside, stats, flag, queue, acc);
        }
    }
}

__global__ void k_zero2(int32_t* a) // overflow flag, work counter
{
    a[0] = 0;
    a[1] = 0;
}

template <bool ST, int WV, bool PE, int NB>
void* traverse_fn()
{
    return reinterpret_cast<void*>(&k_traverse<ST, WV, PE, NB>);
}

// banks: traversal stack banks the tree needs (1: 64 entries, 3: kStack entries)
template <typename... Args>
void launch_traverse(bool stats, int waves, bool persist, int banks, int width, unsigned nblk, hipStream_t s,
                     Args... args)
{
#define FWN_TRAV(ST, WV, PE)                                                                               \
    do {                                                                                                   \
        const size_t lds = (WV) * traverse_lds_bytes(width);                                               \
        if (banks == 1)                                                                                    \
            hipLaunchKernelGGL((k_traverse<ST, WV, PE, 1>), dim3(nblk), dim3(WV * 64), lds, s, args...);   \
        else                                                                                               \
            hipLaunchKernelGGL((k_traverse<ST, WV, PE, 3>), dim3(nblk), dim3(WV * 64), lds, s, args...);   \
    } while (0)
    if (stats) {
        FWN_TRAV(true, 1, false);
        return;
    }
    switch (waves * 2 + (persist ? 1 : 0)) {
    case 2: FWN_TRAV(false, 1, false); break;
    case 3: FWN_TRAV(false, 1, true); break;
    case 4: FWN_TRAV(false, 2, false); break;
    case 5: FWN_TRAV(false, 2, true); break;
    case 8: FWN_TRAV(false, 4, false); break;
    case 9: FWN_TRAV(false, 4, true); break;
    case 16: FWN_TRAV(false, 8, false); break;
    case 17: FWN_TRAV(false, 8, true); break;
    default: fail(FWN_INVALID_ARGUMENT, "unknown traversal launch shape (waves per block 1, 2, 4 or 8)");
    }
#undef FWN_TRAV
}

// resident workgroups per CU of a traversal variant (persistent grid size)
int resident_blocks(bool persist, int waves, int banks, int width)
{
    const void* f = nullptr;
    const bool one = banks == 1;
    switch (waves * 2 + (persist ? 1 : 0)) {
    case 3: f = one ? traverse_fn<false, 1, true, 1>() : traverse_fn<false, 1, true, 3>(); break;
    case 5: f = one ? traverse_fn<false, 2, true, 1>() : traverse_fn<false, 2, true, 3>(); break;
    case 9: f = one ? traverse_fn<false, 4, true, 1>() : traverse_fn<false, 4, true, 3>(); break;
    case 17: f = one ? traverse_fn<false, 8, true, 1>() : traverse_fn<false, 8, true, 3>(); break;
    default: fail(FWN_INVALID_ARGUMENT, "unknown persistent launch shape (waves per block 1, 2, 4 or 8)");
    }
    int nb = 0;
    FWN_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, f, waves * 64, waves * traverse_lds_bytes(width)));
    return nb > 0 ? nb : 1;
}

// Multi-mesh calls (and calls with another launch shape than the default) of at most this many
// points skip the Morton sort (12 small launches that would cost more than the coherence they buy)
// and move host data through the pinned staging buffer.
constexpr int64_t kSmallBatch = 2048;

// Calls of at most this many points of one mesh run one wave per point without a sort (run_points).
// Device calls in us, this path / the sorted traversals: 1,000 points 38 / 116 (F = 20,172) and 41 /
// 140 (F = 940,800); 8,192 points 72 / 203 and 75 / 227; 16,384 points 110 / 199 and 112 / 250,
// near the surface 162 / 208 and 208 / 404; 32,768 points 189 / 207 and 193 / 303, near the surface
// 288 / 216 and 379 / 386.
constexpr int64_t kPointCalls = 16384;
//
// Where the walks outgrow the LDS records (they are then done twice, the second time depth first), only
// calls of up to kSmallBatch points take this path: a walk grows with the square of the accuracy scale and
// with the depth of the tree.  16,384 points' walks fit while scale^2 log2(F / 64) <= kPointWalk and scale
// <= kPointScale (8-wide and Morton trees outgrow them sooner).  8,192 points, uniform and near the
// surface: F = 20,172, scale 3 (75) 81 / 184 and 111 / 216, scale 4 (132) 323 / 244 and 722 / 294, scale 8
// 2222 / 586 and 3144 / 675; F = 199,692, scale 2.5 (73) 76 / 173 and 122 / 258, scale 3 (104) 228 / 216 and
// 308 / 316.  Trees of buckets, whose near leaves hold more to add, cross at half as many points: 16,384
// near the surface, buckets of 8, scale 1, F = 4,800 147 / 83, 8,192 91 / 83.
constexpr double kPointWalk = 90.0, kPointScale = 3.0;

} // namespace

char* host_stage(Engine& e, size_t bytes)
{
    if (e.h_stage_bytes < bytes) {
        if (e.h_stage) FWN_HIP(hipHostFree(e.h_stage));
        e.h_stage = nullptr;
        e.h_stage_bytes = 0;
        const size_t nb = std::max<size_t>(bytes, 1 << 16);
        FWN_HIP(hipHostMalloc(&e.h_stage, nb, hipHostMallocDefault));
        e.h_stage_bytes = nb;
    }
    return static_cast<char*>(e.h_stage);
}

namespace {

// Host calls of a single-mesh engine larger than one chunk are pipelined: chunk k's points are
// copied (several host threads) into a pinned buffer and sent to the device on one copy stream
// while chunk k-1 is answered on the engine's stream and chunk k-2's results come back on a
// second copy stream and are copied out to the caller's arrays.  Each chunk is an independent
// Morton-sorted query (a point's result does not depend on the other points of its call).  Chunks run
// k_traverse and the 24-bit sort whatever their size: the slots-in-lanes traversal, which answers 2M spread
// points of F = 874,800 in 0.65 of the time, is not chosen here.
constexpr int64_t kPipeChunk = 1 << 21; // points per chunk

void parallel_copy(void* dst, const void* src, size_t bytes)
{
    const size_t piece = (size_t)4 << 20; // at least 4 MB per thread
    const int nt = (int)std::min<size_t>(8, std::max<size_t>(1, bytes / piece));
    if (nt <= 1) {
        std::memcpy(dst, src, bytes);
        return;
    }
    const size_t part = (bytes + nt - 1) / nt;
    std::vector<std::thread> th;
    for (int t = 1; t < nt; ++t) {
        const size_t a = (size_t)t * part, b = std::min(bytes, a + part);
        if (a < b) th.emplace_back([=] { std::memcpy((char*)dst + a, (const char*)src + a, b - a); });
    }
    std::memcpy(dst, src, std::min(bytes, part));
    for (auto& x : th) x.join();
}

void run_queries_pipelined(Engine& e, const float* Q, int64_t nQ, float* omega, uint8_t* inside, int banks)
{
    hipStream_t s = e.stream;
    const int64_t C = kPipeChunk;
    const int64_t nch = (nQ + C - 1) / C;
    const size_t in_b = sizeof(float) * 3 * (size_t)C, om_b = sizeof(float) * (size_t)C, i8_b = (size_t)C;
    const size_t slot_b = in_b + om_b + i8_b;
    if (e.h_pipe_bytes < 2 * slot_b) {
        if (e.h_pipe) FWN_HIP(hipHostFree(e.h_pipe));
        e.h_pipe = nullptr;
        e.h_pipe_bytes = 0;
        FWN_HIP(hipHostMalloc(&e.h_pipe, 2 * slot_b, hipHostMallocDefault));
        e.h_pipe_bytes = 2 * slot_b;
    }
    if (!e.cs_in) FWN_HIP(hipStreamCreateWithFlags(&e.cs_in, hipStreamNonBlocking));
    if (!e.cs_out) FWN_HIP(hipStreamCreateWithFlags(&e.cs_out, hipStreamNonBlocking));
    if (!e.pev[0])
        for (auto& ev : e.pev) FWN_HIP(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
    // timing: the call spans the first upload to the last download; each chunk's traversal has
    // its own event pair (the tuner and fwn_last_timing read these)
    if (!e.ev[0])
        for (int k = 0; k < 4; ++k) FWN_HIP(hipEventCreate(&e.ev[k]));
    while ((int64_t)e.tev.size() < 2 * nch) {
        hipEvent_t ev = nullptr;
        FWN_HIP(hipEventCreate(&ev));
        e.tev.push_back(ev);
    }
    char* pin = static_cast<char*>(e.h_pipe);
    auto pin_in = [&](int sl) { return reinterpret_cast<float*>(pin + sl * slot_b); };
    auto pin_om = [&](int sl) { return reinterpret_cast<float*>(pin + sl * slot_b + in_b); };
    auto pin_i8 = [&](int sl) { return reinterpret_cast<uint8_t*>(pin + sl * slot_b + in_b + om_b); };

    e.q_in.reserve(sizeof(float) * 3 * nQ);
    e.q_om.reserve(sizeof(float) * nQ);
    if (inside) e.q_in8.reserve(nQ);
    float* dIn3 = e.q_in.as<float>();
    float* dOm = e.q_om.as<float>();
    uint8_t* dIn = inside ? e.q_in8.as<uint8_t>() : nullptr;
    for (int k = 0; k < 2; ++k) {
        e.q_keys[k].reserve(sizeof(uint32_t) * C);
        e.q_vals[k].reserve(sizeof(uint32_t) * C);
    }
    // per chunk: q_off {0, n}, b_off {0, batches}, mesh order {0} (5 int64 words)
    std::vector<int64_t> meta(5 * nch, 0);
    for (int64_t k = 0; k < nch; ++k) {
        const int64_t ck = std::min(C, nQ - k * C);
        meta[5 * k + 1] = ck;
        meta[5 * k + 3] = (ck + 63) / 64;
    }
    e.q_pmeta.reserve(sizeof(int64_t) * meta.size());
    FWN_HIP(hipMemcpyAsync(e.q_pmeta.p, meta.data(), sizeof(int64_t) * meta.size(), hipMemcpyHostToDevice, s));
    e.q_pflags.reserve(sizeof(int32_t) * 2 * nch);
    const int waves = e.opt.waves_per_block > 0 ? e.opt.waves_per_block : 1;
    const bool persist = e.opt.launch_mode == FWN_LAUNCH_PERSISTENT;
    if (persist && e.n_cu == 0) {
        hipDeviceProp_t prop;
        FWN_HIP(hipGetDeviceProperties(&prop, e.device));
        e.n_cu = prop.multiProcessorCount;
    }
    const float beta2 = e.opt.accuracy_scale * e.opt.accuracy_scale;

    for (int64_t k = 0; k <= nch; ++k) {
        if (k < nch) {
            const int sl = (int)(k & 1);
            const int64_t off = k * C, ck = std::min(C, nQ - off);
            if (k >= 2) FWN_HIP(hipEventSynchronize(e.pev[sl])); // chunk k-2's upload has read the buffer
            parallel_copy(pin_in(sl), Q + 3 * off, sizeof(float) * 3 * (size_t)ck);
            if (k == 0) FWN_HIP(hipEventRecord(e.ev[0], e.cs_in));
            FWN_HIP(hipMemcpyAsync(dIn3 + 3 * off, pin_in(sl), sizeof(float) * 3 * (size_t)ck, hipMemcpyHostToDevice,
                                   e.cs_in));
            FWN_HIP(hipEventRecord(e.pev[sl], e.cs_in));
            FWN_HIP(hipStreamWaitEvent(s, e.pev[sl], 0));
            // chunk k on the engine's stream: sort and traversal (no host wait)
            const float* dQ = dIn3 + 3 * off;
            const int64_t* d_qoff = e.q_pmeta.as<int64_t>() + 5 * k;
            const int64_t* d_boff = d_qoff + 2;
            const int32_t* d_order = reinterpret_cast<const int32_t*>(d_qoff + 4);
            uint32_t* kp = e.q_keys[0].as<uint32_t>();
            uint32_t* vp = e.q_vals[0].as<uint32_t>();
            uint32_t* kp2 = e.q_keys[1].as<uint32_t>();
            uint32_t* vp2 = e.q_vals[1].as<uint32_t>();
            hipLaunchKernelGGL(k_query_keys, dim3(grid_blocks(ck, QT)), dim3(QT), 0, s, dQ, ck, d_qoff, 1, 0,
                               e.mesh_info.as<float>(), kp, (int32_t*)nullptr, Look());
            FWN_LAUNCH_CHECK("k_query_keys");
            radix_sort_pairs32(kp, vp, kp2, vp2, ck, 8, 32, true, e.q_hist, e.q_rowsum, s);
            const int64_t nb = (ck + 63) / 64;
            int64_t nblk = (nb + waves - 1) / waves;
            if (persist) nblk = std::min<int64_t>(nblk, (int64_t)e.n_cu * resident_blocks(true, waves, banks, e.width));
            int32_t* dflag = e.q_pflags.as<int32_t>() + 2 * k;
            uint32_t* dwork = reinterpret_cast<uint32_t*>(dflag + 1);
            hipLaunchKernelGGL(k_zero2, dim3(1), dim3(1), 0, s, dflag);
            FWN_HIP(hipEventRecord(e.tev[2 * k], s));
            launch_traverse(false, waves, persist, banks, e.width, (unsigned)nblk, s, e.slots.as<uint32_t>(), e.width,
                            e.tris.as<uint32_t>(), e.roots.as<int32_t>(), e.mesh_info.as<float>(), dQ, vp, d_qoff,
                            d_boff, d_order, 1, nb, 64, 0, beta2, dOm + off, dIn ? dIn + off : nullptr,
                            (int32_t*)nullptr, dflag, dwork);
            FWN_LAUNCH_CHECK("k_traverse");
            FWN_HIP(hipEventRecord(e.tev[2 * k + 1], s));
            FWN_HIP(hipEventRecord(e.pev[2 + sl], s));
            // chunk k's results back to the pinned buffer on the other copy stream; chunk k-2's
            // results were copied out of that buffer in the previous iteration
            FWN_HIP(hipStreamWaitEvent(e.cs_out, e.pev[2 + sl], 0));
            FWN_HIP(hipMemcpyAsync(pin_om(sl), dOm + off, sizeof(float) * (size_t)ck, hipMemcpyDeviceToHost, e.cs_out));
            if (inside)
                FWN_HIP(hipMemcpyAsync(pin_i8(sl), dIn + off, (size_t)ck, hipMemcpyDeviceToHost, e.cs_out));
            FWN_HIP(hipEventRecord(e.pev[4 + sl], e.cs_out));
            if (k == nch - 1) FWN_HIP(hipEventRecord(e.ev[3], e.cs_out));
        }
        if (k >= 1) { // chunk k-1 to the caller's arrays
            const int64_t j = k - 1;
            const int sl = (int)(j & 1);
            const int64_t off = j * C, cj = std::min(C, nQ - off);
            FWN_HIP(hipEventSynchronize(e.pev[4 + sl]));
            parallel_copy(omega + off, pin_om(sl), sizeof(float) * (size_t)cj);
            if (inside) parallel_copy(inside + off, pin_i8(sl), (size_t)cj);
        }
    }
    std::vector<int32_t> fl(2 * nch);
    FWN_HIP(hipMemcpyAsync(fl.data(), e.q_pflags.p, sizeof(int32_t) * 2 * nch, hipMemcpyDeviceToHost, s));
    FWN_HIP(hipStreamSynchronize(s));
    FWN_HIP(hipStreamSynchronize(e.cs_in));
    FWN_HIP(hipStreamSynchronize(e.cs_out));
    float t_all = 0.0f;
    double t_tr = 0.0;
    FWN_HIP(hipEventElapsedTime(&t_all, e.ev[0], e.ev[3]));
    for (int64_t k = 0; k < nch; ++k) {
        float t = 0.0f;
        FWN_HIP(hipEventElapsedTime(&t, e.tev[2 * k], e.tev[2 * k + 1]));
        t_tr += t;
    }
    e.last_traverse_ms = t_tr / (double)nch; // average over the chunks' launches
    e.last_total_ms = t_all;
    for (int64_t k = 0; k < nch; ++k)
        if (fl[2 * k]) fail(FWN_LIMIT_EXCEEDED, "traversal stack overflow");
}

} // namespace

void launch_point_keys(Engine& e, const float* dQ, int64_t nQ, uint32_t* keys, hipStream_t s)
{
    hipLaunchKernelGGL(k_query_keys, dim3(grid_blocks(nQ, QT)), dim3(QT), 0, s, dQ, nQ, (const int64_t*)nullptr, 1, 0,
                       e.mesh_info.as<float>(), keys, (int32_t*)nullptr, Look());
    FWN_LAUNCH_CHECK("k_query_keys");
}

void launch_traverse_inplace(Engine& e, int banks, const float* dQ, const uint32_t* perm, const int64_t* meta,
                             int64_t nQ, float* omega, uint8_t* inside, int32_t* flag, hipStream_t s)
{
    const int64_t nb = (nQ + 63) / 64;
    if (nb > INT32_MAX) fail(FWN_LIMIT_EXCEEDED, "too many point batches");
    const float beta2 = e.opt.accuracy_scale * e.opt.accuracy_scale;
    const int64_t* q_off = meta;
    const int64_t* b_off = meta + 2;
    const int32_t* order = reinterpret_cast<const int32_t*>(meta + 4);
    launch_traverse(false, 1, false, banks, e.width, (unsigned)nb, s, e.slots.as<uint32_t>(), e.width,
                    e.tris.as<uint32_t>(), e.roots.as<int32_t>(), e.mesh_info.as<float>(), dQ, perm, q_off, b_off,
                    order, 1, nb, 64, 0, beta2, omega, inside, (int32_t*)nullptr, flag, (uint32_t*)nullptr);
    FWN_LAUNCH_CHECK("k_traverse");
}

bool few_points(const Engine& e, int64_t nQ)
{
    const double b = e.opt.accuracy_scale, F = (double)e.h_f_off[1];
    const bool fits = b <= kPointScale && b * b * std::log2(std::max(F, 1.0) / 64.0) <= kPointWalk;
    return nQ <= (!fits ? kSmallBatch : (e.opt.leaf_max > 1 ? kPointCalls / 2 : kPointCalls)) && default_shape(e);
}

void run_queries(Engine& e, const float* Q, const int64_t* q_off_host, int64_t nQ, float* omega, uint8_t* inside,
                 int32_t* stats, bool dev, const uint32_t* point_order, Points where)
{
    hipStream_t s = e.stream;
    const int M = e.n_meshes;
    std::vector<int64_t> qoff(M + 1);
    if (q_off_host) {
        for (int m = 0; m <= M; ++m) qoff[m] = q_off_host[m];
        if (qoff[0] != 0) fail(FWN_INVALID_ARGUMENT, "q_off[0] must be 0");
        for (int m = 0; m < M; ++m)
            if (qoff[m + 1] < qoff[m]) fail(FWN_INVALID_ARGUMENT, "q_off must be non-decreasing");
        nQ = qoff[M];
    } else {
        if (M != 1) fail(FWN_INVALID_ARGUMENT, "per-mesh point offsets are required for a multi-mesh engine");
        qoff[0] = 0;
        qoff[1] = nQ;
    }
    if (nQ < 0) fail(FWN_INVALID_ARGUMENT, "negative point count");
    if (nQ == 0) return;
    if (nQ > (int64_t)UINT32_MAX / 2) fail(FWN_LIMIT_EXCEEDED, "more than 2^31 points in one call");
    const int banks = stack_banks(e.width, e.max_depth);
    if (banks == 0) fail(FWN_LIMIT_EXCEEDED, "tree deeper than the traversal stack supports");
    if (!dev && !stats && M == 1 && nQ > kPipeChunk) {
        run_queries_pipelined(e, Q, nQ, omega, inside, banks);
        return;
    }
    if (!stats && M == 1 &&
        ((!dev && nQ <= kSmallBatch) || few_points(e, nQ))) {
        run_points(e, Q, nQ, omega, inside, banks, dev);
        return;
    }

    // batches of 64 points, numbered over the meshes in decreasing triangle count so that a
    // persistent launch starts the deepest trees first
    std::vector<int32_t> order(M);
    for (int m = 0; m < M; ++m) order[m] = m;
    std::stable_sort(order.begin(), order.end(), [&](int32_t a, int32_t b) {
        return e.h_f_off[a + 1] - e.h_f_off[a] > e.h_f_off[b + 1] - e.h_f_off[b];
    });
    // points per wave: 64, or fewer for small calls so that their waves spread over the device
    // (a point's result does not depend on which points share its wave)
    const bool small = nQ <= kSmallBatch && !stats;
    int most = order[0]; // the mesh with the most points, of several the one with the most triangles
    for (int m : order)
        if (qoff[m + 1] - qoff[m] > qoff[most + 1] - qoff[most]) most = m;
    const int64_t n_most = qoff[most + 1] - qoff[most];
    // points that come in an order are not looked at (the kernel that makes the keys does)
    if (point_order && where == Points::Any) where = Points::Close;
    const Quads choice = small || stats ? Quads::No : use_quads(e, nQ, n_most, banks, where);
    bool quad = choice == Quads::Yes; // Quads::Look: known once the points are looked at
    const int bpts = small ? (int)std::min<int64_t>(64, std::max<int64_t>(1, (nQ + 1023) / 1024))
                           : (quad ? quad_points(e, nQ) : 64);
    auto batches = [&](int pts) {
        std::vector<int64_t> off(M + 1, 0);
        for (int k = 0; k < M; ++k) off[k + 1] = off[k] + (qoff[order[k] + 1] - qoff[order[k]] + pts - 1) / pts;
        return off;
    };
    const std::vector<int64_t> boff = batches(bpts);
    // a call that is looked at has its batches for the slots-in-lanes traversal behind the others
    const std::vector<int64_t> boff_quad = choice == Quads::Look ? batches(kQuadPoints) : std::vector<int64_t>();
    int64_t nb = boff[M];

    const bool stage_io = small && !dev; // points in and results out through the pinned stage
    // metadata (and the points of a small host batch) in one staged copy: q_off[M+1], b_off[M+1], the other
    // b_off[M+1] of a call that is looked at (int64), mesh order[M] (int32), then the points at 16 B
    const size_t off_b = sizeof(int64_t) * (M + 1), offs = choice == Quads::Look ? 3 : 2;
    const size_t meta_b = (offs * off_b + sizeof(int32_t) * M + 15) & ~(size_t)15;
    const size_t in_b = meta_b + (stage_io ? sizeof(float) * 3 * (size_t)nQ : 0);
    const size_t out_b = stage_io ? 16 + (sizeof(float) + 1) * (size_t)nQ : 0; // flags, omega, inside
    const size_t look_at = (std::max(in_b, out_b) + 15) & ~(size_t)15; // the look's results behind it all
    char* hs = host_stage(e, look_at + sizeof(uint32_t) * (1 + kLookWalks));
    std::memcpy(hs, qoff.data(), off_b);
    std::memcpy(hs + off_b, boff.data(), off_b);
    if (choice == Quads::Look) std::memcpy(hs + 2 * off_b, boff_quad.data(), off_b);
    std::memcpy(hs + offs * off_b, order.data(), sizeof(int32_t) * M);
    if (stage_io) std::memcpy(hs + meta_b, Q, sizeof(float) * 3 * (size_t)nQ);
    const void* meta_before = e.q_meta.p;
    e.q_meta.reserve(in_b);
    // repeated calls of one shape (same meshes, point counts and batch size) find the metadata
    // already on the device and skip the upload
    const bool meta_on_device = !stage_io && e.q_meta.p == meta_before && e.meta_dev.size() == meta_b &&
                                std::memcmp(e.meta_dev.data(), hs, meta_b) == 0;
    if (!meta_on_device) {
        FWN_HIP(hipMemcpyAsync(e.q_meta.p, hs, in_b, hipMemcpyHostToDevice, s));
        e.meta_dev.assign(hs, hs + meta_b);
    }
    const int64_t* d_qoff = e.q_meta.as<int64_t>();
    const int64_t* d_boff = d_qoff + (M + 1);
    const int32_t* d_order = reinterpret_cast<const int32_t*>(d_qoff + offs * (M + 1));

    const float* dQ = Q;
    float* dOm = omega;
    uint8_t* dIn = inside;
    int32_t* dSt = stats;
    if (!dev) {
        e.q_om.reserve(sizeof(float) * nQ);
        if (stage_io) {
            dQ = reinterpret_cast<const float*>(e.q_meta.as<char>() + meta_b);
        } else {
            e.q_in.reserve(sizeof(float) * 3 * nQ);
            FWN_HIP(hipMemcpyAsync(e.q_in.p, Q, sizeof(float) * 3 * nQ, hipMemcpyHostToDevice, s));
            dQ = e.q_in.as<float>();
        }
        dOm = e.q_om.as<float>();
        if (inside) {
            e.q_in8.reserve(nQ);
            dIn = e.q_in8.as<uint8_t>();
        }
        if (stats) {
            e.q_stats.reserve(sizeof(int32_t) * 4 * nQ);
            dSt = e.q_stats.as<int32_t>();
        }
    }
    e.q_flag.reserve(3 * sizeof(int32_t));

    if (!small && !point_order) {
        for (int k = 0; k < 2; ++k) {
            e.q_keys[k].reserve(sizeof(uint32_t) * nQ);
            e.q_vals[k].reserve(sizeof(uint32_t) * nQ);
        }
    }
    if (!e.ev[0])
        for (int k = 0; k < 4; ++k) FWN_HIP(hipEventCreate(&e.ev[k]));

    FWN_HIP(hipEventRecord(e.ev[0], s));
    int32_t* dflag = e.q_flag.as<int32_t>();
    uint32_t* dwork = reinterpret_cast<uint32_t*>(dflag + 1);
    Look look;
    volatile uint32_t* seen = reinterpret_cast<volatile uint32_t*>(hs + look_at);
    if (choice == Quads::Look) {
        std::memset(hs + look_at, 0xFF, sizeof(uint32_t) * (1 + kLookWalks));
        look.Q = dQ + 3 * qoff[most];
        look.n = n_most;
        look.minfo = e.mesh_info.as<float>() + 8 * most;
        look.slots = e.slots.as<uint32_t>();
        look.root = e.h_roots[2 * most];
        look.root_ns = e.h_roots[2 * most + 1];
        look.depth = quads_near_surface(e, nQ) ? std::max(e.max_depth, 1) : 0;
        look.result = reinterpret_cast<uint32_t*>(hs + look_at);
    }
    // sorted position -> input index (nullptr: small calls keep the input order)
    const uint32_t* vp = small ? nullptr : point_order;
    if (small || point_order) {
        hipLaunchKernelGGL(k_zero2, dim3(1), dim3(1), 0, s, dflag);
    } else {
        uint32_t* kp = e.q_keys[0].as<uint32_t>();
        uint32_t* kp2 = e.q_keys[1].as<uint32_t>();
        uint32_t* vals = e.q_vals[0].as<uint32_t>();
        uint32_t* vp2 = e.q_vals[1].as<uint32_t>();
        int mesh_bits = 0;
        while ((1 << mesh_bits) < M) ++mesh_bits;
        if (mesh_bits > 24) fail(FWN_LIMIT_EXCEEDED, "more than 2^24 meshes in one engine");
        // few tiles: 20 bits (the mesh among them) separate 2^20 cells of a mesh's box, or about 60,000 along
        // a surface, where at most 524,288 points leave little for more bits to order
        if (few_tiles(nQ) <= kFewTiles && mesh_bits <= 8) {
            e.q_hist.reserve(sizeof(int32_t) * 1024 * (size_t)few_tiles(nQ));
            if (choice == Quads::Look) look.blocks = look_blocks(1024, look.depth > 0);
            hipLaunchKernelGGL(k_query_keys_few, dim3(few_tiles(nQ) + look.blocks), dim3(1024), 0, s, dQ, nQ, d_qoff, M,
                               mesh_bits, e.mesh_info.as<float>(), kp, e.q_hist.as<int32_t>(), dflag, look);
            FWN_LAUNCH_CHECK("k_query_keys_few");
            sort_few_tiles(kp, kp2, vp2, vals, nQ, e.q_hist.as<int32_t>(), s);
        } else {
            if (choice == Quads::Look) look.blocks = look_blocks(QT, look.depth > 0);
            hipLaunchKernelGGL(k_query_keys, dim3(grid_blocks(nQ, QT) + look.blocks), dim3(QT), 0, s, dQ, nQ, d_qoff, M,
                               mesh_bits, e.mesh_info.as<float>(), kp, dflag, look);
            FWN_LAUNCH_CHECK("k_query_keys");
            radix_sort_pairs32(kp, vals, kp2, vp2, nQ, 8, 32, true, e.q_hist, e.q_rowsum, s);
        }
        vp = vals;
    }
    int quad_bpts = bpts;
    if (choice == Quads::Look) { // its results come while the points are sorted; a failed launch ends the wait
        const int words = 1 + (look.depth > 0 ? kLookWalks : 0);
        int k = 0;
        bool over = false;
        for (uint32_t spin = 1;; ++spin) {
            while (k < words && seen[k] != kLookUnset) ++k;
            if (k == words) break;
            if (over) fail(FWN_HIP_ERROR, "no result of the look at the points");
            if ((spin & 255u) == 0u && hipStreamQuery(s) != hipErrorNotReady) {
                FWN_HIP(hipStreamSynchronize(s));
                over = true;
            }
        }
        std::atomic_thread_fence(std::memory_order_acquire);
        float last[kLookWalks];
        for (int j = 0; j + 1 < words; ++j) {
            const uint32_t u = seen[1 + j];
            std::memcpy(last + j, &u, sizeof(u));
        }
        quad = quads_after_look(e, most, n_most, (int)seen[0], last, words - 1);
        if (quad) {
            nb = boff_quad[M];
            d_boff += M + 1;
            quad_bpts = kQuadPoints;
        }
    }

    const int waves = e.opt.waves_per_block > 0 && !stats ? e.opt.waves_per_block : 1; // stats: one wave a block
    const bool persist = (e.opt.launch_mode == FWN_LAUNCH_PERSISTENT) && !stats;
    int64_t nblk = (nb + waves - 1) / waves;
    if (persist) {
        if (e.n_cu == 0) {
            hipDeviceProp_t prop;
            FWN_HIP(hipGetDeviceProperties(&prop, e.device));
            e.n_cu = prop.multiProcessorCount;
        }
        nblk = std::min<int64_t>(nblk, (int64_t)e.n_cu * resident_blocks(true, waves, banks, e.width));
    }
    if (nblk > INT32_MAX) fail(FWN_LIMIT_EXCEEDED, "too many point batches");
    const float beta2 = e.opt.accuracy_scale * e.opt.accuracy_scale;
    FWN_HIP(hipEventRecord(e.ev[1], s));
    if (quad) {
        launch_quads(e, dQ, vp, d_qoff, d_boff, d_order, M, nb, quad_bpts, where, dOm, dIn, dflag, s);
    } else {
        launch_traverse(stats != nullptr, waves, persist, banks, e.width, (unsigned)nblk, s, e.slots.as<uint32_t>(),
                        e.width, e.tris.as<uint32_t>(), e.roots.as<int32_t>(), e.mesh_info.as<float>(), dQ, vp, d_qoff,
                        d_boff, d_order, M, nb, bpts, e.uneven ? 16 : 0, beta2, dOm, dIn, dSt, dflag, dwork);
        FWN_LAUNCH_CHECK("k_traverse");
    }
    FWN_HIP(hipEventRecord(e.ev[2], s));
    // the flag (and a small host call's results in the same wait) through the pinned stage, whose
    // metadata bytes were uploaded before, in order
    int32_t h_fl = 0;
    FWN_HIP(hipMemcpyAsync(hs, dflag, sizeof(h_fl), hipMemcpyDeviceToHost, s));
    if (stage_io) {
        FWN_HIP(hipMemcpyAsync(hs + 16, dOm, sizeof(float) * nQ, hipMemcpyDeviceToHost, s));
        if (inside) FWN_HIP(hipMemcpyAsync(hs + 16 + sizeof(float) * nQ, dIn, nQ, hipMemcpyDeviceToHost, s));
    }
    FWN_HIP(hipStreamSynchronize(s));
    std::memcpy(&h_fl, hs, sizeof(h_fl));
    if (h_fl) fail(FWN_LIMIT_EXCEEDED, "traversal stack overflow");
    if (stage_io) {
        std::memcpy(omega, hs + 16, sizeof(float) * nQ);
        if (inside) std::memcpy(inside, hs + 16 + sizeof(float) * nQ, nQ);
    } else if (!dev) {
        FWN_HIP(hipMemcpyAsync(omega, dOm, sizeof(float) * nQ, hipMemcpyDeviceToHost, s));
        if (inside) FWN_HIP(hipMemcpyAsync(inside, dIn, nQ, hipMemcpyDeviceToHost, s));
        if (stats) FWN_HIP(hipMemcpyAsync(stats, dSt, sizeof(int32_t) * 4 * nQ, hipMemcpyDeviceToHost, s));
        FWN_HIP(hipStreamSynchronize(s));
    }
    float t_tr = 0.0f, t_all = 0.0f;
    FWN_HIP(hipEventElapsedTime(&t_tr, e.ev[1], e.ev[2]));
    FWN_HIP(hipEventElapsedTime(&t_all, e.ev[0], e.ev[2]));
    e.last_traverse_ms = t_tr;
    e.last_total_ms = t_all;
}

const uint32_t* sort_points_single(Engine& e, const float* dQ, int64_t nQ)
{
    if (e.n_meshes != 1) fail(FWN_INVALID_ARGUMENT, "a single-mesh engine is required");
    if (nQ > (int64_t)UINT32_MAX / 2) fail(FWN_LIMIT_EXCEEDED, "more than 2^31 points in one call");
    hipStream_t s = e.stream;
    for (int k = 0; k < 2; ++k) {
        e.q_keys[k].reserve(sizeof(uint32_t) * nQ);
        e.q_vals[k].reserve(sizeof(uint32_t) * nQ);
    }
    uint32_t* kp = e.q_keys[0].as<uint32_t>();
    uint32_t* vp = e.q_vals[0].as<uint32_t>();
    uint32_t* kp2 = e.q_keys[1].as<uint32_t>();
    uint32_t* vp2 = e.q_vals[1].as<uint32_t>();
    hipLaunchKernelGGL(k_query_keys, dim3(grid_blocks(nQ, QT)), dim3(QT), 0, s, dQ, nQ, (const int64_t*)nullptr, 1, 0,
                       e.mesh_info.as<float>(), kp, (int32_t*)nullptr, Look());
    FWN_LAUNCH_CHECK("k_query_keys");
    radix_sort_pairs32(kp, vp, kp2, vp2, nQ, 8, 32, true, e.q_hist, e.q_rowsum, s);
    return vp;
}

} // namespace fwn
