// Winding number queries with a node's slots in the lanes of a wave (gfx950): the batched
// traversal of calls whose points are far apart compared with the mesh's triangles.  Compiled
// without machine LICM: it would keep the FP64 constants of the near-field evaluation in 40 vector
// registers through the whole walk (118 registers, 4 waves per SIMD, instead of 64 and the 6 and a
// half that the LDS allows).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "fwn_eval.h"
#include "fwn_internal.h"
#include "fwn_order.h"

namespace fwn {

namespace {

// Slots-in-lanes traversal of 4-wide trees: 16 points per wave, lane 4 p + s holding point p and
// taking slot s of every node the wave visits, so that a node's four slots are tested, expanded
// and (leaves) evaluated in one parallel step.  k_traverse walks 64 points per wave and takes the
// slots one after the other from scalar registers, which costs less when all 64 lanes have work
// in the slot; here a wave's points are 4 times closer together, a visit has a quarter of the
// dependent steps and a call has 4 times the waves.
//
// A node is fetched into the LDS buffer of its stack position when it is pushed
// (global_load_lds), so the wave waits for one fetch on the child popped next and its siblings
// are there when their turn comes.  The terms of a node reach the point's sum in slot order, as
// in k_traverse: every lane's pair (a, b), far terms as (t, inv3), near FP32 triangles as
// (1, value), other slots as (0, 0), goes through om = fmaf(a, b, om) by quad broadcasts (the
// four lanes of a point hold the same sum).  FP64 near leaves are queued in LDS and evaluated 64
// at a time, one leaf per lane, their sums added in 2^-40 fixed point (associative) to the
// point's LDS accumulator.  Results are bit for bit those of k_traverse.
//
// Bound: VALU issue (400k points near the surface, F = 190k: 9,700 VALU and 6,100 SALU instructions per
// wave over 100 node visits, three quarters of the issue slots) once a call has enough waves, the chain
// of node visits below that.  Leaf triangles are loaded before the far terms they arrive behind, FP64
// leaves flushed outside the node loop and their lanes not evaluated in FP32 too: 400k points, F =
// 199,692, 254 -> 221 us uniform and 564 -> 497 near the surface.  Kernels alone, k_traverse then this
// one: 20,000 uniform points, F = 20,172 353 and 97 us; 100k points, F = 199,692 667 and 146 us uniform,
// 754 and 216 near the surface.
constexpr int kQuadQueue = 128; // FP64 leaves waiting (at most 63 before a node adds 64)
constexpr int kQuadNodeBytes = 4 * kSlotWords * 4; // one 4-wide node

template <int S>
__device__ __forceinline__ float quad_bcast(float v) // lane 4 p + S of each quad
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), S * 0x55, 0xF, 0xF, true));
}
// om = fmaf(a_s, b_s, om) for the quad's lanes s = 0..3 in order: the multiplicand of each v_fmac
// is read through DPP (two instructions a term; the compiler's form takes three)
__device__ __forceinline__ float quad_terms(float a, float b, float om)
{
    float t;
    asm("s_nop 1\n\t" // a DPP operand is read two wait states after its write at the earliest
        "v_mov_b32_dpp %1, %3 quad_perm:[0,0,0,0] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %2, %1 quad_perm:[0,0,0,0] row_mask:0xf bank_mask:0xf\n\t"
        "v_mov_b32_dpp %1, %3 quad_perm:[1,1,1,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %2, %1 quad_perm:[1,1,1,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_mov_b32_dpp %1, %3 quad_perm:[2,2,2,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %2, %1 quad_perm:[2,2,2,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_mov_b32_dpp %1, %3 quad_perm:[3,3,3,3] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %2, %1 quad_perm:[3,3,3,3] row_mask:0xf bank_mask:0xf"
        : "+v"(om), "=&v"(t)
        : "v"(a), "v"(b));
    return om;
}
// 64-bit lane masks whose quads are points: s_quadmask_b64 (bit p: any lane of quad p) and its
// inverse (all four lanes of each point) by two s_bitreplicate_b64_b32; LLVM intrinsics that
// clang exposes under no builtin name
extern "C" __device__ uint64_t fwn_llvm_quadmask(uint64_t m) __asm("llvm.amdgcn.s.quadmask.i64");
extern "C" __device__ uint64_t fwn_llvm_bitreplicate(uint32_t m) __asm("llvm.amdgcn.s.bitreplicate");
__device__ __forceinline__ uint32_t quad_mask(uint64_t m) { return (uint32_t)fwn_llvm_quadmask(m); }
__device__ __forceinline__ uint64_t quad_expand(uint32_t m16)
{
    return fwn_llvm_bitreplicate((uint32_t)fwn_llvm_bitreplicate(m16));
}

// LDS: node buffers (lds_nodes of them), the FP64 queue, per point its accumulator and position
inline size_t quad_lds_bytes(int lds_nodes)
{
    return (size_t)lds_nodes * kQuadNodeBytes + kQuadQueue * sizeof(uint2) +
           kQuadPoints * (sizeof(unsigned long long) + 4 * sizeof(float));
}

// BUCKET: leaves hold up to 8 triangles (1 otherwise)
template <bool BUCKET>
__global__ __launch_bounds__(64) void k_traverse_quad(
    const uint32_t* __restrict__ slots, const uint32_t* __restrict__ tris, const int32_t* __restrict__ roots,
    const float* __restrict__ minfo, const float* __restrict__ Q, const uint32_t* __restrict__ perm,
    const int64_t* __restrict__ q_off, const int64_t* __restrict__ b_off, const int32_t* __restrict__ mesh_order,
    int M, int64_t n_batches, int bpts, int run, int lds_nodes, float* __restrict__ omega,
    uint8_t* __restrict__ inside, int32_t* __restrict__ flag)
{
    extern __shared__ uint4 quad_lds[];
    uint2* queue = reinterpret_cast<uint2*>(reinterpret_cast<char*>(quad_lds) + (size_t)lds_nodes * kQuadNodeBytes);
    unsigned long long* acc = reinterpret_cast<unsigned long long*>(queue + kQuadQueue);
    float4* qpos = reinterpret_cast<float4*>(acc + kQuadPoints);
    constexpr int kNode4 = kQuadNodeBytes / 16; // uint4 per node
    const int lane = threadIdx.x;
    const int p = lane >> 2, s = lane & 3;
    const int64_t batch =
        run > 0 ? xcd_remap_runs(blockIdx.x, gridDim.x, (uint32_t)run) : xcd_remap(blockIdx.x, gridDim.x);
    if (batch >= n_batches) return;
    const int pos = mesh_of64(b_off, M, batch);
    const int m = mesh_order[pos];
    const int64_t start = q_off[m] + (batch - b_off[pos]) * bpts;
    const int64_t cnt64 = q_off[m + 1] - start;
    const int cnt = cnt64 < bpts ? (int)cnt64 : bpts;
    const bool valid = p < cnt;
    const uint32_t jpos = (uint32_t)(start + p);
    const uint32_t orig = valid ? (perm ? perm[jpos] : jpos) : 0u;
    const float qx = valid ? Q[3 * (int64_t)orig] : 0.0f;
    const float qy = valid ? Q[3 * (int64_t)orig + 1] : 0.0f;
    const float qz = valid ? Q[3 * (int64_t)orig + 2] : 0.0f;
    const int32_t root = roots[2 * m];
    const int32_t root_ns = roots[2 * m + 1];
    const uint64_t tau_mask = __ballot(minfo[8 * m + 6] > 0.0f); // all lanes or none
    if (s == 0) {
        acc[p] = 0ull;
        qpos[p] = make_float4(qx, qy, qz, 0.0f);
    }

    float om = 0.0f;
    int nq = 0; // queued FP64 leaves
    if (root >= 0) {
        // stack: entry k in lane k, a node's link and the 16-bit mask of the points that visit it
        uint32_t st_link = ((uint32_t)root << 4) | (uint32_t)root_ns, st_mask = quad_mask(__ballot(valid));
        auto fetch = [&](uint32_t lk, int at) __attribute__((always_inline)) {
            const uint32_t* nb = slots + (size_t)(lk >> 4) * (size_t)(4 * kSlotWords);
            asm("" : "+s"(nb)); // the node's address stays scalar
            fetch_node(nb, quad_lds + at * kNode4, 4, lane);
        };
        fetch(st_link, 0);
        int sp = 1, sp_max = 1;
        do {
            while (((sp - 1) | (63 - nq)) >= 0) { // sp > 0 and nq < 64
                --sp;
                const uint32_t e = (uint32_t)__builtin_amdgcn_readlane((int)st_link, sp);
                const uint32_t m16 = (uint32_t)__builtin_amdgcn_readlane((int)st_mask, sp);
                uint4 x[kSlotWords / 4];
                if (sp < lds_nodes) {
                    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // this node's fetch has landed
                    const uint4* src = quad_lds + sp * kNode4 + s * (kSlotWords / 4);
#pragma unroll
                    for (int k = 0; k < kSlotWords / 4; ++k) x[k] = src[k];
                } else { // a stack position without a buffer
                    const char* nb = reinterpret_cast<const char*>(slots + (size_t)(e >> 4) * (size_t)(4 * kSlotWords));
                    const uint4* src = reinterpret_cast<const uint4*>(nb + (uint32_t)s * (kSlotWords * 4));
#pragma unroll
                    for (int k = 0; k < kSlotWords / 4; ++k) x[k] = src[k];
                }
                // the lanes with a point to test: the points of the mask, the node's occupied slots
                const uint64_t mk = quad_expand(m16) & __ballot(s < (int)(e & 15u));
                float w[FWN_W_LINK];
#pragma unroll
                for (int k = 0; k < FWN_W_LINK; ++k) w[k] = __uint_as_float(reinterpret_cast<const uint32_t*>(x)[k]);
                const uint32_t link = x[5].w;
                const float dx = w[FWN_W_PX] - qx, dy = w[FWN_W_PY] - qy, dz = w[FWN_W_PZ] - qz;
                const float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
                const uint64_t farb = __ballot(d2 > w[FWN_W_THR]);
                const uint64_t nearm = mk & ~farb;
                const uint64_t leafm = nearm & __ballot((int32_t)link < 0);
                // children, in slot order, each fetched as it is pushed: the node's words are in
                // registers before a fetch overwrites its buffer
                const uint64_t inner = nearm & ~leafm;
                if (inner != 0ull) {
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const uint64_t mc = inner & (0x1111111111111111ull << c);
                        if (mc != 0ull) {
                            const uint32_t lc = (uint32_t)__builtin_amdgcn_readlane((int)link, c);
                            st_link = wave_writelane(lc, sp & 63, st_link);
                            st_mask = wave_writelane(quad_mask(mc), sp & 63, st_mask);
                            if (sp < lds_nodes) fetch(lc, sp);
                            ++sp;
                        }
                    }
                    sp_max = max(sp_max, sp);
                }
                // the leaves' triangles are on their way while the far terms are evaluated
                const int32_t first = (int32_t)((link & ~FWN_LINK_LEAF) >> 3);
                const int32_t tcnt = BUCKET ? (int32_t)(link & 7u) + 1 : 1;
                uint4 y[kTriWords / 4];
                if (leafm != 0ull) { // lanes without a leaf: the first triangle, in one line for all of them
                    const uint32_t at = __builtin_amdgcn_inverse_ballot_w64(leafm) ? (uint32_t)first : 0u;
                    const uint4* tp = reinterpret_cast<const uint4*>(tris + (size_t)at * kTriWords);
#pragma unroll
                    for (int k = 0; k < kTriWords / 4; ++k) y[k] = tp[k];
                }
                float a = 0.0f, b = 0.0f;
                if (__builtin_amdgcn_inverse_ballot_w64(mk & farb))
                    far_field_terms(LaneWords{w}, dx, dy, dz, d2, a, b);
                if (leafm != 0ull) {
                    float tw[kTriWords];
#pragma unroll
                    for (int k = 0; k < kTriWords / 4; ++k) {
                        tw[4 * k] = __uint_as_float(y[k].x);
                        tw[4 * k + 1] = __uint_as_float(y[k].y);
                        tw[4 * k + 2] = __uint_as_float(y[k].z);
                        tw[4 * k + 3] = __uint_as_float(y[k].w);
                    }
                    const float nd = fmaf(dx, w[FWN_W_NX], fmaf(dy, w[FWN_W_NY], dz * w[FWN_W_NZ]));
                    uint64_t plane = __ballot(nd * nd < tw[FWN_T_PLANE]);
                    if (BUCKET) plane |= __ballot(tcnt > 1);
                    const uint64_t m64 = leafm & tau_mask & plane & __ballot(d2 < tw[FWN_T_NEAR2]);
                    const bool use64 = __builtin_amdgcn_inverse_ballot_w64(m64);
                    const bool use32 = __builtin_amdgcn_inverse_ballot_w64(leafm & ~m64);
                    if (use32) {
                        a = 1.0f;
                        b = tri_f32(tw, qx, qy, qz);
                    }
                    if (m64 != 0ull) {
                        if (use64) {
                            const uint32_t below = __builtin_amdgcn_mbcnt_hi(
                                (uint32_t)(m64 >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m64, 0u));
                            queue[nq + (int)below] = make_uint2(link & ~FWN_LINK_LEAF, (uint32_t)p);
                        }
                        nq += (int)__popcll(m64);
                    }
                    if (BUCKET) {
                        const int n32 = use32 ? tcnt : 0;
                        const uint64_t more = __ballot(n32 > 1);
                        if (more != 0ull) {
                            // the buckets' other triangles, then every slot's terms in order
                            float v[8];
#pragma unroll
                            for (int k = 1; k < 8; ++k) {
                                v[k] = 0.0f;
                                const uint32_t* tk = tris + (size_t)(first + k) * kTriWords;
                                if (k < n32) v[k] = tri_f32(reinterpret_cast<const float*>(tk), qx, qy, qz);
                            }
                            auto slot_terms = [&](auto c) __attribute__((always_inline)) {
                                om = fmaf(quad_bcast<c.value>(a), quad_bcast<c.value>(b), om);
                                if ((more & (0x1111111111111111ull << c.value)) != 0ull) {
#pragma unroll
                                    for (int k = 1; k < 8; ++k) om += quad_bcast<c.value>(v[k]);
                                }
                            };
                            slot_terms(std::integral_constant<int, 0>{});
                            slot_terms(std::integral_constant<int, 1>{});
                            slot_terms(std::integral_constant<int, 2>{});
                            slot_terms(std::integral_constant<int, 3>{});
                            continue;
                        }
                    }
                }
                om = quad_terms(a, b, om);
            }
            // 64 queued leaves, or what is left at the end
            __syncthreads();
            while (nq >= 64 || (sp == 0 && nq > 0)) {
                const int take = min(nq, 64);
                nq -= take;
                if (lane < take) {
                    const uint2 it = queue[nq + lane];
                    const float4 q = qpos[it.y];
                    const uint32_t first = it.x >> 3, n = BUCKET ? (it.x & 7u) + 1u : 1u;
                    double s64 = 0.0;
                    for (uint32_t t = first; t < first + n; ++t)
                        s64 += tri_f64(reinterpret_cast<const float*>(tris + (size_t)t * kTriWords), q.x, q.y, q.z);
                    atomicAdd(&acc[it.y], (unsigned long long)__double2ll_rn(s64 * kFixScale));
                }
            }
            __syncthreads();
        } while (sp > 0);
        if (sp_max > 64 && lane == 0) atomicOr(flag, 1); // never with the host's stack bound
    }
    if (valid && s == 0) {
        const long long v = (long long)acc[p];
        if (v != 0) om = (float)((double)om + (double)v * (1.0 / kFixScale));
        omega[orig] = om;
        if (inside) inside[orig] = ((double)om / (4.0 * 3.14159265358979323846) > 0.5) ? 1 : 0;
    }
}

} // namespace

// Whether a call of nQ points, q_off per mesh, goes to the slots-in-lanes traversal: 4-wide trees
// of the default launch shape (the other shapes are k_traverse's, chosen by the tuner or the
// caller), up to kQuadCross * cbrt(F) points for a mesh of F triangles (several: of the mean F)
// and, for several meshes, kQuadSparse points a triangle more, as each mesh's share of the points
// is sparse on it however many the call has.  The two kernels' costs cross where the 64 points of a
// k_traverse wave are close together compared with the nodes they visit, for points near the surface
// (both kernels walk to the triangles) at fewer points than for uniform ones; the line lies between the
// two crossings.  k_traverse / this kernel in us, with the
// sort,
//   uniform: F = 972 138 / 120 (200k points) and 170 / 182 (400k); F = 20,172 349 / 336 (800k), 455 /
//     516 (1.5M); F = 199,692 731 / 567 (1.5M), 858 / 814 (2.5M), 1038 / 1215 (4M); F = 940,800
//     1278 / 883 (2.5M), 1456 / 1269 (4M);
//   near the surface: F = 972 150 / 143 (200k), 187 / 225 (400k); F = 20,172 348 / 350 (400k), 495 /
//     567 (800k); F = 199,692 861 / 844 (800k), 1119 / 1355 (1.5M); F = 940,800 1380 / 1287 (800k), 1800 /
//     2021 (1.5M);
//   several meshes, uniform / near the surface (the kernels alone): 64 x 20k points, F = 199,692
//     1800 / 808 and 5516 / 2818, F = 19,200 1058 / 669 and 1589 / 1241, F = 1,728 535 / 528 and 608 /
//     713; 32 x 100k points, F = 19,200 1322 / 1169 and 1920 / 2164; 8 meshes of 14k to 48k, 1M
//     points, 703 / 409; 32 of 1.7k to 181k, 3.7M points, 1199 / 1214.
//
// Points in a layer at a distance from the surface, where few walks go deep, are close together at far fewer
// points than these lines say.  k_traverse / this kernel for layers 5 % of the diagonal off: F = 199,692 170 /
// 185 us (400k points), 208 / 244 (600k) and 249 / 327 (1M); 16 such meshes 379 / 485 (100k points each) and 762 /
// 1178 (300k); 64 of 20,172 triangles 477 / 557 (25k each).  Above kQuadAny points the slots-in-lanes traversal
// is therefore taken only for points that, looked at (look_at_points), spread over the box of the mesh with the
// most of them, or are close to its surface for their density.  One mesh's points near the surface: up to
// kQuadNear * log2(F / 170) of them, as the kernels cross early there (F = 20,172 454 / 435 at 499k points and 484
// / 495 at 600k; 199,692 834 / 727 at 600k and 979 / 1026 at 1M; 874,800 1502 / 1483 at 1M).  Several meshes': up to
// the line above (64 of 199,692 triangles, 12k points each near the surface 4780 / 2207, 1 % off 1647 / 836; 16
// with 300k 5235 / 4904).  The look costs 7 to 9 us.  (As a kernel of its own ahead of the sort, with a fixed
// stride and a copy back, it cost 25 to 35, did not see several meshes, and took grids of 128^3 points for layers:
// F = 750,000 1226 us, 785 now.)
//
// A caller that knows its points to lie along a surface (the orientation probes) has a line of its own,
// kQuadLayer * cbrt(F), and no look at the points: whole calls of two probes a facet, 0.01 / 1 / 5 / 30 % of
// the size off the surface, k_traverse 1060 / 818 / 394 / 231 us and this kernel 641 / 604 / 346 / 229 at 479k
// probes, 1250 / 887 / 398 / 239 and 752 / 711 / 386 / 258 at 569k, 1707 / 1108 / 449 / 271 and 1135 / 981 /
// 507 / - at 912k: the line lies where no distance loses.
constexpr double kQuadCross = 24000.0, kQuadSparse = 2.0, kQuadAny = 450000.0, kQuadNear = 73000.0, kQuadLayer = 8000.0;
constexpr int64_t kLookLeast = 1 << kLookBits;
Quads use_quads(const Engine& e, int64_t nQ, int64_t most, int banks, Points where)
{
    if (e.width != 4 || banks != 1 || !default_shape(e)) return Quads::No;
    const double F = (double)e.h_f_off[e.n_meshes];
    if (where == Points::Layer && e.n_meshes == 1)
        return (double)nQ <= kQuadLayer * std::cbrt(F) ? Quads::Yes : Quads::No;
    if ((double)nQ > kQuadCross * std::cbrt(F / e.n_meshes) + (e.n_meshes > 1 ? kQuadSparse * F : 0.0)) return Quads::No;
    if ((double)nQ <= kQuadAny || most < kLookLeast || where == Points::Spread) return Quads::Yes;
    return where == Points::Close ? Quads::No : Quads::Look;
}

bool quads_near_surface(const Engine& e, int64_t nQ)
{
    return e.n_meshes > 1 || (double)nQ <= kQuadNear * std::log2((double)e.h_f_off[1] / 170.0);
}

// Close to the surface for their density: the last slot's threshold of half of the walks is below kLookNear
// times the extent^2 of 64 neighbours, 64 times the layer's area over n, with about a cell's mean face of area
// for each filled cell.
bool quads_after_look(const Engine& e, int mesh, int64_t n, int cells, const float* last, int walks)
{
    if ((double)cells >= kSpreadLeast * (double)(1 << kLookBits)) return true;
    const float* inv = &e.h_info[8 * (size_t)mesh + 3];
    double side[3]; // of a cell: 32 x 16 x 16 of them
    for (int d = 0; d < 3; ++d) side[d] = inv[d] > 0.0f ? (d == 0 ? 1.0 / 32 : 1.0 / 16) / inv[d] : 0.0;
    const double face = (side[0] * side[1] + side[1] * side[2] + side[2] * side[0]) / 3.0;
    const double line = kLookNear * 64.0 * cells * face / (double)n;
    return walks > 0 && 2 * std::count_if(last, last + walks, [&](float t) { return t <= line; }) >= walks;
}

// Points per wave: 16, the wave's lanes, or 8 where so few waves run that the longest decides (up to 500
// cbrt(F) points of one mesh, at most 32,000).  8 / 16 in us: 20k points, F = 199,692 97 / 115 uniform,
// 142 / 184 near the surface, F = 940,800 106 / 128 and 197 / 278; 30k points 103 / 127 and 159 / 178,
// 109 / 135 and 202 / 270; against it 50k points near the surface, 199 / 172 and 314 / 279, and F = 20,172,
// 30k points near the surface 94 / 86.
int quad_points(const Engine& e, int64_t nQ)
{
    return e.n_meshes == 1 && (double)nQ <= std::min(500.0 * std::cbrt((double)e.h_f_off[1]), 32000.0) ? 8 : kQuadPoints;
}

void launch_quads(Engine& e, const float* dQ, const uint32_t* perm, const int64_t* q_off, const int64_t* b_off,
                  const int32_t* order, int M, int64_t nb, int bpts, Points where, float* omega, uint8_t* inside,
                  int32_t* flag, hipStream_t s)
{
    // Blocks to the XCDs in runs for several meshes (xcd_batch) and for layers of 8,192 waves or more, whose
    // expensive waves lie together: probes 1 % off, one run per XCD / runs of 64, 400k points 488 / 454 us (F =
    // 199,692) and 530 / 473 (F = 940,800), 500k 565 / 527 and 625 / 543; uniform points lose 8 to 18 % to runs
    const int run = M > 1 ? 16 : (where == Points::Layer && nb >= 8192 ? 64 : 0);
    // node buffers per wave: 20 (9 KB, room for 4 waves per SIMD) while the call has no more waves
    // than that, else 12 (6 KB: 6 and a half); entries above them are rare.  F = 199,692, uniform and
    // near the surface, 9 / 12 / 20 buffers: 20k points 135 / 132 / 118 and 215 / 200 / 178 us, 400k
    // points 224 / 221 / 246 and 573 / 497 / 565 us
    const int lds_nodes = std::min(nb <= 4096 ? 20 : 12, 1 + 3 * std::max(e.max_depth, 1));
    const size_t lds = quad_lds_bytes(lds_nodes);
#define FWN_QUAD(BUCKET)                                                                                            \
    hipLaunchKernelGGL(k_traverse_quad<BUCKET>, dim3((unsigned)nb), dim3(64), lds, s, e.slots.as<uint32_t>(),      \
                       e.tris.as<uint32_t>(), e.roots.as<int32_t>(), e.mesh_info.as<float>(), dQ, perm, q_off,     \
                       b_off, order, M, nb, bpts, run, lds_nodes, omega, inside, flag)
    if (e.opt.leaf_max > 1) FWN_QUAD(true);
    else FWN_QUAD(false);
#undef FWN_QUAD
    FWN_LAUNCH_CHECK("k_traverse_quad");
}

} // namespace fwn
