// Internal declarations of the MI355X fast winding number engine (not part of the C ABI).
#pragma once

#include <hip/hip_runtime.h>

#include <condition_variable>
#include <cstdint>
#include <algorithm>
#include <atomic>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include "../../include/fwn.h"

namespace fwn {

// ---------------------------------------------------------------------------------------
// error plumbing: C-ABI functions never throw; internal code throws fwn::Failure which the
// ABI layer turns into a status code + thread-local message.
// ---------------------------------------------------------------------------------------
struct Failure {
    int status;
    std::string msg;
};

void set_error(const std::string& msg);
[[noreturn]] void fail(int status, const std::string& msg);
void hip_check(hipError_t e, const char* what, const char* file, int line);

#define FWN_HIP(call) ::fwn::hip_check((call), #call, __FILE__, __LINE__)
#define FWN_LAUNCH_CHECK(name) ::fwn::hip_check(hipGetLastError(), name, __FILE__, __LINE__)

// ---------------------------------------------------------------------------------------
// constants shared by host and device code
// ---------------------------------------------------------------------------------------
constexpr int kWidth = FWN_WIDTH;          // maximum slots per node
constexpr int kSlotWords = FWN_SLOT_WORDS; // 32-bit words per slot
constexpr int kTriWords = FWN_TRI_WORDS;   // 32-bit words per stored triangle
constexpr int kBoxWords = 16;              // 32-bit words per slot box record
constexpr int kRecWords = 32;              // doubles per binary-node moment record
constexpr int kStack = 192;                // per-wave traversal stack entries
constexpr double kFixScale = 1099511627776.0; // 2^40: fixed-point scale of FP64 near-field sums
constexpr int kWave = 64;

// binary-node moment record layout (doubles)
enum : int { R_A = 0, R_P = 1, R_N = 4, R_M1 = 7, R_S = 16, R_LO = 26, R_HI = 29 };

// RAII device buffer
struct DBuf {
    void* p = nullptr;
    size_t bytes = 0;
    DBuf() = default;
    DBuf(const DBuf&) = delete;
    DBuf& operator=(const DBuf&) = delete;
    ~DBuf() { release(); }
    void release();
    void alloc(size_t n);          // exact (re)allocation, contents undefined
    void reserve(size_t n);        // grow only
    template <class T> T* as() const { return static_cast<T*>(p); }
};

// one single-point query waiting to be answered in a coalesced batch
struct PointRequest {
    float q[3];
    float omega = 0.0f;
    uint8_t inside = 0;
    int status = 0;
    std::string err;
    std::atomic<bool> done{false}; // set (release) after the fields above, under the engine's pt_mu
};

struct Engine {
    int device = 0;
    hipStream_t stream = nullptr;
    std::mutex mu;
    // concurrent single-point calls are answered together: a caller that finds no batch running
    // takes every pending request and answers them in one query
    std::mutex pt_mu;
    std::condition_variable pt_cv;
    std::vector<PointRequest*> pt_pending;
    bool pt_busy = false;
    size_t pt_conc = 1; // requests the last coalesced batch held (how many callers to expect)
    fwn_options opt{};

    int32_t n_meshes = 0;
    bool uneven = false; // several meshes, the largest of at least 1.5 times their mean number of triangles
    int32_t width = 4;         // slots per node
    int64_t n_tris = 0;
    int64_t n_nodes = 0;
    int32_t max_depth = 0;
    double build_ms = 0.0;

    // tree (resident)
    DBuf slots;      // n_nodes * width * kSlotWords u32
    DBuf boxes;      // n_nodes * width * kBoxWords, for distance queries: each slot's box (lo, hi), its link and its
                     // disk (t, c, R, n): the triangles are within t of the plane through c normal to n and within
                     // R of the axis; infinity where that bounds nothing
    DBuf tris;       // n_tris * kTriWords u32
    DBuf roots;      // 2 int32 per mesh: wide root, occupied slots
    DBuf mesh_info;  // per mesh: 8 floats: qbox lo[3], qbox inv[3], tau, pad
    std::vector<int32_t> h_roots;
    std::vector<float> h_tau;
    std::vector<float> h_info; // host copy of mesh_info
    std::vector<int64_t> h_f_off;

    // query scratch (grown on demand)
    DBuf q_keys[2], q_vals[2], q_hist, q_rowsum, q_in, q_om, q_in8, q_stats, q_flag;
    DBuf q_bf;
    DBuf v_pts, v_om, v_in, v_ijk; // query points generated on the device and their outputs
    DBuf c_V, c_F, c_err, c_out, c_pos, c_scan, c_outp; // orientation / sampling scratch
    DBuf d_d2, d_tri, d_cp;                               // closest-point outputs for host callers
    int n_cu = 0;

    // pinned host staging: metadata, points and results of small calls, and the words the host polls.  A call
    // that has polled its words returns before its kernels have retired, and the next one writes the stage at
    // once: no kernel touches the stage after the mark that the host waits for (k_point_bfs and k_publish
    // fence the overflow flag before it), and every other use ends with the stream synchronised.
    void* h_stage = nullptr;
    size_t h_stage_bytes = 0;
    DBuf q_ptflag; // overflow flag of few-point calls
    DBuf q_meta; // device copy of the staged metadata (and small host batches' points)
    std::vector<char> meta_dev; // the metadata bytes q_meta holds (compared before an upload)
    // pipelined host calls: pinned double buffers (points in, results out), a stream per copy
    // direction, per-chunk flags
    void* h_pipe = nullptr;
    size_t h_pipe_bytes = 0;
    hipStream_t cs_in = nullptr, cs_out = nullptr;
    hipEvent_t pev[6] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr}; // h2d[2], comp[2], d2h[2]
    DBuf q_pmeta, q_pflags;

    hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
    std::vector<hipEvent_t> tev; // pipelined calls: a (start, end) pair around each chunk's traversal
    double last_traverse_ms = 0.0;
    double last_total_ms = 0.0;
};

// sorting / scanning primitives (fwn_sort.hip)
// Stable LSD radix sort of (keys, vals) pairs by key bits [0, nbits).  Result ends in keys/vals
// (swapping with the scratch buffers as needed; the pointers are updated).
void radix_sort_pairs(uint64_t*& keys, uint32_t*& vals, uint64_t*& keys_alt, uint32_t*& vals_alt, int64_t n,
                      int nbits, DBuf& hist, DBuf& rowsum, hipStream_t s);
// Same for 32-bit keys, sorting key bits [begin_bit, end_bit) only (low bits keep input order).
// vals_are_index: the input values are not read; value i is taken to be i (the sorted values are
// then the permutation), so the key kernel need not write them.
void radix_sort_pairs32(uint32_t*& keys, uint32_t*& vals, uint32_t*& keys_alt, uint32_t*& vals_alt, int64_t n,
                        int begin_bit, int end_bit, bool vals_are_index, DBuf& hist, DBuf& rowsum, hipStream_t s);
// The same over caller-provided histogram scratch (no allocation): hist holds
// radix_sort_hist_words(n) int32, rowsum 256 int32.
int64_t radix_sort_hist_words(int64_t n);
// The top 20 bits of at most kFewTiles tiles of keys, whose first 10-bit digit (bits 12 to 21) the kernel
// that made them has counted into hist (kFewTile keys a tile, 1,024 int32 each): vals receives the input
// positions in stable order of those bits.
constexpr int kFewTile = 4096, kFewTiles = 128;
inline int few_tiles(int64_t n) { return (int)((n + kFewTile - 1) / kFewTile); }
void sort_few_tiles(const uint32_t* keys, uint32_t* keys_alt, uint32_t* vals_alt, uint32_t* vals, int64_t n,
                    int32_t* hist, hipStream_t s);
void radix_sort_pairs32_scratch(uint32_t*& keys, uint32_t*& vals, uint32_t*& keys_alt, uint32_t*& vals_alt, int64_t n,
                                int begin_bit, int end_bit, bool vals_are_index, int32_t* hist, int32_t* rowsum,
                                hipStream_t s);
// exclusive scan of int32 (in may alias out); returns nothing, total in out[n] if out has n+1 slots
void exclusive_scan_i32(const int32_t* in, int32_t* out, int64_t n, DBuf& tmp, hipStream_t s);

// build (fwn_build.hip)
void build_engine(Engine& e, int32_t n_meshes, const float* V_host, const int64_t* v_off, const int32_t* F_host,
                  const int64_t* f_off);

// Scratch of one build: pieces taken from a few device allocations, all freed at the end.  The
// allocations stay below 64 MB where a single piece does not need more (hipFree takes 12-25 us up to
// 64 MB and 300 us above, per allocation).
struct Arena {
    static constexpr size_t kBlock = (size_t)60 << 20;
    std::vector<std::unique_ptr<DBuf>> blocks;
    size_t used = 0, expect = 0; // of the last block; bytes still expected to be taken
    explicit Arena(size_t expected) : expect(expected) {}
    void* take_bytes(size_t n)
    {
        n = (std::max<size_t>(n, 1) + 255) & ~(size_t)255;
        if (blocks.empty() || used + n > blocks.back()->bytes) {
            blocks.emplace_back(new DBuf());
            blocks.back()->alloc(std::max(n, std::min(kBlock, std::max<size_t>(expect, (size_t)1 << 20))));
            used = 0;
        }
        void* p = static_cast<char*>(blocks.back()->p) + used;
        used += n;
        expect -= std::min(expect, n);
        return p;
    }
    template <class T>
    T* take(int64_t count)
    {
        return static_cast<T*>(take_bytes(sizeof(T) * (size_t)std::max<int64_t>(count, 0)));
    }
};

// SAH topology (fwn_sah.hip): top-down binned box-area splits of each mesh's triangles down to
// single triangles, in the binary tree layout of the LBVH path: internal nodes [0, n-1), leaf j
// -> n-1+j for the triangle at sorted position j, `items` = sorted position -> triangle,
// left/right/first/last per internal node, parent per node of a mesh's tree, is_root (the caller
// fills 0) and root_bin per mesh.  boxes: the triangle setup's 12 ints per mesh.  A mid segment (at
// most kSahMid triangles, 4 ints in the returned list: lo, hi, parent, side) is a subtree over the
// sorted positions [lo, hi) whose internal nodes have the ids [lo, hi - 2].
constexpr int kSahMid = 1024;
struct SahMids {
    const int32_t* seg; // device
    int64_t count;
};
SahMids build_topology_sah(Engine& e, Arena& ar, const float* cen, const float* tbox, const int32_t* boxes, int64_t nF,
                           const int64_t* f_off, int M, int32_t* items, int32_t* left, int32_t* right, int32_t* parent,
                           int32_t* first, int32_t* last, uint8_t* is_root, int32_t* root_bin);

// What a caller knows of its points (a choice of kernel only, the results are the same): nothing, that they
// lie in layers along a surface, or that they are a dense grid, spread over the mesh's box or not.
enum class Points { Any, Layer, Spread, Close };
// queries (fwn_query.hip).  order: device positions -> points of one mesh that are already in an order
// of waves (nullptr: the call sorts its points); not read by calls that need no order (few_points).
void run_queries(Engine& e, const float* Q, const int64_t* q_off_host, int64_t nQ, float* omega, uint8_t* inside,
                 int32_t* stats, bool device_ptrs, const uint32_t* order = nullptr, Points where = Points::Any);
// whether a device call of nQ points of one mesh runs one wave per point
bool few_points(const Engine& e, int64_t nQ);
void run_bruteforce(Engine& e, const float* Q, int64_t nQ, double* out, bool device_ptrs);
// pinned staging buffer of at least this many bytes (contents undefined when it grows)
char* host_stage(Engine& e, size_t bytes);
// whether the engine has the default launch shape (the others are k_traverse's, chosen by the tuner
// or the caller)
inline bool default_shape(const Engine& e)
{
    return e.opt.launch_mode == FWN_LAUNCH_GRID && e.opt.waves_per_block <= 1;
}
// Calls of few points of a single-mesh engine, one wave per point (fwn_point.hip).
void run_points(Engine& e, const float* Q, int64_t nQ, float* omega, uint8_t* inside, int banks, bool device_ptrs);
// The slots-in-lanes traversal (fwn_quad.hip): whether a call goes to it, and its launch over nb batches of
// bpts points (metadata as k_traverse's); FP64 near leaves are evaluated in the kernel, flag is set on a
// stack overflow.  Look: quads_after_look says, once the n points of the mesh with the most of them (`most`)
// have been looked at: how many of 2^kLookBits cells of its box hold one of as many points, and (none unless
// quads_near_surface) the threshold of the last slot of kLookWalks walks.
constexpr int kQuadPoints = 16;
constexpr int kLookBits = 13, kLookWalks = 256;
// Layers cross where 64 neighbours extend over about 1.8 times their distance from the surface, and the last
// slot's threshold is about twice that distance^2.  k_traverse / slots in lanes in us at extent / distance: 64
// meshes of 199,692 triangles, 1 % of the diagonal off, 8 (12k points each) 1647 / 836, 5.5 (25k) 2039 / 1337, 3.9
// (50k) 2733 / 2135; 16 of them 2.8 (100k) 1087 / 974, 1.6 (300k) 2171 / 2364; 5 % off 1.6 (64 x 12k) 337 / 342,
// 1.1 (64 x 25k) 460 / 534, 0.8 (16 x 50k) 278 / 310
constexpr float kLookNear = 0.6f;
enum class Quads { No, Yes, Look };
Quads use_quads(const Engine& e, int64_t nQ, int64_t most, int banks, Points where);
bool quads_near_surface(const Engine& e, int64_t nQ);
bool quads_after_look(const Engine& e, int mesh, int64_t n, int cells, const float* last, int walks);
void launch_quads(Engine& e, const float* dQ, const uint32_t* perm, const int64_t* q_off, const int64_t* b_off,
                  const int32_t* order, int M, int64_t nb, int bpts, Points where, float* omega, uint8_t* inside,
                  int32_t* flag, hipStream_t s);
int quad_points(const Engine& e, int64_t nQ); // points per wave, kQuadPoints at most
// Pieces of a query that uses no engine scratch (single-mesh engine, device points): the 32-bit
// point keys, and the traversal in sorted order `perm`; meta holds q_off {0, nQ}, b_off {0, batches} and the mesh order {0} (5 int64
// words), flag one int32 (set on stack overflow).  Results equal run_queries' bit for bit.
void launch_point_keys(Engine& e, const float* dQ, int64_t nQ, uint32_t* keys, hipStream_t s);
void launch_traverse_inplace(Engine& e, int banks, const float* dQ, const uint32_t* perm, const int64_t* meta,
                             int64_t nQ, float* omega, uint8_t* inside, int32_t* flag, hipStream_t s);
// fwn_solid_angle_noalloc (fwn_noalloc.hip): device points of a single-mesh engine through a fixed
// device scratch array; no allocation
void run_queries_noalloc(Engine& e, const float* dQ, int64_t nQ, float* dOm, uint8_t* dIn);
// Morton order of nQ device points of a single-mesh engine: returns the permutation (sorted
// position -> original index) in the engine's query scratch, valid until the next query call.
const uint32_t* sort_points_single(Engine& e, const float* dQ, int64_t nQ);

// closest point on the mesh of a single-mesh engine (fwn_closest.hip): squared distance (double),
// original facet index (-1 for an empty mesh) and, when cp is not NULL, the point (3 doubles)
void run_closest(Engine& e, const float* Q, int64_t nQ, double* d2, int32_t* tri, double* cp, bool device_ptrs);

// voxel signs (fwn_voxel.hip): centres float(voxel_size * ijk + voxel_size / 2) made on the device
void sign_voxel_box(Engine& e, const int32_t lo[3], const int32_t dims[3], double voxel_size, uint8_t* inside,
                    float* omega, bool device_ptrs);
void sign_voxel_list(Engine& e, const int32_t* ijk, int64_t n, double voxel_size, uint8_t* inside, float* omega,
                     bool device_ptrs);

// batched example callers (fwn_callers.hip)
void orientation_criterion(Engine& e, const float* V, int64_t nV, const int32_t* F, int64_t nF, float eps,
                           double* crit, bool device_ptrs);
void sample_inside(Engine& e, const float lo[3], const float hi[3], int64_t n, uint64_t seed, float* out,
                   int64_t* n_inside, bool device_ptrs);

int grid_blocks(int64_t n, int threads);

// validates an options struct (throws Failure)
void check_options(const fwn_options& o);

// Sets the current device for a scope and restores the previous one.
struct DeviceGuard {
    int prev = -1;
    explicit DeviceGuard(int dev)
    {
        if (hipGetDevice(&prev) != hipSuccess) prev = -1;
        FWN_HIP(hipSetDevice(dev));
    }
    ~DeviceGuard()
    {
        if (prev >= 0) (void)hipSetDevice(prev);
    }
};

// Runs body, turning failures into a status code and the thread-local error message.
template <class Body>
int guarded(const char* fn, Body&& body)
{
    try {
        body();
        return FWN_OK;
    } catch (const Failure& f) {
        set_error(std::string(fn) + ": " + f.msg);
        return f.status;
    } catch (const std::bad_alloc&) {
        set_error(std::string(fn) + ": host allocation failed");
        return FWN_OUT_OF_MEMORY;
    } catch (...) {
        set_error(std::string(fn) + ": unknown failure");
        return FWN_HIP_ERROR;
    }
}

} // namespace fwn

// ---------------------------------------------------------------------------------------
// device helpers
// ---------------------------------------------------------------------------------------
namespace fwn {

__device__ __forceinline__ uint32_t expand10(uint32_t v)
{
    v &= 0x3FFu;
    v = (v | (v << 16)) & 0x030000FFu;
    v = (v | (v << 8)) & 0x0300F00Fu;
    v = (v | (v << 4)) & 0x030C30C3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

// (c - lo) * inv scaled to [0, 1023]; same float operations as the CPU check
__device__ __forceinline__ uint32_t quant10(float c, float lo, float inv)
{
    float t = (c - lo) * inv;
    float s = t * 1024.0f;
    if (!(s > 0.0f)) return 0u;
    if (s >= 1023.0f) return 1023u;
    return (uint32_t)s;
}

__device__ __forceinline__ uint32_t morton30(float x, float y, float z, const float* lo, const float* inv)
{
    return (expand10(quant10(x, lo[0], inv[0])) << 2) | (expand10(quant10(y, lo[1], inv[1])) << 1) |
           expand10(quant10(z, lo[2], inv[2]));
}

// one key's digit into the block's counters; called with whole waves (a wave whose keys share one
// digit adds its count with one atomic: LDS atomics on one address serialise)
__device__ __forceinline__ void count_digit(int32_t* cnt, uint32_t d, bool valid)
{
    const uint64_t live = __ballot(valid);
    const uint32_t d0 = __builtin_amdgcn_readfirstlane(d);
    if ((__ballot(d != d0) & live) == 0ull) {
        if ((threadIdx.x & 63) == 0 && live != 0ull) atomicAdd(&cnt[d0], (int32_t)__popcll(live));
    } else if (valid) {
        atomicAdd(&cnt[d], 1);
    }
}

// order-preserving float <-> int maps for atomic min/max
__device__ __forceinline__ int32_t f2ord(float f)
{
    int32_t i = __float_as_int(f);
    return i >= 0 ? i : (i ^ 0x7FFFFFFF);
}
__host__ __device__ inline float ord2f(int32_t i)
{
    int32_t j = i >= 0 ? i : (i ^ 0x7FFFFFFF);
    float f;
    __builtin_memcpy(&f, &j, 4);
    return f;
}

// v_writelane_b32: returns `old` with lane `lane` replaced by the wave-uniform `v` (the LLVM
// intrinsic, which clang exposes under no builtin name)
extern "C" __device__ int fwn_llvm_writelane(int v, int lane, int old) __asm("llvm.amdgcn.writelane.i32");
__device__ __forceinline__ uint32_t wave_writelane(uint32_t v, int lane, uint32_t old)
{
    return (uint32_t)fwn_llvm_writelane((int)v, lane, (int)old);
}

// Wave-private traversal stack of (node entry, 64-bit lane mask), one entry per lane and bank:
// entry k lives in lane k % 64 of bank k / 64.  NB = 1 (64 entries, enough for trees with
// 1 + (width - 1) * depth <= 64) or 3 (kStack entries).  The entry and the mask are
// wave-uniform, so a push is one v_writelane per word (the written register is tied to the old
// one: no copies at the join of a conditional push) and a pop is one v_readlane per word; the
// bank is chosen by uniform branches, so nothing invites the optimiser to turn the banks into an
// indexed private array in scratch memory.  A push past the capacity writes no lane (callers
// report it as an overflow).
template <int NB>
struct WaveStack;

template <>
struct WaveStack<1> {
    static constexpr int kCap = 64;
    uint32_t n0 = 0, l0 = 0, h0 = 0;
    // sp < kCap is the caller's contract (the host launches this stack only for trees whose
    // bound fits; callers still flag sp >= kCap as an overflow): no guard here, so the push is
    // three writelanes with no branch around them
    __device__ __forceinline__ void push(int sp, int /*lane*/, uint32_t e, uint64_t mk)
    {
        n0 = wave_writelane(e, sp & 63, n0);
        l0 = wave_writelane((uint32_t)mk, sp & 63, l0);
        h0 = wave_writelane((uint32_t)(mk >> 32), sp & 63, h0);
    }
    __device__ __forceinline__ void pop(int sp, uint32_t& e, uint64_t& mk) const
    {
        const int l = sp & 63;
        e = __builtin_amdgcn_readlane(n0, l);
        const uint32_t lo = __builtin_amdgcn_readlane(l0, l), hi = __builtin_amdgcn_readlane(h0, l);
        mk = ((uint64_t)hi << 32) | lo;
    }
};

template <>
struct WaveStack<3> {
    static constexpr int kCap = kStack;
    uint32_t n0 = 0, n1 = 0, n2 = 0, l0 = 0, l1 = 0, l2 = 0, h0 = 0, h1 = 0, h2 = 0;
    __device__ __forceinline__ void push(int sp, int /*lane*/, uint32_t e, uint64_t mk)
    {
        const int l = sp & 63;
        const uint32_t mlo = (uint32_t)mk, mhi = (uint32_t)(mk >> 32);
        if (sp < 64) {
            n0 = wave_writelane(e, l, n0);
            l0 = wave_writelane(mlo, l, l0);
            h0 = wave_writelane(mhi, l, h0);
        } else if (sp < 128) {
            n1 = wave_writelane(e, l, n1);
            l1 = wave_writelane(mlo, l, l1);
            h1 = wave_writelane(mhi, l, h1);
        } else if (sp < kStack) {
            n2 = wave_writelane(e, l, n2);
            l2 = wave_writelane(mlo, l, l2);
            h2 = wave_writelane(mhi, l, h2);
        }
    }
    __device__ __forceinline__ void pop(int sp, uint32_t& e, uint64_t& mk) const
    {
        const int l = sp & 63;
        const uint32_t a0 = __builtin_amdgcn_readlane(n0, l), a1 = __builtin_amdgcn_readlane(n1, l),
                       a2 = __builtin_amdgcn_readlane(n2, l);
        const uint32_t c0 = __builtin_amdgcn_readlane(l0, l), c1 = __builtin_amdgcn_readlane(l1, l),
                       c2 = __builtin_amdgcn_readlane(l2, l);
        const uint32_t d0 = __builtin_amdgcn_readlane(h0, l), d1 = __builtin_amdgcn_readlane(h1, l),
                       d2 = __builtin_amdgcn_readlane(h2, l);
        const uint32_t lo = sp < 64 ? c0 : (sp < 128 ? c1 : c2);
        const uint32_t hi = sp < 64 ? d0 : (sp < 128 ? d1 : d2);
        e = sp < 64 ? a0 : (sp < 128 ? a1 : a2);
        mk = ((uint64_t)hi << 32) | lo;
    }
};

// stack banks a tree of this width and depth needs (1 or 3), 0 if it is too deep.  The bound
// 1 + (width - 1) depth on the live entries keeps one position free above the top: the traversal
// writes that position for leaf slots too (and only advances over it for internal ones).
inline int stack_banks(int width, int depth)
{
    const int need = 1 + (width - 1) * depth;
    return need < 64 ? 1 : (need < kStack ? 3 : 0);
}

// XCD-aware block remap: hardware hands consecutive workgroups to the 8 XCDs round-robin;
// this bijection gives each XCD one contiguous run of logical blocks (shared L2 reuse).
__device__ __forceinline__ uint32_t xcd_remap(uint32_t b, uint32_t nb)
{
    uint32_t per = nb / 8u, rem = nb % 8u;
    uint32_t x = b % 8u, i = b / 8u;
    return (x < rem) ? x * (per + 1u) + i : rem * (per + 1u) + (x - rem) * per + i;
}
// The same for blocks of uneven cost (numbered by mesh size, or of points deep inside a mesh): runs
// of `run` logical blocks go to the XCDs in turn, the rest of the grid as above.
__device__ __forceinline__ uint32_t xcd_remap_runs(uint32_t b, uint32_t nb, uint32_t run)
{
    const uint32_t dealt = nb / (8u * run) * (8u * run);
    if (b >= dealt) return dealt + xcd_remap(b - dealt, nb - dealt);
    const uint32_t x = b % 8u, i = b / 8u;
    return (i / run * 8u + x) * run + i % run;
}
// Batches of several meshes are numbered from the largest mesh to the smallest: in one run per XCD the last
// XCDs end early where the meshes are uneven (Engine::uneven), while even ones share less of an L2 in several.
// k_traverse in one run per XCD / in runs of 16 / 64: 32 meshes of 1.7k to 200k triangles, 50,000 points each,
// uniform 1636 / 1038 / 1073 us, near the surface 4141 / 1648 / 1648; 64 even ones of 20,172 triangles, a layer 12k
// 358 / 377 / 369 and 50k 713 / 750 / 735
__device__ __forceinline__ uint32_t xcd_batch(uint32_t b, uint32_t nb, int run)
{
    return run > 0 ? xcd_remap_runs(b, nb, (uint32_t)run) : xcd_remap(b, nb);
}

} // namespace fwn
