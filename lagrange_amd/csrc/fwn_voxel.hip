// Winding-number sign of voxels: the interior test that lagrange::volume::mesh_to_volume runs
// per voxel with Sign::WindingNumber (modules/volume/src/mesh_to_volume.cpp:156-183), batched.
//
// The reference maps voxel (i, j, k) to world space with OpenVDB's linear transform of scale
// voxel_size post-translated by voxel_size / 2 (mesh_to_volume.cpp:147-149), in double, then
// rounds each coordinate to float (:175-181) and calls is_inside.  Here the voxel centres are
// generated on the device with the same double arithmetic (a multiply and an add, each rounded,
// no fused multiply-add), rounded to float, and answered by the query path of the engine.  The
// caller never builds a host array of points.
#include <hip/hip_runtime.h>

#include <cstring>

#include "fwn_internal.h"
#include "fwn_order.h"

namespace fwn {
namespace {

__device__ __forceinline__ float voxel_coord(int64_t idx, double vs, double half)
{
#pragma clang fp contract(off)
    const double w = (double)idx * vs;
    return (float)(w + half);
}

// a / b for b that may be beyond 32 bits (then 0: a is not)
__device__ __forceinline__ uint32_t quotient(uint32_t a, uint64_t b)
{
    return b > a ? 0u : a / (uint32_t)b;
}

// Dense box: voxel t = x + dx (y + dy z) has index lo + (x, y, z); n < 2^31 voxels.  With `order`, also
// the voxels in the order the batched traversals want them, close together in space: blocks of 4 x 4
// x 4 (those at the far faces cut short), x fastest, a whole block's voxels in Morton order so that
// every 8 and 16 of them are compact too.  A wave of 64 points is a block, or parts of two neighbours
// after a cut one.  One 4-byte write per voxel in place of point keys and three sort passes (3.5M
// voxels: 21 us, the centres and the sort before 17 + 100; the traversal 791 -> 779 us in this order).
__global__ __launch_bounds__(256) void k_voxel_box(int32_t lx, int32_t ly, int32_t lz, uint32_t dx, uint32_t dy,
                                                   uint32_t dz, uint32_t n, double vs, float* __restrict__ P,
                                                   uint32_t* __restrict__ order)
{
    const uint32_t j = blockIdx.x * 256u + threadIdx.x;
    if (j >= n) return;
    const uint64_t layer = (uint64_t)dx * dy;
    uint32_t x, y, z;
    if (!order) {
        z = quotient(j, layer);
        const uint32_t r = j - z * (uint32_t)layer;
        y = r / dx;
        x = r - y * dx;
    } else {
        const uint32_t z0 = quotient(j, 4 * layer) * 4, hz = min(dz - z0, 4u);
        const uint32_t in_layer = j - z0 * (uint32_t)layer;
        const uint32_t y0 = quotient(in_layer, (uint64_t)dx * 4 * hz) * 4, hy = min(dy - y0, 4u);
        const uint32_t in_row = in_layer - y0 * dx * hz;
        const uint32_t x0 = in_row / (4 * hy * hz) * 4, hx = min(dx - x0, 4u);
        const uint32_t k = in_row - x0 * hy * hz;
        if (hx == 4 && hy == 4 && hz == 4) {
            x = (k & 1) | ((k >> 2) & 2);
            y = ((k >> 1) & 1) | ((k >> 3) & 2);
            z = ((k >> 2) & 1) | ((k >> 4) & 2);
        } else {
            x = k % hx;
            y = k / hx % hy;
            z = k / (hx * hy);
        }
        x += x0;
        y += y0;
        z += z0;
    }
    const uint32_t t = x + dx * (y + dy * z);
    if (order) order[j] = t;
    const double half = vs * 0.5;
    P[3 * (size_t)t + 0] = voxel_coord((int64_t)lx + x, vs, half);
    P[3 * (size_t)t + 1] = voxel_coord((int64_t)ly + y, vs, half);
    P[3 * (size_t)t + 2] = voxel_coord((int64_t)lz + z, vs, half);
}

// explicit list of (i, j, k) int32 triples
__global__ __launch_bounds__(256) void k_voxel_list(const int32_t* __restrict__ ijk, int64_t n, double vs,
                                                    float* __restrict__ P)
{
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= 3 * n) return;
    P[t] = voxel_coord(ijk[t], vs, vs * 0.5);
}

} // namespace

// Generate the centres (and, for a box, their order) into the engine's scratch and answer them;
// outputs host or device.
static void sign_centres(Engine& e, int64_t n, uint8_t* inside, float* omega, bool dev,
                         const uint32_t* (*gen)(Engine&, float*, const void*), const void* arg, Points where)
{
    hipStream_t s = e.stream;
    e.v_pts.reserve(sizeof(float) * 3 * n);
    const uint32_t* order = gen(e, e.v_pts.as<float>(), arg);
    float* dOm = omega;
    uint8_t* dIn = inside;
    if (!dev || !omega) {
        e.v_om.reserve(sizeof(float) * n);
        dOm = e.v_om.as<float>();
    }
    if (!dev) {
        e.v_in.reserve(n);
        dIn = e.v_in.as<uint8_t>();
    }
    run_queries(e, e.v_pts.as<float>(), nullptr, n, dOm, dIn, nullptr, true, order, where);
    if (!dev) {
        FWN_HIP(hipMemcpyAsync(inside, dIn, n, hipMemcpyDeviceToHost, s));
        if (omega) FWN_HIP(hipMemcpyAsync(omega, dOm, sizeof(float) * n, hipMemcpyDeviceToHost, s));
    }
    FWN_HIP(hipStreamSynchronize(s));
}

struct BoxArg {
    int32_t lo[3];
    int64_t dims[3];
    int64_t n;
    double vs;
};
struct ListArg {
    const int32_t* ijk;
    int64_t n;
    double vs;
    bool dev;
};

static const uint32_t* gen_box(Engine& e, float* P, const void* a)
{
    const BoxArg& b = *static_cast<const BoxArg*>(a);
    uint32_t* order = nullptr;
    if (!few_points(e, b.n)) { // those are answered in any order
        e.q_vals[0].reserve(sizeof(uint32_t) * b.n);
        order = e.q_vals[0].as<uint32_t>();
    }
    hipLaunchKernelGGL(k_voxel_box, dim3(grid_blocks(b.n, 256)), dim3(256), 0, e.stream, b.lo[0], b.lo[1], b.lo[2],
                       (uint32_t)b.dims[0], (uint32_t)b.dims[1], (uint32_t)b.dims[2], (uint32_t)b.n, b.vs, P, order);
    FWN_LAUNCH_CHECK("k_voxel_box");
    return order;
}

static const uint32_t* gen_list(Engine& e, float* P, const void* a)
{
    const ListArg& l = *static_cast<const ListArg*>(a);
    const int32_t* dijk = l.ijk;
    if (!l.dev) {
        e.v_ijk.reserve(sizeof(int32_t) * 3 * l.n);
        FWN_HIP(hipMemcpyAsync(e.v_ijk.p, l.ijk, sizeof(int32_t) * 3 * l.n, hipMemcpyHostToDevice, e.stream));
        dijk = e.v_ijk.as<int32_t>();
    }
    hipLaunchKernelGGL(k_voxel_list, dim3(grid_blocks(3 * l.n, 256)), dim3(256), 0, e.stream, dijk, l.n, l.vs, P);
    FWN_LAUNCH_CHECK("k_voxel_list");
    return nullptr;
}

static void check_voxel_size(double vs)
{
    if (!(vs > 0.0) || !(vs < 1e300)) fail(FWN_INVALID_ARGUMENT, "voxel_size must be a positive finite number");
}

void sign_voxel_box(Engine& e, const int32_t lo[3], const int32_t dims[3], double vs, uint8_t* inside, float* omega,
                    bool dev)
{
    check_voxel_size(vs);
    BoxArg b{};
    b.n = 1;
    for (int d = 0; d < 3; ++d) {
        if (dims[d] < 0) fail(FWN_INVALID_ARGUMENT, "negative box dimension");
        if ((int64_t)lo[d] + dims[d] - 1 > INT32_MAX) fail(FWN_INVALID_ARGUMENT, "voxel index beyond int32");
        b.lo[d] = lo[d];
        b.dims[d] = dims[d];
        b.n *= dims[d];
        if (b.n > (int64_t)UINT32_MAX / 2) fail(FWN_LIMIT_EXCEEDED, "more than 2^31 voxels in one call");
    }
    b.vs = vs;
    if (b.n == 0) return;
    if (!inside) fail(FWN_INVALID_ARGUMENT, "inside_out is NULL");
    // no sort runs while the points could be looked at, and a box says where they lie
    Points where = Points::Any;
    if (e.n_meshes == 1) {
        double from[3], to[3];
        for (int d = 0; d < 3; ++d) {
            from[d] = vs * lo[d];
            to[d] = vs * ((double)lo[d] + dims[d]);
        }
        where = box_spreads(from, to, e.h_info.data()) ? Points::Spread : Points::Close;
    }
    sign_centres(e, b.n, inside, omega, dev, gen_box, &b, where);
}

void sign_voxel_list(Engine& e, const int32_t* ijk, int64_t n, double vs, uint8_t* inside, float* omega, bool dev)
{
    check_voxel_size(vs);
    if (n < 0) fail(FWN_INVALID_ARGUMENT, "negative voxel count");
    if (n == 0) return;
    if (!ijk || !inside) fail(FWN_INVALID_ARGUMENT, "NULL voxel list or inside_out");
    if (n > (int64_t)UINT32_MAX / 2) fail(FWN_LIMIT_EXCEEDED, "more than 2^31 voxels in one call");
    ListArg l{ijk, n, vs, dev};
    sign_centres(e, n, inside, omega, dev, gen_list, &l, Points::Any);
}

} // namespace fwn
