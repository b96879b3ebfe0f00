// FP64 sum of every triangle's exact solid angle at each point (verification hook).
//
// Bound: FP64 VALU.  Built with machine LICM, which keeps the constants of the arctangent and the square
// roots in registers through the loop over the triangles: 4,000 points of 20,172 triangles 10.8 ms, 12.7
// without it, as the traversals are built.
#include <hip/hip_runtime.h>

#include "fwn_eval.h"
#include "fwn_internal.h"

namespace fwn {

namespace {

__global__ __launch_bounds__(256) void k_bruteforce(const uint32_t* __restrict__ tris, int64_t first, int64_t cnt,
                                                    const float* __restrict__ Q, int64_t nQ,
                                                    double* __restrict__ out)
{
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    bool valid = i < nQ;
    float qx = valid ? Q[3 * i] : 0.0f, qy = valid ? Q[3 * i + 1] : 0.0f, qz = valid ? Q[3 * i + 2] : 0.0f;
    double s = 0.0;
    for (int64_t t = first; t < first + cnt; ++t)
        s += tri_f64(reinterpret_cast<const float*>(tris + t * kTriWords), qx, qy, qz);
    if (valid) out[i] = s;
}

} // namespace

void run_bruteforce(Engine& e, const float* Q, int64_t nQ, double* out, bool dev)
{
    hipStream_t s = e.stream;
    if (nQ <= 0) return;
    const float* dQ = Q;
    double* dOut = out;
    if (!dev) {
        e.q_in.reserve(sizeof(float) * 3 * nQ);
        e.q_bf.reserve(sizeof(double) * nQ);
        FWN_HIP(hipMemcpyAsync(e.q_in.p, Q, sizeof(float) * 3 * nQ, hipMemcpyHostToDevice, s));
        dQ = e.q_in.as<float>();
        dOut = e.q_bf.as<double>();
    }
    // mesh 0's triangles are the first f_off[1] entries of the sorted triangle array
    const int64_t cnt = e.h_f_off.size() > 1 ? e.h_f_off[1] : 0;
    hipLaunchKernelGGL(k_bruteforce, dim3(grid_blocks(nQ, 256)), dim3(256), 0, s, e.tris.as<uint32_t>(), (int64_t)0,
                       cnt, dQ, nQ, dOut);
    FWN_LAUNCH_CHECK("k_bruteforce");
    if (!dev) FWN_HIP(hipMemcpyAsync(out, dOut, sizeof(double) * nQ, hipMemcpyDeviceToHost, s));
    FWN_HIP(hipStreamSynchronize(s));
}

} // namespace fwn
