// Layout of the point keys and the points of a call that are looked at, in plain C++ for the kernels and
// for the host.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>

#ifdef __HIPCC__
#define FWN_HD __host__ __device__ __forceinline__
#else
#define FWN_HD inline
#endif

namespace fwn {

// 32-bit point key: mesh id in the top mesh_bits bits, then the leading bits of the point's 30-bit
// Morton code, `first` of them unused below the mesh id (a sort of fewer bits than the key has takes 0;
// 2 - mesh_bits, where that is positive, is the code as it is).
FWN_HD uint32_t point_key_of(uint32_t code30, uint32_t mesh, int mesh_bits, int first)
{
    const int bits = 32 - mesh_bits - first; // left for the code
    const uint32_t key = bits >= 30 ? code30 << (bits - 30) : code30 >> (30 - bits);
    return mesh_bits > 0 ? key | mesh << (32 - mesh_bits) : key;
}

// bits below the mesh id that the sort of 24 bits leaves unused: its order is that of the 22 leading
// Morton bits of a single mesh, and closest points of exact ties depend on it
FWN_HD int sort24_first(int mesh_bits) { return mesh_bits < 2 ? 2 - mesh_bits : 0; }

// The 2^bits points of a call of n >= 2^bits that are looked at: one from each of as many equal parts, at a
// hashed place (a fixed stride meets the same few columns of a regular grid again and again)
FWN_HD int64_t look_index(uint32_t part, int bits, int64_t n)
{
    const int64_t a = (int64_t)part * n >> bits, e = ((int64_t)part + 1) * n >> bits;
    uint32_t h = part;
    h ^= h >> 16;
    h *= 0x7feb352du;
    h ^= h >> 15;
    h *= 0x846ca68bu;
    h ^= h >> 16;
    return a + (int64_t)((uint64_t)h * (uint64_t)(e - a) >> 32);
}

// Whether points are spread over a mesh's box: of 8,192 cells of the box (points outside it count at its
// faces), the share that holds one of 8,192 points taken evenly from the call.  Uniform points and grids in
// the box 0.63, in one 1.2 and 1.5 times its size 0.49 to 0.55 and 0.42; layers on and off the surface of
// spheres, tori, plates and rods 0.19 to 0.27; 3 times its size (1 point in 27 inside) 0.19.
constexpr double kSpreadLeast = 0.35;

// The same for a dense grid of points in the box [lo, hi] against a mesh's box (info: its lower corner and
// the reciprocals of its sides, 0 for a flat one), without a look: the share of the mesh's box that the grid
// covers and the share of its points that lie there (cells at the faces, about 0.1, are left out).
inline bool box_spreads(const double lo[3], const double hi[3], const float info[6])
{
    double covered = 1.0, inside = 1.0;
    for (int d = 0; d < 3; ++d) {
        const double a = info[d], b = info[3 + d] > 0.0f ? a + 1.0 / info[3 + d] : a;
        const double both = std::max(std::min(hi[d], b) - std::max(lo[d], a), 0.0);
        if (b > a) covered *= both / (b - a);
        if (hi[d] > lo[d]) inside *= b > a ? both / (hi[d] - lo[d]) : 1.0;
    }
    return covered > 0.0 && covered * (1.0 - std::exp(-inside / covered)) >= kSpreadLeast - 0.15;
}

} // namespace fwn
