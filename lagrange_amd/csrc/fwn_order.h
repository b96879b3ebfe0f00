// Layout of the point keys, in plain C++ for the kernels and for the host.
#pragma once

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

} // namespace fwn
