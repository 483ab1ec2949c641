// field_limits.hpp -- which volumes the kernels with 32-bit byte offsets into a
// field of three floats a voxel may take.  Plain C++ (no HIP), so the limits are
// tested on a CPU-only host.
#pragma once

#include <cstddef>

namespace tiplhip {

constexpr size_t kVoxelBytes = 12;  // a displacement: three floats

// Unsigned offsets: the whole field, its length included, below 2^32 bytes.
inline bool field_fits_32(size_t voxels) { return voxels * kVoxelBytes < (size_t(1) << 32); }

// Signed offsets that also run over the planes and rows a marched tile reaches
// outside the volume: below 2^31.
inline bool marched_field_fits(size_t voxels, size_t plane, size_t row)
{
    return (voxels + 8 * plane + 64 * row + 64) * kVoxelBytes < (size_t(1) << 31);
}

}  // namespace tiplhip
