// Memory of the cells that the voxel medium's adjoint adds its density gradient into (grid.hip).
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace cupbr {

constexpr uint32_t kGradCopies = 8;
constexpr size_t kMaxGradCopyBytes = (size_t)8 << 30;  // of all copies

// Copies of the cells (`bytes` each) to use: kGradCopies, halved until they fit kMaxGradCopyBytes and, beyond the
// `held` bytes that the scene has already, a quarter of the free memory: the buffer stays with the scene, and a
// program's own tensors need the rest. 256^3 voxels: 4.3 GB. 0: none, the adjoint adds to the gradient itself.
inline uint32_t cell_copies(size_t bytes, size_t held, size_t free_bytes) {
    const size_t limit = std::min(kMaxGradCopyBytes, std::max(held, free_bytes / 4 + held / 4));
    uint32_t copies = kGradCopies;
    while (copies > 0 && bytes * copies > limit) copies >>= 1;
    return copies;
}

}  // namespace cupbr
