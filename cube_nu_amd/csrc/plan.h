// plan.h -- the kick's meshes within the workspace budget.
#pragma once
#include <algorithm>
#include <cstdint>

namespace cube {

// Bytes of one n^3 mesh of `real`-byte numbers and its half-complex transform, and
// of the six faces of one window of n^3 floats.
constexpr int64_t mesh_bytes(int64_t n, int64_t real) { return n * n * n * real + n * n * (n / 2 + 1) * 2 * real; }
constexpr int64_t face_bytes(int64_t n) { return 6 * n * n * 4; }

// Whether a whole-image mesh has room: at most half the budget (beyond that the
// windows' batches would suffer), and under a budget the caller has set, one mesh
// of the largest level beside it.
inline bool image_fits(int64_t budget, bool set, int64_t image, int64_t largest) {
  return image <= budget / 2 && (!set || image + largest <= budget);
}

// Meshes of a level held at once.  reserved: the bytes of whole-image meshes, which a
// budget the caller has set holds, too; the automatic one is that of the batches.
inline int64_t level_batch(int64_t budget, bool set, int64_t reserved, int64_t per, int64_t nmesh) {
  return std::max<int64_t>(1, std::min<int64_t>(nmesh, (budget - (set ? reserved : 0)) / per));
}

}  // namespace cube
