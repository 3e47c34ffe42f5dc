// drift_check.h -- what the counts of a drift must agree in (drift.f90:139-143).
#pragma once
#include <cstdint>

namespace cube {

// A drift that counts its destinations from the offsets: the particles that the rank
// pass gave a place (ranked) are those the offsets hold (placed).  Where every
// buffer cell is the image of a physical one (images), each physical particle (of
// `physical`, negative: not known) goes to one destination.
inline bool drift_counts_agree(int64_t ranked, int64_t placed, bool images, int64_t physical) {
  return ranked == placed && (!images || physical < 0 || placed == physical);
}

}  // namespace cube
