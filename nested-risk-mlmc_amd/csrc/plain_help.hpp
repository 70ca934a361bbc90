// When a block of a plain model call that has ended its own virtual thread stops
// looking for others' postings (k_model_parity's helping, model.hpp).
#pragma once
#include <stdint.h>

namespace nmlmc {

// started, ended: counters of blocks over all calls (they wrap); base: their value
// before this call, as the host has it.  A block leaves when every block of the
// call has ended, or at once while some have not started (they need the room).  The
// wait ends whatever base is: the counters of a call grow by `blocks` together, so
// that ended - base stays at or above `blocks` once it is there, and where base lies
// ahead of the counters both differences wrap to large values.  (Equality for the
// first test would be stepped over for good by a base that is behind.)
constexpr bool helper_leaves(uint32_t started, uint32_t ended, uint32_t base, uint32_t blocks) {
    return ended - base >= blocks || started - base < blocks;
}

}  // namespace nmlmc
