// What the prompt launches share (dense_tile.hip, prompt.hip): the sizes of a prompt's A and B fragments and of a block's
// sums in shared memory.
#pragma once

#include "dense.hpp"

namespace esp {

constexpr int TILE_FRAG = 512;                  // halves an MFMA operand block (16 rows or columns, 32 k): 64 lanes x 8
constexpr int RED_STRIDE = 132;                 // floats between two rows of the block's sums (banks apart)

typedef __attribute__((address_space(3))) const f16x8* lds_f16x8_ptr;

}  // namespace esp
