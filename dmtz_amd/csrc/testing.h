// Entry points for this repository's tests, not part of the library's interface (include/dmtz.h): the sizes
// at which a context changes its route, and the device arrays that its last call left.
#pragma once
#include <cstdint>

#include "../../include/dmtz.h"

extern "C" {

// The sizes of dmtz_ctx::lim, in its order; a negative value restores the library's own.
constexpr int DMTZ_TESTING_LIMITS = 6;
void dmtz_testing_limits(dmtz_ctx* ctx, const int64_t* values);

// Star codes of f and g (4 n words each, word by word), the f-critical and the mismatch masks (n each) and
// the tiles' counts ((n + 2047) / 2048) of the last call on n vertices.
int dmtz_testing_state(dmtz_ctx* ctx, int64_t n, uint64_t* code_f, uint64_t* code_g, uint64_t* critf_lo,
                       uint32_t* critf_hi, uint64_t* mm_lo, uint32_t* mm_hi, uint32_t* tile_nz);
}
