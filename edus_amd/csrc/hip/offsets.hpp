// Sizes of a context's arrays and the byte offsets of the 1..4-band stage kernel.
// No HIP in here: the tests compile it for the host.
#pragma once

#include <climits>
#include <cstddef>
#include <type_traits>

// Doubles of a context's packed state, padding included: its count is an int.
constexpr long long kMaxStateElems = INT_MAX;

// Byte offset of a k in a row of a structure-of-arrays state (1..4 bands, a row of
// padded k per packed element): 32 bits wherever the state's limit keeps 8 k below
// 2^32, which leaves a load's address to the scalar row and one register.  One band
// alone may have 2^29 k and more.
template <int NB>
using SmallOff = std::conditional_t<8ULL * (kMaxStateElems / (NB * NB)) <= UINT_MAX, unsigned, size_t>;

template <int NB>
constexpr SmallOff<NB> small_offset(int k) {
    return SmallOff<NB>(8) * static_cast<SmallOff<NB>>(k);
}
