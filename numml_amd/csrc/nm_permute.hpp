// Values between row-major and column-major order: see nm_permute.hip.
#pragma once

#include "nm_common.hpp"

namespace nm {

struct PermutePlan {
    int32_t *run;
    uint16_t *local, *from;
};

// Carves the plan out of `base` (nullptr: size query only); returns bytes.
inline size_t permute_layout(int64_t nnz, void *base, PermutePlan *p) {
    const size_t wide = ((size_t)nnz * 4 + 255) & ~size_t(255), narrow = ((size_t)nnz * 2 + 255) & ~size_t(255);
    char *b = (char *)base;
    if (p) *p = PermutePlan{(int32_t *)b, (uint16_t *)(b + wide), (uint16_t *)(b + wide + narrow)};
    return wide + 2 * narrow;
}

// `rows` and `columns` hold nnz values in row-major and in column-major order; `staged` is work memory for as many
// (it may be where neither input nor result is).
template <typename T> int to_columns(const PermutePlan &p, int64_t nnz, const T *rows, T *staged, T *columns, hipStream_t s);
template <typename T> int to_rows(const PermutePlan &p, int64_t nnz, const T *columns, T *staged, T *rows, hipStream_t s);

}  // namespace nm
