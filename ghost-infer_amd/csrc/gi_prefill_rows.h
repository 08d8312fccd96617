// The packed query rows of a prefill launch, for the kernels and the host: row r of a set of `group` query heads (all of
// one kv head) is token r / group, head r % group of the set.
#ifndef GI_PREFILL_ROWS_H
#define GI_PREFILL_ROWS_H

#include <stdint.h>

#ifdef __HIPCC__
#define GI_ROWS_FN __host__ __device__ inline
#else
#define GI_ROWS_FN inline
#endif

// ceil(2^31 / group) where row / group over n tokens can be taken as a product (gi_row_token), else 0
GI_ROWS_FN uint32_t gi_row_mul(long long n, int group) {
    return n * group * group < 1ll << 31 ? (uint32_t)(((1ll << 31) + group - 1) / group) : 0;
}
// row / group. The product form is exact for row * group < 2^31: 2 row ceil(2^31 / group) exceeds 2^32 row / group by
// less than 2 row, so the quotient's fraction stays below the next integer. (A 32-bit division is some 40
// instructions; four in a row before the first tile's loads cost a short prompt 0.5 us.)
GI_ROWS_FN int gi_row_token(int row, uint32_t mul, int group) {
    return mul ? (int)(((uint64_t)(2u * (uint32_t)row) * mul) >> 32) : row / group;
}

#endif
