#pragma once

#include <stdint.h>

namespace c0ven {

__global__ void moe_dequant(const uint8_t *mat, uint32_t type, uint32_t rows, uint32_t k, const uint8_t *codebooks,
                            float *out);

// An expert's matrices in the file's layout (device memory: gate, up, down) and where its device layout goes. down0: the blocks
// of a down row's first part where down is two regions (part 0 of every row, then part 1 of every row); 0: whole rows.
struct RepackExpert {
  const uint8_t *src[3];
  uint8_t *dst;
  uint32_t down0, pad;
};
struct RepackShape {
  uint32_t type[3], rows[3], cols[3];  // rows multiples of 64
  uint64_t off[3];                     // the matrices' offsets from dst
};
// Grid: (row tiles of the tallest matrix, 3, experts) work-groups of 256.
__global__ void moe_repack(const RepackExpert *experts, RepackShape s);

}  // namespace c0ven
