// The repack of a matrix from the file's layout (ggml blocks, row-major) into the device layout (layout.h): which bytes go
// where, for the device's kernel (moe_repack) and the host's form below.
#pragma once

#include <cstring>
#include <vector>

#include "layout.h"

namespace c0ven {

// A run of a unit's bytes: bytes (2, 4, 8 or 16) at off of the unit's block blk go to sub of the piece'th stride-byte piece of
// the field based at field (layout.h), or zeros when the row has no such block.
struct RepackPiece {
  uint32_t field, piece, stride, sub, bytes, blk, off;
};
C0VEN_HD uint32_t repack_pieces(uint32_t type) {
  switch (type) {
    case QT_Q8_0: return 24;
    case QT_IQ4_NL: return 16;
    case QT_Q2_0: return 8;
    case QT_Q4_K: return 12;
    case QT_IQ3_S: return 10;
    case QT_IQ3_XXS: return 7;
    case QT_IQ2_S: return 7;
    case QT_IQ4_XS: return 9;
    case QT_Q5_K: return 14;
    default: return 14;  // QT_Q6_K
  }
}
C0VEN_HD RepackPiece repack_piece(uint32_t type, uint32_t j) {
  // Piece j of a field of 256-value blocks: n pieces of size bytes from off on.
  const auto at = [](uint32_t field, uint32_t p, uint32_t size, uint32_t off) { return RepackPiece{field, p, size, 0, size, 0, off + p * size}; };
  switch (type) {
    case QT_Q8_0:
      return j < 16 ? RepackPiece{q8_0t::kQs, j, 16, 0, 16, j / 2, 2 + (j % 2) * 16} : RepackPiece{q8_0t::kD, 0, 16, 2 * (j - 16), 2, j - 16, 0};
    case QT_IQ4_NL:
      return j < 8 ? RepackPiece{iq4_nlt::kQs, j, 16, 0, 16, j, 2} : RepackPiece{iq4_nlt::kD, 0, 16, 2 * (j - 8), 2, j - 8, 0};
    case QT_Q2_0:
      return j < 4 ? RepackPiece{q2_0t::kQs, j, 16, 0, 16, j, 2} : RepackPiece{q2_0t::kD, 0, 8, 2 * (j - 4), 2, j - 4, 0};
    case QT_Q4_K: return j < 8 ? at(q4_kt::kQs, j, 16, 16) : j < 11 ? at(q4_kt::kScales, j - 8, 4, 4) : at(q4_kt::kDm, 0, 4, 0);
    case QT_IQ3_S:
      return j < 4 ? at(iq3_st::kQs, j, 16, 2) : j < 6 ? at(iq3_st::kSigns, j - 4, 16, 74) : j < 8 ? at(iq3_st::kQh, j - 6, 4, 66)
             : j < 9 ? at(iq3_st::kScales, 0, 4, 106) : at(iq3_st::kD, 0, 2, 0);
    case QT_IQ3_XXS: return j < 4 ? at(iq3_xxst::kQs, j, 16, 2) : j < 6 ? at(iq3_xxst::kSs, j - 4, 16, 66) : at(iq3_xxst::kD, 0, 2, 0);
    case QT_IQ2_S:
      return j < 2 ? at(iq2_st::kQs, j, 16, 2) : j < 4 ? at(iq2_st::kSigns, j - 2, 16, 34) : j < 5 ? at(iq2_st::kQh, 0, 8, 66)
             : j < 6 ? at(iq2_st::kScales, 0, 8, 74) : at(iq2_st::kD, 0, 2, 0);
    case QT_IQ4_XS: return j < 8 ? at(iq4_xst::kQs, j, 16, 8) : at(iq4_xst::kMeta, 0, 8, 0);
    case QT_Q5_K:
      return j < 8 ? at(q5_kt::kQs, j, 16, 48) : j < 10 ? at(q5_kt::kQh, j - 8, 16, 16) : j < 13 ? at(q5_kt::kScales, j - 10, 4, 4)
             : at(q5_kt::kDm, 0, 4, 0);
    default:  // QT_Q6_K
      return j < 8 ? at(q6_kt::kQl, j, 16, 0) : j < 12 ? at(q6_kt::kQh, j - 8, 16, 128) : j < 13 ? at(q6_kt::kScales, 0, 16, 192)
             : at(q6_kt::kD, 0, 2, 208);
  }
}

// Row r's unit u in the file's layout: the bytes of its blocks (Q8_0: 8 blocks of 34 B; IQ4_NL: 8 of 18 B; Q2_0: 4
// of 18 B; the 256-value types: one block).
inline const uint8_t *file_unit(const uint8_t *m, uint32_t type, uint32_t k, uint32_t r, uint32_t u) {
  const uint64_t row = (uint64_t)k / quant_block_values(type) * quant_block_bytes(type);
  return m + r * row + (uint64_t)u * unit_bytes(type);
}

// One unit's bytes into pair idx of a tile of nl = 64 U pairs.
inline void put_unit(uint8_t *tile, uint32_t type, uint32_t idx, uint32_t nl, const uint8_t *b) {
  const uint32_t bb = quant_block_bytes(type);
  for (uint32_t j = 0; j < repack_pieces(type); j++) {
    const RepackPiece p = repack_piece(type, j);
    std::memcpy(tile + (uint64_t)p.field * nl + ((uint64_t)p.piece * nl + idx) * p.stride + p.sub, b + p.blk * bb + p.off, p.bytes);
  }
}

// rows x k values of type: file layout -> device layout (dst has matrix_bytes(type, rows, k); rows past the last of
// the final tile are zero, which decodes to zero weights). A partial last unit (k % 256, 32-value block types) takes
// its blocks and leaves the rest zero.
inline void repack_matrix(uint32_t type, const uint8_t *src, uint32_t rows, uint32_t k, uint8_t *dst) {
  const uint32_t U = units_of(k), nrt = (rows + kTileRows - 1) / kTileRows, nl = kTileRows * U;
  const uint64_t tb = tile_bytes(type, U);
  const uint32_t bv = quant_block_values(type), bb = quant_block_bytes(type);
  std::vector<uint8_t> part(unit_bytes(type));
  std::memset(dst, 0, matrix_bytes(type, rows, k));
  for (uint32_t rt = 0; rt < nrt; rt++) {
    uint8_t *tile = dst + (uint64_t)rt * tb;
    for (uint32_t l = 0; l < kTileRows && rt * kTileRows + l < rows; l++)
      for (uint32_t u = 0; u < U; u++) {
        const uint8_t *b = file_unit(src, type, k, rt * kTileRows + l, u);
        if ((u + 1) * kUnit > k) {  // the partial last unit: its blocks, then zero blocks
          std::memset(part.data(), 0, part.size());
          std::memcpy(part.data(), b, (uint64_t)(k - u * kUnit) / bv * bb);
          b = part.data();
        }
        put_unit(tile, type, pair_idx(l, u), nl, b);
      }
  }
}

}  // namespace c0ven
