// Decoding a matrix in the device layout back to fp32 with the kernels' own loaders (units.h): the check that the
// layout and the field extraction give the format's values (moe_dequantize).
#include <hip/hip_runtime.h>

#include "aux.h"
#include "iq3s_grid.h"
#include "repack.h"
#include "units.h"

namespace c0ven {

__device__ __constant__ static const uint32_t kGridAux[512] = {C0VEN_IQ3S_GRID_VALUES};

// Grid: one work-group of 64 (a wave) per tile; lane l writes row rt * 64 + l, all its units. The values are
// formed as ggml's dequantize_row_* forms them: Q8_0 d q; Q4_K (d sc) q - (dmin m); IQ3_S (d (1 + 2 s)) (sign grid);
// IQ3_XXS and IQ2_S with the grid the caller's codebooks hold.
__global__ void __launch_bounds__(64) moe_dequant(const uint8_t *mat, uint32_t type, uint32_t rows, uint32_t k,
                                                  const uint8_t *codebooks, float *out) {
  __shared__ uint32_t grid[2048];
  if (type == QT_IQ3_S) {
    for (uint32_t i = threadIdx.x; i < 512; i += 64) grid[i] = kGridAux[i];
  } else if (type == QT_IQ3_XXS || type == QT_IQ2_S) {
    const uint32_t *src = (const uint32_t *)(codebooks + (type == QT_IQ2_S ? QGRID_IQ2S : QGRID_IQ3XXS));
    for (uint32_t i = threadIdx.x; i < (type == QT_IQ2_S ? 2048u : 256u); i += 64) grid[i] = src[i];
  }
  __syncthreads();
  const uint32_t U = units_of(k), rt = blockIdx.x, lane = threadIdx.x, nl = kTileRows * U;
  const uint32_t row = rt * kTileRows + lane;
  const uint8_t *tile = mat + (uint64_t)rt * tile_bytes(type, U);
  const bool live = row < rows;
  for (uint32_t u = 0; u < U; u++) {
  const uint32_t idx = pair_idx(lane, u), nv = min(kUnit, k - u * kUnit);  // nv: the unit's values (partial last)
  float *o = out + (uint64_t)row * k + u * kUnit;
  if (q8_family(type)) {  // a code and its 32-value block's scale: d q, d kvalues[nibble], d (q - 1)
    UnitQ8_0 w;
    if (type == QT_IQ4_NL)
      static_cast<UnitIQ4_NL &>(w).load(tile, idx, nl);
    else if (type == QT_Q2_0)
      static_cast<UnitQ2_0 &>(w).load(tile, idx, nl);
    else
      w.load(tile, idx, nl);
    if (live)
      for (uint32_t i = 0; i < nv; i++) o[i] = __fmul_rn(w.d[i / 32], (float)(int8_t)(w.q[i / 4] >> (8 * (i % 4))));
  } else if (type == QT_Q4_K) {
    UnitQ4_K w;
    w.load(tile, idx, nl);
    if (live)
      for (int wd = 0; wd < 32; wd++)
        for (int i = 0; i < 4; i++) {
          const int c = wd / 8, v = 64 * c + 4 * (wd % 8) + i;
          const float dl = __fmul_rn(w.d, (float)w.sc[2 * c]), ml = __fmul_rn(w.dmin, (float)w.mn[2 * c]);
          const float dh = __fmul_rn(w.d, (float)w.sc[2 * c + 1]), mh = __fmul_rn(w.dmin, (float)w.mn[2 * c + 1]);
          o[v] = __fsub_rn(__fmul_rn(dl, (float)((w.lo[wd] >> (8 * i)) & 0xff)), ml);
          o[v + 32] = __fsub_rn(__fmul_rn(dh, (float)((w.hi[wd] >> (8 * i)) & 0xff)), mh);
        }
  } else if (type == QT_Q5_K) {  // (d sc) q - (dmin m), q 0..31
    UnitQ5_K w;
    w.load(tile, idx, nl);
    if (live)
      for (int wd = 0; wd < 32; wd++)
        for (int i = 0; i < 4; i++) {
          const int c = wd / 8, v = 64 * c + 4 * (wd % 8) + i;
          const float dl = __fmul_rn(w.d, (float)w.sc[2 * c]), ml = __fmul_rn(w.dmin, (float)w.mn[2 * c]);
          const float dh = __fmul_rn(w.d, (float)w.sc[2 * c + 1]), mh = __fmul_rn(w.dmin, (float)w.mn[2 * c + 1]);
          o[v] = __fsub_rn(__fmul_rn(dl, (float)((w.lo[wd] >> (8 * i)) & 0xff)), ml);
          o[v + 32] = __fsub_rn(__fmul_rn(dh, (float)((w.hi[wd] >> (8 * i)) & 0xff)), mh);
        }
  } else if (type == QT_Q6_K) {  // (d sc) (q - 32)
    UnitQ6_K w;
    w.load(tile, idx, nl);
    if (live)
      for (int i = 0; i < 256; i++)
        o[i] = __fmul_rn(__fmul_rn(w.d, (float)w.sc[i / 16]), (float)(int8_t)(w.w[i / 4] >> (8 * (i % 4))));
  } else if (type == QT_IQ4_XS) {  // (d (ls - 32)) kvalues[nibble]
    UnitIQ4_XS w;
    w.load(tile, idx, nl);
    if (live)
      for (int i = 0; i < 256; i++)
        o[i] = __fmul_rn(__fmul_rn(w.d, (float)w.ls[i / 32]), (float)(int8_t)(w.q[i / 4] >> (8 * (i % 4))));
  } else if (type == QT_IQ3_XXS) {  // (d (0.5 + s)) 0.5, times the signed grid value
    UnitIQ3_XXS w;
    w.load(tile, idx, nl, grid);
    if (live)
      for (int i = 0; i < 256; i++) {
        const float db = __fmul_rn(__fmul_rn(w.d, 0.5f + (float)((w.ls[i / 32] - 1) / 2)), 0.5f);
        o[i] = __fmul_rn(db, (float)(int8_t)(w.w[i / 4] >> (8 * (i % 4))));
      }
  } else if (type == QT_IQ2_S) {  // (d (0.5 + s)) 0.25 for each half sub-block, times the signed grid value
    UnitIQ2_S w;
    w.load(tile, idx, nl, grid);
    if (live)
      for (int i = 0; i < 256; i++) {
        const float db = __fmul_rn(__fmul_rn(w.d, 0.5f + (float)((w.ls[i / 16] - 1) / 2)), 0.25f);
        o[i] = __fmul_rn(db, (float)(int8_t)(w.w[i / 4] >> (8 * (i % 4))));
      }
  } else {
    UnitIQ3_S w;
    w.load(tile, idx, nl, grid);
    if (live)
      for (int i = 0; i < 256; i++) {
        const float db = __fmul_rn(w.d, (float)w.ls[i / 32]);
        o[i] = __fmul_rn(db, (float)(int8_t)(w.w[i / 4] >> (8 * (i % 4))));
      }
  }
  }
}

// File layout to device layout (repack.h's pieces), a row tile of one matrix a work-group: thread e takes piece e / (64 U) of
// pair e % (64 U), so that a wave's stores are one run of a field. The reads go through L2 (a row tile's file bytes are at most a
// few hundred KB, each line read by its unit's pieces). What bounds a call is the upload of the same
// bytes: 4 tokens' borrowed experts of 2560 x 640 (52 MB, IQ3_XXS and IQ4_NL) take 1.86 ms, 7.30 where the host repacked them.
__global__ void __launch_bounds__(256) moe_repack(const RepackExpert *experts, RepackShape s) {
  const uint32_t m = blockIdx.y, rt = blockIdx.x, type = s.type[m], k = s.cols[m];
  if (rt * kTileRows >= s.rows[m]) return;
  const RepackExpert &ex = experts[blockIdx.z];
  const uint32_t U = units_of(k), nl = kTileRows * U, bb = quant_block_bytes(type), bv = quant_block_values(type);
  const uint32_t nb = k / bv, ub = kUnit / bv;  // blocks a row, blocks a unit
  const uint8_t *src = ex.src[m];
  const uint32_t b0 = m == 2 && ex.down0 ? ex.down0 : nb;  // blocks a row in the first region
  uint8_t *tile = ex.dst + s.off[m] + (uint64_t)rt * tile_bytes(type, U);
  for (uint32_t e = threadIdx.x; e < nl * repack_pieces(type); e += 256) {
    const uint32_t idx = e % nl, u = idx / kTileRows;
    const uint64_t row = rt * kTileRows + idx % kTileRows;
    const RepackPiece p = repack_piece(type, e / nl);
    const uint32_t blk = u * ub + p.blk;
    const uint8_t *b = src + (blk < b0 ? (row * b0 + blk) * bb : ((uint64_t)s.rows[m] * b0 + row * (nb - b0) + (blk - b0)) * bb) + p.off;
    uint8_t *d = tile + (uint64_t)p.field * nl + ((uint64_t)p.piece * nl + idx) * p.stride + p.sub;
    const bool live = blk < nb;
    // (The file's blocks are 2-byte aligned, the fields' pieces are aligned to their size.)
    const auto move = [&](auto v) {
      if (live) __builtin_memcpy(&v, b, sizeof v);
      *(decltype(v) *)d = v;
    };
    if (p.bytes == 16)
      move(uint4{0, 0, 0, 0});
    else if (p.bytes == 8)
      move(uint2{0, 0});
    else if (p.bytes == 4)
      move(0u);
    else
      move((uint16_t)0);
  }
}

}  // namespace c0ven
