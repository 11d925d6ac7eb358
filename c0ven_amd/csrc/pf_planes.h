// Prefill gate/up as two int8 planes: a wave takes 16 rows of gate and of up, a work-group 64 of each against up to 128
// positions of one expert.
//
// What bounds it, and why this form: the VALU. A unit's weights are decoded (grid lookups, signs) once for the positions the
// work-group holds, already multiplied by their blocks' integer scales and split into two int8 planes, isum = f D_hi +-
// D_lo, so that a position tile's integer sum is two chains of v_mfma_i32_16x16x64_i8: no per-block multiply and add
// a result element (32 of 46 VALU instructions a tile and unit in the block-by-block form). 128 positions halve the
// decodes of the experts with many tokens, which under skewed routing hold 95% of the positions; the position tiles past
// an expert's count are neither loaded nor run. Gate's products come before up's, so that one matrix's planes
// are live at a time (three waves a SIMD).
// Measured against the block-by-block kernels at their 64-position tiles (one launch, top 10 of 512 experts, Zipf): IQ2_S
// 2560 x 640 at 4096 tokens 1331 -> 502 us, IQ3_XXS at 301 tokens 183 -> 106, IQ3_S 2048 x 512 at 2048 tokens 320 -> 209,
// Q4_K 178 -> 166 and at 37 tokens 81 -> 74; a whole forward of IQ4_XS 2048 x 512 at 2048 tokens 748 -> 500. An earlier form that decoded into LDS for 256 positions and took the activations
// straight into registers measured 717, 150, 277 and 309 us: its activation reads were what bounded it.
#pragma once

#include <type_traits>

#include "device_math.h"
#include "layout.h"
#include "mfma_q4k.h"
#include "units.h"

namespace c0ven {
namespace {

typedef short s16x2_t __attribute__((ext_vector_type(2)));

// A 16-row tile's matrix operands of one unit: the lane's A row l % 16, bytes 8 g .. 8 g + 7 of each block (g = l / 16) times
// the block's scale, in two planes of the x64 MFMA's order (step c: blocks 2 c, 2 c + 1), and the row's scale.
struct PlaneA {
  v4i_t lo[4], hi[4];
  float d;  // the A row's scale
};
// Q4_K's: also the minima (f16, the x16 MFMA's operand) and their scale.
struct PlaneAMin : PlaneA {
  float dmin;
  long mn;
};

// Four signed codes (bytes of w) times the scale kk (both halves) as digits p = 64 hi + lo, lo in [0, 63], hi = floor.
__device__ __forceinline__ void plane_digits(uint32_t w, s16x2_t kk, int &hi, int &lo) {
  const s16x2_t v = __builtin_bit_cast(s16x2_t, w);
  const s16x2_t e = (s16x2_t)((v << 8) >> 8) * kk, o = (s16x2_t)(v >> 8) * kk;
  const uint32_t he = __builtin_bit_cast(uint32_t, (s16x2_t)(e >> 6)), ho = __builtin_bit_cast(uint32_t, (s16x2_t)(o >> 6));
  hi = (int)__builtin_amdgcn_perm(ho, he, 0x06020400u);
  lo = (int)(__builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, o), __builtin_bit_cast(uint32_t, e), 0x06020400u) & 0x3f3f3f3fu);
}

// The codebook types' digit tables in LDS, after the coded grid: for scale nibble s and level v (of the codebook's at most
// eight byte values, IQ2_S four), p = v (1 + 2 s) as 64 H - L with H = p / 64 + 1 and L in 1..64, both bytes never
// zero: 16 bytes a scale, H of eight levels then L of them (IQ2_S: four levels, then the negated digits).
constexpr uint32_t kPlaneDigits = 2048;  // words from the grid's start

// Where the wave's 16-row tile lies: the matrix's 64-row tile as the resource's base, the lane's offsets from its row.
struct PlaneAt {
  __amdgpu_buffer_rsrc_t r;
  uint32_t nl, rr;  // pairs a tile; the tile's first row within it
};

template <uint32_t kType>
struct PlaneRaw;

template <>
struct PlaneRaw<QT_IQ3_S> {
  uint32_t qs[8], sg[8], qh[2], sc, dh;
  __device__ __forceinline__ void load(const PlaneAt &t, uint32_t u, uint32_t lane) {
    const uint32_t g = lane / 16, pu = u * kTileRows, la = t.rr + lane % 16, nl = t.nl;
#pragma unroll
    for (uint32_t ib = 0; ib < 8; ib++)
      qs[ib] = __builtin_amdgcn_raw_buffer_load_b32(t.r, la * 16 + 4 * (g / 2) + 8 * (ib % 2), ((ib / 2) * nl + pu) * 16, 0);
#pragma unroll
    for (uint32_t p = 0; p < 2; p++) {
      const auto v = __builtin_amdgcn_raw_buffer_load_b128(t.r, la * 16, iq3_st::kSigns * nl + (p * nl + pu) * 16, 0);
      sg[4 * p] = v[0], sg[4 * p + 1] = v[1], sg[4 * p + 2] = v[2], sg[4 * p + 3] = v[3];
      qh[p] = __builtin_amdgcn_raw_buffer_load_b32(t.r, la * 4, iq3_st::kQh * nl + (p * nl + pu) * 4, 0);
    }
    sc = __builtin_amdgcn_raw_buffer_load_b32(t.r, la * 4, iq3_st::kScales * nl + pu * 4, 0);
    dh = __builtin_amdgcn_raw_buffer_load_b16(t.r, la * 2, iq3_st::kD * nl + pu * 2, 0);
  }
  // (kNeg: isum() gives the sum negated, one multiply-add, and the term is subtracted.)
  // ls = 1 + 2 s as 8 h - l, h = s / 4 + 1 in 1..4 and l = 7 - 2 (s % 4) in 1..7: the grid's magnitudes (at most 15) times
  // either fit a byte and are never zero, so a word's signs apply without carries.
  __device__ __forceinline__ void decode(PlaneA &a, uint32_t lane, const uint32_t *grid) const {
    const uint32_t g = lane / 16;
#pragma unroll
    for (uint32_t ib = 0; ib < 8; ib++) {
      const uint32_t s = (sc >> (4 * ib)) & 15u;
      const uint32_t kh = ((s >> 2) + 1u) * 0x00010001u, kl = (7u - 2u * (s & 3u)) * 0x00010001u;
#pragma unroll
      for (uint32_t j = 0; j < 2; j++) {
        const uint32_t byte = (qs[ib] >> (8 * (2 * (g % 2) + j))) & 0xffu;
        const uint32_t hb = (qh[ib / 4] >> (8 * (ib % 4) + 2 * g + j)) & 1u;
        const uint32_t gv = grid[byte | (hb << 8)];
        const uint32_t x = sign_bits((sg[ib] >> (4 * (2 * g + j))) & 15u), m = sign_mask(x);
        a.lo[ib / 2][2 * (ib % 2) + j] = (int)((mul_bytes(gv, kl) ^ m) + x);
        a.hi[ib / 2][2 * (ib % 2) + j] = (int)((mul_bytes(gv, kh) ^ m) + x);
      }
    }
    a.d = h2f((uint16_t)dh);
  }
  static constexpr bool kNeg = true;
  static __device__ __forceinline__ int isum(int hi, int lo) { return __mul24(hi, -8) + lo; }
  static constexpr float kFactor = 1.0f;
};

template <>
struct PlaneRaw<QT_IQ3_XXS> {
  uint32_t qs[8], ss[8], dh;
  __device__ __forceinline__ void load(const PlaneAt &t, uint32_t u, uint32_t lane) {
    const uint32_t g = lane / 16, pu = u * kTileRows, la = t.rr + lane % 16, nl = t.nl;
#pragma unroll
    for (uint32_t ib = 0; ib < 8; ib++)
      qs[ib] = __builtin_amdgcn_raw_buffer_load_b32(t.r, la * 16 + 4 * (g / 2) + 8 * (ib % 2), ((ib / 2) * nl + pu) * 16, 0);
#pragma unroll
    for (uint32_t p = 0; p < 2; p++) {
      const auto v = __builtin_amdgcn_raw_buffer_load_b128(t.r, la * 16, iq3_xxst::kSs * nl + (p * nl + pu) * 16, 0);
      ss[4 * p] = v[0], ss[4 * p + 1] = v[1], ss[4 * p + 2] = v[2], ss[4 * p + 3] = v[3];
    }
    dh = __builtin_amdgcn_raw_buffer_load_b16(t.r, la * 2, iq3_xxst::kD * nl + pu * 2, 0);
  }
  // The grid (coded) gives each value's level, the scale's digit table (8 levels a plane) its digits: one byte permute a
  // plane and four values. The digits are never zero, so a word's signs apply without carries.
  __device__ __forceinline__ void decode(PlaneA &a, uint32_t lane, const uint32_t *grid) const {
    const uint32_t g = lane / 16;
    const uint4 *digits = (const uint4 *)(grid + kPlaneDigits);
#pragma unroll
    for (uint32_t ib = 0; ib < 8; ib++) {
      const uint4 t = digits[ss[ib] >> 28];
      const uint32_t s7 = (ss[ib] >> (7 * g)) & 127u, sb = s7 | ((uint32_t)(__popc(s7) & 1) << 7);
#pragma unroll
      for (uint32_t j = 0; j < 2; j++) {
        const uint32_t code = grid[(qs[ib] >> (8 * (2 * (g % 2) + j))) & 0xffu];
        const uint32_t x = sign_bits((sb >> (4 * j)) & 15u), m = sign_mask(x);
        a.hi[ib / 2][2 * (ib % 2) + j] = (int)((__builtin_amdgcn_perm(t.y, t.x, code) ^ m) + x);
        a.lo[ib / 2][2 * (ib % 2) + j] = (int)((__builtin_amdgcn_perm(t.w, t.z, code) ^ m) + x);
      }
    }
    a.d = h2f((uint16_t)dh);
  }
  static constexpr bool kNeg = true;
  static __device__ __forceinline__ int isum(int hi, int lo) { return __mul24(hi, -64) + lo; }
  static constexpr float kFactor = 0.25f;
};

template <>
struct PlaneRaw<QT_IQ2_S> {
  uint32_t qs[8], sg[8], qh[2], sc[2], dh;
  __device__ __forceinline__ void load(const PlaneAt &t, uint32_t u, uint32_t lane) {
    const uint32_t pu = u * kTileRows, la = t.rr + lane % 16, nl = t.nl;
#pragma unroll
    for (uint32_t p = 0; p < 2; p++) {
      const auto v = __builtin_amdgcn_raw_buffer_load_b128(t.r, la * 16, iq2_st::kQs * nl + (p * nl + pu) * 16, 0);
      const auto w = __builtin_amdgcn_raw_buffer_load_b128(t.r, la * 16, iq2_st::kSigns * nl + (p * nl + pu) * 16, 0);
      qs[4 * p] = v[0], qs[4 * p + 1] = v[1], qs[4 * p + 2] = v[2], qs[4 * p + 3] = v[3];
      sg[4 * p] = w[0], sg[4 * p + 1] = w[1], sg[4 * p + 2] = w[2], sg[4 * p + 3] = w[3];
    }
    const auto h = __builtin_amdgcn_raw_buffer_load_b64(t.r, la * 8, iq2_st::kQh * nl + pu * 8, 0);
    const auto c = __builtin_amdgcn_raw_buffer_load_b64(t.r, la * 8, iq2_st::kScales * nl + pu * 8, 0);
    qh[0] = h[0], qh[1] = h[1], sc[0] = c[0], sc[1] = c[1];
    dh = __builtin_amdgcn_raw_buffer_load_b16(t.r, la * 2, iq2_st::kD * nl + pu * 2, 0);
  }
  // As IQ3_XXS, with at most four levels: a value's sign joins its level in the permute's selector (levels 4-7 the negated
  // digits).
  __device__ __forceinline__ void decode(PlaneA &a, uint32_t lane, const uint32_t *grid) const {
    const uint32_t g = lane / 16;
    const uint4 *digits = (const uint4 *)(grid + kPlaneDigits);
#pragma unroll
    for (uint32_t ib = 0; ib < 8; ib++) {
      const uint4 t = digits[(sc[ib / 4] >> (8 * (ib % 4) + 4 * (g / 2))) & 15u];  // the lane's half sub-block
      const uint32_t ix = ((qs[ib] >> (8 * g)) & 0xffu) | (((qh[ib / 4] >> (8 * (ib % 4) + 2 * g)) & 3u) << 8);
      const uint2 code = *(const uint2 *)(grid + 2 * ix);
      const uint32_t sb = (sg[ib] >> (8 * g)) & 0xffu;
#pragma unroll
      for (uint32_t j = 0; j < 2; j++) {  // 0x00810204: sign_bits' spread, two bits up
        const uint32_t sel = (j ? code.y : code.x) | ((((sb >> (4 * j)) & 15u) * 0x00810204u) & 0x04040404u);
        a.hi[ib / 2][2 * (ib % 2) + j] = (int)__builtin_amdgcn_perm(t.y, t.x, sel);
        a.lo[ib / 2][2 * (ib % 2) + j] = (int)__builtin_amdgcn_perm(t.w, t.z, sel);
      }
    }
    a.d = h2f((uint16_t)dh);
  }
  static constexpr bool kNeg = true;
  static __device__ __forceinline__ int isum(int hi, int lo) { return __mul24(hi, -64) + lo; }
  static constexpr float kFactor = 0.125f;
};

template <>
struct PlaneRaw<QT_IQ4_XS> {
  uint32_t qs[16], meta[2];
  __device__ __forceinline__ void load(const PlaneAt &t, uint32_t u, uint32_t lane) {
    const uint32_t g = lane / 16, pu = u * kTileRows, la = t.rr + lane % 16, nl = t.nl;
#pragma unroll
    for (uint32_t ib = 0; ib < 8; ib++) {
      const auto q = __builtin_amdgcn_raw_buffer_load_b64(t.r, la * 16 + 8 * (g % 2), iq4_xst::kQs * nl + (ib * nl + pu) * 16, 0);
      qs[2 * ib] = q[0], qs[2 * ib + 1] = q[1];
    }
    const auto m = __builtin_amdgcn_raw_buffer_load_b64(t.r, la * 8, iq4_xst::kMeta * nl + pu * 8, 0);
    meta[0] = m[0], meta[1] = m[1];
  }
  __device__ __forceinline__ void decode(PlaneA &a, uint32_t lane, const uint32_t *) const {
    const uint32_t sh = 4 * (lane / 32);
#pragma unroll
    for (uint32_t ib = 0; ib < 8; ib++) {
      const int ls = (int)(((meta[1] >> (4 * ib)) & 15u) | (((meta[0] >> (16 + 2 * ib)) & 3u) << 4)) - 32;
      const s16x2_t kk = s16x2_t{(short)ls, (short)ls};
#pragma unroll
      for (uint32_t j = 0; j < 2; j++) {
        int h, l;
        plane_digits(iq4nl_lookup((qs[2 * ib + j] >> sh) & 0x0f0f0f0fu), kk, h, l);
        a.lo[ib / 2][2 * (ib % 2) + j] = l, a.hi[ib / 2][2 * (ib % 2) + j] = h;
      }
    }
    a.d = h2f((uint16_t)meta[0]);
  }
  static constexpr bool kNeg = false;
  static __device__ __forceinline__ int isum(int hi, int lo) { return 64 * hi + lo; }
  static constexpr float kFactor = 1.0f;
};

template <>
struct PlaneRaw<QT_Q4_K> {
  uint32_t qs[8], sc[3], dm;
  __device__ __forceinline__ void load(const PlaneAt &t, uint32_t u, uint32_t lane) {
    const uint32_t g = lane / 16, pu = u * kTileRows, la = t.rr + lane % 16, nl = t.nl;
#pragma unroll
    for (uint32_t c = 0; c < 4; c++) {
      const auto v = __builtin_amdgcn_raw_buffer_load_b64(t.r, (g / 2) * nl * 16 + la * 16 + 8 * (g % 2), q4_kt::kQs * nl + (2 * c * nl + pu) * 16, 0);
      qs[2 * c] = v[0], qs[2 * c + 1] = v[1];
    }
#pragma unroll
    for (uint32_t i = 0; i < 3; i++)
      sc[i] = __builtin_amdgcn_raw_buffer_load_b32(t.r, la * 4, q4_kt::kScales * nl + (i * nl + pu) * 4, 0);
    dm = __builtin_amdgcn_raw_buffer_load_b32(t.r, la * 4, q4_kt::kDm * nl + pu * 4, 0);
  }
  // Q4kA::decode's planes (mfma_q4k.h), with the row's own scales.
  __device__ __forceinline__ void decode(PlaneAMin &a, uint32_t lane, const uint32_t *) const {
    Q4kRaw r;
#pragma unroll
    for (uint32_t c = 0; c < 4; c++) r.qs[c] = make_uint2(qs[2 * c], qs[2 * c + 1]);
#pragma unroll
    for (uint32_t i = 0; i < 3; i++) r.sc[i] = sc[i];
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) r.dm[i] = dm;
    Q4kA q;
    q.decode<true>(r, lane);
#pragma unroll
    for (uint32_t c = 0; c < 4; c++) a.lo[c] = q.lo[c], a.hi[c] = q.hi[c];
    a.mn = q.mn, a.d = q.d[0], a.dmin = q.dmin[0];
  }
  static constexpr bool kNeg = false;
  static __device__ __forceinline__ int isum(int hi, int lo) { return 8 * hi + lo; }
  static constexpr float kFactor = 1.0f;
};

__device__ __forceinline__ float plane_dmin(const PlaneA &) { return 0.0f; }
__device__ __forceinline__ float plane_dmin(const PlaneAMin &a) { return a.dmin; }

// A struct of words as the operands of an empty volatile asm with a memory clobber (pin above, for any raw or decoded set).
template <typename T>
__device__ __forceinline__ void pin_words(T &r) {
  static_assert(sizeof(T) % 4 == 0, "words");
  uint32_t *w = reinterpret_cast<uint32_t *>(&r);
#pragma unroll
  for (uint32_t i = 0; i < sizeof(T) / 4; i++) asm volatile("" : "+v"(w[i]));
  asm volatile("" ::: "memory");
}

// One position tile's (scale_products): element i is row 4 (l / 16) + i, position l % 16 (d and a of lanes 0-15 used; the other
// three of the instruction's products are 0 x 0).
__device__ __forceinline__ v4f_t scale_products1(float d, float a, uint32_t lane) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(lane < 16 ? d : 0.0f, lane < 16 ? a : 0.0f, v4f_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
}

// Sixteen (four) bytes a lane from the resource straight to LDS: the wave's 64 pieces in lane order from lds (wave-uniform).
// (Functions: in a kernel's lambda the cast to LDS makes this compiler's host pass drop the kernel's launch stub.)
__device__ __forceinline__ void lds_load16(__amdgpu_buffer_rsrc_t r, void *lds, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void *)lds, 16, voff, soff, 0, 0);
}
__device__ __forceinline__ void lds_load4(__amdgpu_buffer_rsrc_t r, void *lds, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void *)lds, 4, voff, soff, 0, 0);
}

// Positions a work-group takes (its spans). Where decoding a unit is cheap beside its products (Q4_K: 100 VALU instructions a
// matrix; IQ2_S), 64 in two activation buffers; where it is dear (IQ3_S, IQ3_XXS, IQ4_XS: 230-290) 128 in one, which halves
// the decodes of experts with many positions. A constant of the type, a compromise over the token counts. Q4_K's launch, 64
// and 128: 74 and 85 us at 37 tokens, 166 and 170 at 2048. Whole forwards, 2560 x 640 over 512 experts, 64 and 128:
//   tokens             37 even    1000 even   1000 Zipf   4096 even    4096 Zipf
//   IQ3_XXS            353 361    656 681     484 470     1490 1343    1310 1241
//   IQ3_S              365 372    685 715     495 480     1558 1417    1359 1304
//   IQ4_XS             364 370    692 704     491 472     1577 1398    1377 1282
//   IQ2_S              311 319    583 606     438 435     1387 1281    1195 1178
template <uint32_t kType>
constexpr uint32_t plane_pos() { return kType == QT_Q4_K || kType == QT_IQ2_S ? 64u : 128u; }

typedef float v16f_t __attribute__((ext_vector_type(16)));
// d[16-row tile] x a[4 position tiles], each product rounded once, to a subnormal too, as __fmul_rn rounds it, but for the sign
// of a zero: the instruction adds to +0, and -0 becomes +0. No output shows it: each product times an integer joins a sum that
// starts from +0, and there either zero leaves the sum as it is. Lane l's d is row l % 16's, its a position
// 16 (l / 16) + l % 16's; element 4 b + i of the result is row 4 (l / 16) + i, position 16 b + l % 16. One matrix
// instruction for sixteen VALU ones.
__device__ __forceinline__ v16f_t scale_products(float d, float a) {
  v16f_t z;
#pragma unroll
  for (int i = 0; i < 16; i++) z[i] = 0.0f;
  return __builtin_amdgcn_mfma_f32_16x16x1f32(d, a, z, 0, 0, 0);
}

template <uint32_t kType>
__global__ void __launch_bounds__(kPfWG) __attribute__((amdgpu_waves_per_eu(3))) pf_gate_up_planes(PfGemm g) {
  constexpr uint32_t kPos = plane_pos<kType>(), kBufs = kPos == 64 ? 2 : 1, kPt = kPos / 16;
  constexpr bool kMin = kType == QT_Q4_K;
  // A position's 256 code bytes, its sixteen 16-byte chunks XORed with the position (mod 16), so that sixteen positions'
  // chunk q fall in distinct banks; the positions' unit scales and (Q4_K) split block sums (kActSplitH) apart.
  __shared__ __align__(16) uint8_t abuf[kBufs][kPos * 256];
  __shared__ __align__(16) float adt[kBufs][kPos];
  __shared__ __align__(16) uint8_t sums[kBufs][kMin ? kPos * 32 : 16];
  __shared__ uint32_t arow[kPos];
  __shared__ uint64_t tab[32];
  constexpr bool kCoded = kType == QT_IQ3_XXS || kType == QT_IQ2_S;
  __shared__ __align__(16) uint32_t grid[kType == QT_IQ3_S ? 512 : kCoded ? kPlaneDigits + 64 : 4];
  const uint32_t U = g.U, nrb = g.row_blocks;
  uint32_t sp, rb;
  if (!span_item(blockIdx.x, nrb, *g.nspans, &sp, &rb)) return;
  const MoeTile tl = g.spans[sp];
  const uint32_t start = tl.start, count = tl.count, npt = (count + 15) / 16;
  const uint32_t tid = threadIdx.x, wv = (uint32_t)__builtin_amdgcn_readfirstlane(tid >> 6);
  if (tid < 32) tab[tid] = kExp2Tab[tid];
  if constexpr (kType == QT_IQ3_S)
    for (uint32_t i = tid; i < 512; i += kPfWG) grid[i] = kIq3sGridPf[i];
  if constexpr (kCoded) {
    constexpr uint32_t kOff = kType == QT_IQ2_S ? QGRID_IQ2S : QGRID_IQ3XXS, kLevels = kType == QT_IQ2_S ? 4 : 8;
    const uint32_t *src = (const uint32_t *)(g.coded + kOff);
    for (uint32_t i = tid; i < (kType == QT_IQ2_S ? 2048u : 256u); i += kPfWG) grid[i] = src[i];
    if (tid < 128) {  // digit byte tid % 8 of scale tid / 8
      const uint8_t *levels = g.coded + QGRID_IQ3S + (kType == QT_IQ2_S ? 0 : 8);
      const uint32_t s = tid / 8, v = tid % 8, p = levels[v % kLevels] * (1u + 2u * s), H = p / 64 + 1;
      const bool neg = v >= kLevels;
      uint8_t *t = (uint8_t *)(grid + kPlaneDigits + 4 * s) + v;
      t[0] = (uint8_t)(neg ? 0u - H : H), t[8] = (uint8_t)(neg ? p - 64 * H : 64 * H - p);
    }
  }
  if (tid < kPos) arow[tid] = g.perm[start + min(tid, count - 1)] / g.K * U * kActBytes;  // (past the count: never stored)
  const uint64_t tile = (uint64_t)rb * tile_bytes(kType, U);  // 64 rows of gate and of up: one row tile of each
  const uint8_t *Mg = g.mat + (uint64_t)tl.slot * g.stride + tile;
  const __amdgpu_buffer_rsrc_t act_r = uniform_rsrc(g.act);
  const auto at = [&](uint32_t m) { return PlaneAt{uniform_rsrc(Mg + (m ? g.up_off : 0)), kTileRows * U, 16 * wv}; };
  using Raw = PlaneRaw<kType>;
  Raw raw[2];  // gate's and up's, each loaded a unit ahead
  raw[0].load(at(0), 0, lane_id());
  raw[1].load(at(1), 0, lane_id());
  __syncthreads();
  // Unit u's activations to LDS: round k takes position tile k, wave w its positions 4 w .. + 3, a lane one chunk (the LDS
  // bytes of a load are its lanes' in order, so the XOR is in which chunk a lane asks for); the scales four bytes a lane.
  const auto dma = [&](uint32_t u, uint8_t *buf, float *ads, uint8_t *sms) {
    const uint32_t ln = lane_id(), p4 = 4 * wv + ln / 16, chunk = 16 * ((ln & 15u) ^ p4);
#pragma unroll
    for (uint32_t k = 0; k < kPt; k++) {
      if (k >= npt) continue;
      lds_load16(act_r, buf + (16 * k + 4 * wv) * 256, arow[16 * k + p4] + chunk, u * kActBytes);
    }
    if (wv < kPos / 64 && 64 * wv < count)
      lds_load4(act_r, ads + 64 * wv, arow[64 * wv + ln] + kActScales, u * kActBytes);
    if constexpr (kMin)
      if (wv < kPos / 32 && 32 * wv < count)
        lds_load16(act_r, sms + 1024 * wv, arow[32 * wv + ln / 2] + kActSplitH + 16 * (ln % 2), u * kActBytes);
  };
  float acc[2][kPt][4];
#pragma unroll
  for (uint32_t m = 0; m < 2; m++)
#pragma unroll
    for (uint32_t p = 0; p < kPt; p++)
#pragma unroll
      for (int i = 0; i < 4; i++) acc[m][p][i] = 0.0f;
  using A = std::conditional_t<kMin, PlaneAMin, PlaneA>;
  const auto products = [&](const A &a, float(&s)[kPt][4], const uint8_t *__restrict__ buf, const float *__restrict__ ads,
                            const uint8_t *__restrict__ sms) {
    const uint32_t ln = lane_id(), l16 = ln & 15u, lg = ln >> 4;
    // d and the positions' scales multiplied four position tiles at a time; with minima two, d's in elements 0-7 and
    // dmin's in 8-15 (lanes 32-63 of the operands); with 128 positions' sums held, one (four registers).
    constexpr uint32_t kTiles = kMin ? 2 : kPos == 128 ? 1 : 4;
#pragma unroll
    for (uint32_t q = 0; q < kPt / kTiles; q++) {
      if (kTiles * q >= npt) continue;
      std::conditional_t<kTiles == 1, v4f_t, v16f_t> dd;
      if constexpr (kTiles == 1)
        dd = scale_products1(a.d, ads[16 * q + l16], ln);
      else
        dd = scale_products(kMin && ln >= 32 ? plane_dmin(a) : a.d, ads[16 * kTiles * q + ln % (16 * kTiles)]);
#pragma unroll
      for (uint32_t j = 0; j < kTiles; j++) {
        const uint32_t p = kTiles * q + j;
        if (p >= npt) continue;
        v4i_t dl = {0, 0, 0, 0}, dh = {0, 0, 0, 0};
#pragma unroll
        for (uint32_t c = 0; c < 4; c++) {
          const v4i_t b = *(const v4i_t *)(buf + (16 * p + l16) * 256 + 16 * ((4 * c + lg) ^ l16));
          dl = __builtin_amdgcn_mfma_i32_16x16x64_i8(a.lo[c], b, dl, 0, 0, 0);
          dh = __builtin_amdgcn_mfma_i32_16x16x64_i8(a.hi[c], b, dh, 0, 0, 0);
        }
        if constexpr (kMin) {
          const v4h_t bm = *(const v4h_t *)(sms + (16 * p + l16) * 32 + 8 * lg);
          const v4f_t im = __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(v4h_t, a.mn), bm, v4f_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const float pm = __fmul_rn(dd[8 + 4 * j + i], im[i]);
            s[p][i] = __fadd_rn(s[p][i], __builtin_fmaf(dd[4 * j + i], (float)Raw::isum(dh[i], dl[i]), -pm));
          }
        } else {
#pragma unroll
          for (int i = 0; i < 4; i++) {
            // The type's factor, a power of two, last, as UnitIQ3_XXS::term and UnitIQ2_S::term have it: in d it would take a
            // product of the scales below 2^-126 and round it there. (Under 1% of a forward, the product being one more.)
            float t = __fmul_rn(dd[4 * j + i], (float)Raw::isum(dh[i], dl[i]));
            if constexpr (Raw::kFactor != 1.0f) t = __fmul_rn(Raw::kFactor, t);
            s[p][i] = Raw::kNeg ? __fsub_rn(s[p][i], t) : __fadd_rn(s[p][i], t);
          }
        }
      }
    }
  };
  // Two buffers, up to the wait: unit u's decode and gate products, and unit u + 1's activations on their way. buf (read)
  // and nbuf (filled) are restrict pointers, so that the reads of buf do not wait for the loads into nbuf; the wait and the
  // barrier are outside.
  const auto gate_pass = [&](A &a, uint32_t un, const uint8_t *__restrict__ buf, const float *__restrict__ ads,
                             const uint8_t *__restrict__ sms, uint8_t *__restrict__ nbuf, float *__restrict__ nads,
                             uint8_t *__restrict__ nsms) {
    dma(un, nbuf, nads, nsms);  // (every wave has passed the barrier after unit u - 1's products of that buffer)
    pin_words(raw[0]);
    raw[0].decode(a, lane_id(), grid);
    pin_words(a);
    raw[0].load(at(0), un, lane_id());
    products(a, acc[0], buf, ads, sms);
    pin_words(raw[1]);
    raw[1].decode(a, lane_id(), grid);
    pin_words(a);
  };
  const auto unit = [&](uint32_t u) {
    const uint32_t un = min(u + 1, U - 1), b = u % kBufs, n = (u + 1) % kBufs;
    A a;
    if constexpr (kBufs == 2) {
      gate_pass(a, un, abuf[b], adt[b], sums[b], abuf[n], adt[n], sums[n]);
      __builtin_amdgcn_s_waitcnt(vm_wait(0));  // this wave's loads of unit u + 1's activations (and gate's bytes) ...
      raw[1].load(at(1), un, lane_id());
      products(a, acc[1], abuf[b], adt[b], sums[b]);
      unit_barrier();  // ... and every wave's; buffer u % 2 is free
    } else {
      pin_words(raw[0]);
      raw[0].decode(a, lane_id(), grid);
      pin_words(a);
      __builtin_amdgcn_s_waitcnt(vm_wait(0));  // unit u's activations (this wave's loads) ...
      unit_barrier();                          // ... and every wave's
      raw[0].load(at(0), un, lane_id());
      products(a, acc[0], abuf[0], adt[0], sums[0]);
      pin_words(raw[1]);
      raw[1].decode(a, lane_id(), grid);
      pin_words(a);
      raw[1].load(at(1), un, lane_id());
      products(a, acc[1], abuf[0], adt[0], sums[0]);
      unit_barrier();  // every wave is done with the buffer
      if (u + 1 < U) dma(u + 1, abuf[0], adt[0], sums[0]);
    }
  };
  dma(0, abuf[0], adt[0], sums[0]);
  if constexpr (kBufs == 2) {
    __builtin_amdgcn_s_waitcnt(vm_wait(0));
    unit_barrier();
  }
#pragma unroll 1
  for (uint32_t u = 0; u < U; u++) unit(u);
  // Lane l holds rows 4 (l / 16) + i of positions 16 p + l % 16, gate and up alike.
  const uint32_t ln = lane_id(), l16 = ln & 15u, row0 = 64 * rb + 16 * wv + 4 * (ln >> 4);
#pragma unroll
  for (uint32_t p = 0; p < kPt; p++) {
    const uint32_t m = 16 * p + l16;
    if (m < count) {
      v4f_t h;
#pragma unroll
      for (int i = 0; i < 4; i++) h[i] = swiglu_one(acc[0][p][i], acc[1][p][i], g.limit, tab);
      *(v4f_t *)&g.out[(uint64_t)(start + m) * g.out_ld + row0] = h;
    }
  }
}

}  // namespace
}  // namespace c0ven
