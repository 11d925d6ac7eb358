// Prefill down for the q8_0 family (Q8_0, IQ4_NL, Q2_0): a work-group holds the activations of up to 64 positions of one
// expert in LDS, all of K, and its waves walk 16-row tiles of the weights against them, each on its own.
//
// What bounds it, and why this form: the VALU. Each 32-value block's term is rounded on its own, (d_w d_a) dot, then the
// tree: four instructions a result element and block where a matrix instruction gives the dot. Here the scale products
// come from a matrix instruction too (scale_products: four blocks' outer products at once), which leaves three; the
// blocks past K in the last unit (F 640: half of it) are skipped, their terms being zeros; and no barrier or activation load
// follows the first, so a wave's next weights load while its products run. The former kernel took 64 rows
// a work-group through K unit by unit, and its start and end outweighed its two or three units. IQ4_NL 2560 x 640, one
// launch: 690 -> 419 us at 4096 tokens, 108 -> 66 at 301.
#pragma once

#include <type_traits>

#include "device_math.h"
#include "layout.h"
#include "mfma_q4k.h"
#include "units.h"

namespace c0ven {
namespace {

// One lane's bytes of a 16-row tile and unit: its row l % 16's eight codes 8 g .. 8 g + 7 of each block, and the row's
// scales of blocks g and 4 + g (the operands of scale_products), f16.
template <uint32_t kType>
struct DownRaw;

template <>
struct DownRaw<QT_Q8_0> {
  uint32_t w[16], d[2];
  __device__ __forceinline__ void load(const PlaneAt &t, uint32_t u, uint32_t lane) {
    const uint32_t g = lane / 16, pu = u * kTileRows, la = t.rr + lane % 16, nl = t.nl;
#pragma unroll
    for (uint32_t j = 0; j < 8; j++) {
      const auto q = __builtin_amdgcn_raw_buffer_load_b64(t.r, (g / 2) * nl * 16 + la * 16 + 8 * (g % 2), q8_0t::kQs * nl + (2 * j * nl + pu) * 16, 0);
      w[2 * j] = q[0], w[2 * j + 1] = q[1];
    }
#pragma unroll
    for (uint32_t h = 0; h < 2; h++) d[h] = __builtin_amdgcn_raw_buffer_load_b16(t.r, la * 16 + 2 * g, q8_0t::kD * nl + pu * 16 + 8 * h, 0);
  }
  __device__ __forceinline__ void codes(long q[8], uint32_t) const {
#pragma unroll
    for (uint32_t j = 0; j < 8; j++) q[j] = pack2(w[2 * j], w[2 * j + 1]);
  }
};

template <>
struct DownRaw<QT_IQ4_NL> {
  uint32_t w[16], d[2];
  __device__ __forceinline__ void load(const PlaneAt &t, uint32_t u, uint32_t lane) {
    const uint32_t g = lane / 16, pu = u * kTileRows, la = t.rr + lane % 16, nl = t.nl;
#pragma unroll
    for (uint32_t j = 0; j < 8; j++) {
      const auto q = __builtin_amdgcn_raw_buffer_load_b64(t.r, la * 16 + 8 * (g % 2), iq4_nlt::kQs * nl + (j * nl + pu) * 16, 0);
      w[2 * j] = q[0], w[2 * j + 1] = q[1];
    }
#pragma unroll
    for (uint32_t h = 0; h < 2; h++) d[h] = __builtin_amdgcn_raw_buffer_load_b16(t.r, la * 16 + 2 * g, iq4_nlt::kD * nl + pu * 16 + 8 * h, 0);
  }
  __device__ __forceinline__ void codes(long q[8], uint32_t lane) const {
    const uint32_t sh = 4 * (lane / 32);
#pragma unroll
    for (uint32_t j = 0; j < 8; j++)
      q[j] = pack2(iq4nl_lookup((w[2 * j] >> sh) & 0x0f0f0f0fu), iq4nl_lookup((w[2 * j + 1] >> sh) & 0x0f0f0f0fu));
  }
};

template <>
struct DownRaw<QT_Q2_0> {
  uint32_t w[8], d[2];
  __device__ __forceinline__ void load(const PlaneAt &t, uint32_t u, uint32_t lane) {
    const uint32_t g = lane / 16, pu = u * kTileRows, la = t.rr + lane % 16, nl = t.nl;
#pragma unroll
    for (uint32_t j = 0; j < 8; j++)
      w[j] = __builtin_amdgcn_raw_buffer_load_b16(t.r, la * 16 + 2 * g, q2_0t::kQs * nl + ((j / 2) * nl + pu) * 16 + 8 * (j % 2), 0);
#pragma unroll
    for (uint32_t h = 0; h < 2; h++) d[h] = __builtin_amdgcn_raw_buffer_load_b16(t.r, la * 8 + 2 * (g / 2), q2_0t::kD * nl + pu * 8 + 4 * h, 0);
  }
  __device__ __forceinline__ void codes(long q[8], uint32_t) const {
#pragma unroll
    for (uint32_t j = 0; j < 8; j++) q[j] = pack2(q2_spread(w[j] & 0xffu), q2_spread((w[j] >> 8) & 0xffu));
  }
};

constexpr uint32_t kDownPos = 64;  // positions a work-group takes
// LDS bytes of the positions' codes and scales: whole units at 256 bytes a position, a last half unit at 128 (a last
// quarter or three quarters at 256), 32 bytes of scales a unit.
constexpr uint32_t down_lds(uint32_t F) {
  return kDownPos * (F / 256 * 256 + (F % 256 == 0 ? 0 : F % 256 == 128 ? 128 : 256) + (F + 255) / 256 * 32);
}
constexpr uint32_t kDownStatic = 4 * kDownPos;  // the positions' offsets, beside them
// The most a work-group takes, so that two fit a CU: F to 896 (Q8_0 2048 x 896: 5% of a forward less than with pf_gemm16 at
// 2048 tokens); larger F, which were not measured, keep pf_gemm16.
constexpr uint32_t kDownMaxLds = 65 * 1024;
// 64-row groups a work-group walks: fewer where the launch would have less than two rounds of the device's work-groups (three a
// CU to F 640, two above). nrb (n_embd / 64) is a multiple of 8.
constexpr uint32_t kDownGroups = 1536;
__host__ __device__ constexpr uint32_t down_walk(uint32_t nspans, uint32_t nrb) {
  uint32_t W = 8;
  while (W > 1 && (nspans + 7) / 8 * 8 * (nrb / W) < kDownGroups) W /= 2;
  return W;
}

template <uint32_t kType>
__global__ void __launch_bounds__(kPfWG) __attribute__((amdgpu_waves_per_eu(3))) pf_down_q8(PfGemm g) {
  extern __shared__ __align__(16) uint8_t lds[];
  __shared__ uint32_t arow[kDownStatic / 4];
  const uint32_t U = g.U, nsp = *g.nspans, W = down_walk(nsp, g.row_blocks);
  uint32_t sp, rb;
  if (!span_item(blockIdx.x, g.row_blocks / W, nsp, &sp, &rb)) return;
  const MoeTile tl = g.spans[sp];
  const uint32_t start = tl.start, count = tl.count, npt = (count + 15) / 16;
  const uint32_t tid = threadIdx.x, wv = (uint32_t)__builtin_amdgcn_readfirstlane(tid >> 6);
  if (tid < kDownPos) arow[tid] = (start + min(tid, count - 1)) * U * kActBytes;  // (past the count: never stored)
  const __amdgpu_buffer_rsrc_t act_r = uniform_rsrc(g.act);
  const uint8_t *mat = g.mat + (uint64_t)tl.slot * g.stride;
  const uint32_t tb = (uint32_t)tile_bytes(kType, U), S = W * U;  // steps: unit s % U of the wave's tile of group s / U
  const bool half_last = g.K % 256 == 128;                          // (g.K: values of a row)
  const uint32_t wide = half_last ? U - 1 : U;                      // units at 256 bytes a position
  float *const sc = (float *)(lds + kDownPos * (256 * wide + (half_last ? 128 : 0)));  // [unit][position][block]
  using Raw = DownRaw<kType>;
  Raw raw;
  const auto load = [&](uint32_t s) {
    raw.load(PlaneAt{uniform_rsrc(mat + (uint64_t)(rb * W + s / U) * tb), kTileRows * U, 16 * wv}, s % U, lane_id());
  };
  load(0);
  __syncthreads();
  // The activations: a position's sixteen 16-byte chunks of a unit XORed with the position (eight with position / 2 in a half
  // unit's 128 bytes), so that sixteen positions' chunk q fall in distinct banks.
  for (uint32_t u = 0; u < U; u++) {
    const uint32_t ln = lane_id();
    if (u < wide) {
#pragma unroll
      for (uint32_t k = 0; k < 4; k++) {
        const uint32_t p = 16 * k + 4 * wv + ln / 16;
        if (k < npt)
          lds_load16(act_r, lds + kDownPos * 256 * u + (16 * k + 4 * wv) * 256, arow[p] + 16 * ((ln & 15u) ^ (p & 15u)), u * kActBytes);
      }
    } else {
#pragma unroll
      for (uint32_t k = 0; k < 2; k++) {
        const uint32_t p = 32 * k + 8 * wv + ln / 8;
        if (2 * k < npt)
          lds_load16(act_r, lds + kDownPos * 256 * u + (32 * k + 8 * wv) * 128, arow[p] + 16 * ((ln & 7u) ^ ((p >> 1) & 7u)), u * kActBytes);
      }
    }
    if (wv < 2 && 32 * wv < count)
      lds_load16(act_r, sc + (u * kDownPos + 32 * wv) * 8, arow[32 * wv + ln / 2] + kActScales + 16 * (ln % 2), u * kActBytes);
  }
  __builtin_amdgcn_s_waitcnt(vm_wait(0));
  unit_barrier();
  float acc[4][4];
#pragma unroll
  for (int p = 0; p < 4; p++)
#pragma unroll
    for (int i = 0; i < 4; i++) acc[p][i] = 0.0f;
#pragma unroll 1
  for (uint32_t s = 0; s < S; s++) {
    const uint32_t u = s % U, nc = min(4u, (g.K - 256 * u) / 64);  // 64-value steps of the unit
    long q[8];
    pin_words(raw);
    raw.codes(q, lane_id());
    float d[2];
#pragma unroll
    for (int h = 0; h < 2; h++) d[h] = h2f((uint16_t)raw.d[h]);
    pin_words(q);
    load(min(s + 1, S - 1));
    const uint32_t ln = lane_id(), l16 = ln & 15u, lg = ln >> 4;
    // (Values, not pointers, over the two row strides: 256 bytes XOR position, or 128 XOR position / 2.)
    const uint32_t rs = u < wide ? 256u : 128u, x = u < wide ? l16 : (l16 >> 1) & 7u;
    const uint8_t *const base = lds + kDownPos * 256 * u + l16 * rs;
#pragma unroll
    for (uint32_t p = 0; p < 4; p++) {
      if (p >= npt) continue;
      const float *const as = sc + (u * kDownPos + 16 * p + l16) * 8 + lg;
      float half[4], s4[4];
      v16f_t dd;
#pragma unroll
      for (uint32_t c = 0; c < 4; c++) {
        if (c >= nc) continue;  // (uniform; the missing blocks' terms are zeros)
        if (c % 2 == 0) dd = scale_products(d[c / 2], as[2 * c]);
        const v4i_t b = *(const v4i_t *)(base + 16 * p * rs + 16 * ((4 * c + lg) ^ x));
        const v4i_t d0 = __builtin_amdgcn_mfma_i32_16x16x32_i8(q[2 * c], __builtin_bit_cast(long, __builtin_shufflevector(b, b, 0, 1)), v4i_t{0, 0, 0, 0}, 0, 0, 0);
        const v4i_t d1 = __builtin_amdgcn_mfma_i32_16x16x32_i8(q[2 * c + 1], __builtin_bit_cast(long, __builtin_shufflevector(b, b, 2, 3)), v4i_t{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const float t = __fadd_rn(__fmul_rn(dd[8 * (c % 2) + i], (float)d0[i]), __fmul_rn(dd[8 * (c % 2) + 4 + i], (float)d1[i]));
          if (c == 0) half[i] = t;
          if (c == 1) half[i] = __fadd_rn(half[i], t);
          if (c == 2) s4[i] = t;
          if (c == 3) s4[i] = __fadd_rn(s4[i], t);
        }
      }
#pragma unroll
      for (int i = 0; i < 4; i++) acc[p][i] = __fadd_rn(acc[p][i], nc > 2 ? __fadd_rn(half[i], s4[i]) : half[i]);
    }
    if (u == U - 1) {  // the row tile's outputs: rows 4 lg .. + 3 of positions 16 p + l16
      uint8_t *const out = (uint8_t *)(g.out + (uint64_t)start * g.out_ld + (rb * W + s / U) * 64 + 16 * wv);
#pragma unroll
      for (uint32_t p = 0; p < 4; p++) {
        const uint32_t m = 16 * p + l16;
        if (m < count) *(v4f_t *)(out + (m * 4 * g.out_ld + 16 * lg)) = v4f_t{acc[p][0], acc[p][1], acc[p][2], acc[p][3]};
#pragma unroll
        for (int i = 0; i < 4; i++) acc[p][i] = 0.0f;
      }
    }
  }
}

}  // namespace
}  // namespace c0ven
