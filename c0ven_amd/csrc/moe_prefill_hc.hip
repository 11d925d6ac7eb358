// The hyper-connection mix before the prefill block and the combine after it (docs/spec/MODEL_LAYER.md 1.1-1.2; the
// reference's prompt path runs p_hc_mix and p_hc_combine around the block, core/models/qwen4exp/prompt.cpp:478-504).
//
// The results are the decode path's, bit for bit (and the oracle's, orc_hc_pre / orc_hc_post): the norms, silu,
// sigmoid and mix steps are the same fp32 operations; the two bf16 products (W_down and W_inject against n, W_up
// against l) are sums of exact products that the decode kernel adds in fp64 in a fixed order and rounds to fp32 once.
// Here they run on the int8 matrix cores: a row's or token's bf16 values become whole numbers of 2^-29 of its largest
// value's power of two, in four signed byte digits, and the digits' products add exactly in 32 bits. A value more than
// 2^22 below the largest loses bits there; where a tile's rows or tokens lose enough of them to leave more than a few sums
// open, it takes the bf16 values on the fp64 matrix cores instead. Either sum is within
// (n_mine + n_ref) 2^-53 sum|p| <= (n_mine + n_ref) 2^-53 ||w||_2 ||x||_2 of the fixed order's (Cauchy-Schwarz on the
// bf16 values; the digits' lost bits add their own term). Where the fp32 rounding of every value in that interval is the same,
// it is the fixed order's rounding; and where the products' bits span fewer than 53 (the least lsb of the row's and of
// the token's values against the Cauchy-Schwarz bound on sum|p|), both sums are exact, whatever their order (ties of
// fp32 rounding are common for W_up's short sums, and this settles them).
// Otherwise the sum is recomputed in the fixed order, from a list, in a kernel of its own:
// W_up's a k-order chain of at most 512 terms, W_down's and W_inject's the decode kernel's 512-value-chunk tree.
#include <hip/hip_runtime.h>

#include "device_math.h"
#include "prefill_hc.h"

namespace c0ven {
namespace {

typedef int v4i_t __attribute__((ext_vector_type(4)));
typedef double v4d_t __attribute__((ext_vector_type(4)));

constexpr uint32_t kHcWG = 256;
constexpr uint32_t kHcStreams4 = 4;
constexpr uint32_t kDiagonals = 2 * kHcDigits - 1;  // the digit products' weights: 256^0 .. 256^6
constexpr uint32_t kGroupK = 128;  // values an fp64 matrix-core chain sums before its sum joins the total

__device__ __forceinline__ uint32_t lane_of() { return threadIdx.x & 63u; }

// The lsb exponent of a bf16 value's bits (2^(e - 134) for exponent field e, 2^-133 for a subnormal); a large value
// for zero, which adds no bits to a sum.
__device__ __forceinline__ int bf16_lsb_of(float v) {
  const uint32_t u = __float_as_uint(v), e = (u >> 23) & 0xffu;
  return (u & 0x7fff0000u) == 0u ? (1 << 20) : (e == 0u ? -133 : (int)e - 134);
}

__device__ __forceinline__ double bf16_lo(uint32_t w) { return (double)__uint_as_float(w << 16); }
__device__ __forceinline__ double bf16_hi(uint32_t w) { return (double)__uint_as_float(w & 0xffff0000u); }

// A double summed over the work-group (256) in a fixed order: each wave by halving exchanges, then the four waves.
__device__ __forceinline__ double wg_sum(double v, double *red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = __dadd_rn(v, __shfl_xor(v, o, 64));
  __syncthreads();
  if (lane_of() == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  const double s = __dadd_rn(__dadd_rn(red[0], red[1]), __dadd_rn(red[2], red[3]));
  __syncthreads();
  return s;
}

__device__ __forceinline__ int wg_min(int v, int *red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, 64));
  __syncthreads();
  if (lane_of() == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  const int m = min(min(red[0], red[1]), min(red[2], red[3]));
  __syncthreads();
  return m;
}

// Token t (one work-group, 256 threads a stream): each stream as RMSNorm(R_s) gamma_s, the decode kernel's hc_norm_item
// arithmetic (each thread's squares in order, then the stream's sum in wg_sum's order; mean rounded to fp32;
// 1 / sqrtf(mean + 1e-6)): the stream's scale into sc
// (pf_hc_mix forms n again from R, the scale and gamma), bf16(n) into nb, and the 2-norm (rounded up), least lsb
// exponent and largest exponent field of bf16(n). Work-group 0 clears the open lists' counts, each its token's sums of
// lost bits. Latency bound (a thread's H / 256 loads, the sum's exchanges): the four streams side by side
// instead of one after another take 23 us at 1000 tokens of H 2560, 39 before.
__global__ void __launch_bounds__(kHcStreams4 * kHcWG) pf_hc_norm(const float *R, const float *gamma, uint32_t H, float *sc,
                                                                  uint16_t *nb, double *nn, int *nlsb, HcGrid n, HcGrid l,
                                                                  uint32_t *cnt) {
  __shared__ double red[kHcStreams4][4];
  __shared__ int redi[2][kHcStreams4 * 4];
  const uint32_t t = blockIdx.x, s = threadIdx.x / kHcWG, i0 = threadIdx.x % kHcWG, wv = threadIdx.x >> 6;
  if (t == 0 && threadIdx.x < 2) cnt[threadIdx.x] = 0u;
  if (threadIdx.x == 0) n.lost[t] = l.lost[t] = 0u;
  // v summed over the stream's 256 threads, as wg_sum.
  const auto stream_sum = [&](double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = __dadd_rn(v, __shfl_xor(v, o, 64));
    __syncthreads();
    if (lane_of() == 0) red[s][wv % 4] = v;
    __syncthreads();
    return __dadd_rn(__dadd_rn(red[s][0], red[s][1]), __dadd_rn(red[s][2], red[s][3]));
  };
  const float *r = R + ((uint64_t)t * kHcStreams4 + s) * H;
  double ss = 0.0;
#pragma unroll 2
  for (uint32_t i = i0; i < H; i += kHcWG) ss = __dadd_rn(ss, (double)__fmul_rn(r[i], r[i]));
  ss = stream_sum(ss);
  const float mean = (float)(ss / (double)H);
  const float scale = __fdiv_rn(1.0f, sqrtf(__fadd_rn(mean, 1e-6f)));
  if (i0 == 0) sc[t * kHcStreams4 + s] = scale;
  uint16_t *ob = nb + ((uint64_t)t * kHcStreams4 + s) * H;
  double sq = 0.0;
  int lsb = 1 << 20, top = 0;
#pragma unroll 2
  for (uint32_t i = i0; i < H; i += kHcWG) {
    const float v = __fmul_rn(__fmul_rn(r[i], scale), gamma[s * H + i]);
    const float bv = round_bf16(v);
    ob[i] = (uint16_t)(__float_as_uint(bv) >> 16);
    const double b = (double)bv;
    sq = __builtin_fma(b, b, sq);
    lsb = min(lsb, bf16_lsb_of(bv));
    top = max(top, (int)((__float_as_uint(bv) >> 23) & 0xffu));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) lsb = min(lsb, __shfl_xor(lsb, o, 64)), top = max(top, __shfl_xor(top, o, 64));
  if (lane_of() == 0) redi[0][wv] = lsb, redi[1][wv] = top;
  (void)stream_sum(sq);
  if (threadIdx.x == 0) {
    double q = 0.0;
    for (uint32_t k = 0; k < kHcStreams4; k++) q = __dadd_rn(q, __dadd_rn(__dadd_rn(red[k][0], red[k][1]), __dadd_rn(red[k][2], red[k][3])));
    for (uint32_t k = 0; k < kHcStreams4 * 4; k++) lsb = min(lsb, redi[0][k]), top = max(top, redi[1][k]);
    nn[t] = sqrt(q) * (1.0 + 0x1p-30), nlsb[t] = lsb, n.exp[t] = top;
  }
}

// Four values' digits (X as bytes after the carry trick below) as four words of one digit each.
__device__ __forceinline__ void transpose4(const uint32_t y[4], uint32_t d[kHcDigits]) {
  const uint32_t a0 = __builtin_amdgcn_perm(y[1], y[0], 0x05010400u), a1 = __builtin_amdgcn_perm(y[1], y[0], 0x07030602u);
  const uint32_t b0 = __builtin_amdgcn_perm(y[3], y[2], 0x05010400u), b1 = __builtin_amdgcn_perm(y[3], y[2], 0x07030602u);
  d[0] = __builtin_amdgcn_perm(b0, a0, 0x05040100u), d[1] = __builtin_amdgcn_perm(b0, a0, 0x07060302u);
  d[2] = __builtin_amdgcn_perm(b1, a1, 0x05040100u), d[3] = __builtin_amdgcn_perm(b1, a1, 0x07060302u);
}

// The digits of bf16 rows (A0's first M0, then A1's; K values each, a multiple of 8) whose largest exponent fields are
// g.exp: value (-1)^s m 2^(e - 134) is the whole number X = (-1)^s m 2^(e - exp + 22), toward zero (|X| < 2^30), and
// X = sum of d_i 256^i with d_i in -128 .. 127. The rows are laid out as the matrix cores take them: 16-row tile, 64
// values, digit, then lane 16 q + r's 16 values 16 q .. of row r; rows and values past the ends are zeros. After the
// digits, a byte a tile's 64 values: whether any lowest digit is not zero. A wave a tile's
// 64 values: it reads 128 bytes of each row and writes 4 KB whole. g.lost[row] receives the lost bits' sum, in
// 2^-16 of X's units, each rounded up (below 2^31 for K to 32768).
__global__ void __launch_bounds__(kHcWG) pf_hc_digits(const uint16_t *A0, uint32_t M0, const uint16_t *A1, uint32_t M,
                                                      uint32_t K, HcGrid g, uint8_t *out) {
  const uint32_t nch = (K + 63) / 64, ch = blockIdx.y * (kHcWG / 64) + (threadIdx.x >> 6);
  if (ch >= nch) return;
  const uint32_t lane = lane_of(), row = 16 * blockIdx.x + lane % 16, k0 = 64 * ch + 16 * (lane / 16);
  uint32_t v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  int top = 0;
  if (row < M) {
    const uint16_t *src = (row < M0 ? A0 + (uint64_t)row * K : A1 + (uint64_t)(row - M0) * K) + k0;
    top = g.exp[row];
    if (k0 < K) {
      const uint4 q = *(const uint4 *)src;
      v[0] = q.x, v[1] = q.y, v[2] = q.z, v[3] = q.w;
    }
    if (k0 + 8 < K) {
      const uint4 q = *(const uint4 *)(src + 8);
      v[4] = q.x, v[5] = q.y, v[6] = q.z, v[7] = q.w;
    }
  }
  uint32_t lost = 0, d[4][kHcDigits];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    uint32_t y[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const uint32_t u = (v[2 * q + i / 2] >> (16 * (i & 1))) & 0xffffu, e = (u >> 7) & 0xffu;
      const uint32_t m = (u & 0x7fu) | (e ? 0x80u : 0u);
      const int sh = (int)max(e, 1u) - max(top, 1) + 22;  // (at most 22)
      const uint32_t down = (uint32_t)min(max(-sh, 0), 31);
      const uint32_t x = sh >= 0 ? m << sh : m >> down;
      const uint32_t rest = sh < 0 ? m - (x << down) : 0u;  // (of 2^down)
      lost += down <= 16 ? rest << (16 - down) : (rest + (1u << (down - 16)) - 1u) >> (down - 16);
      const uint32_t X = (u & 0x8000u) ? 0u - x : x;
      y[i] = (X + 0x00808080u) ^ 0x00808080u;  // each lower byte's digit as a signed byte, its carry in the next
    }
    transpose4(y, d[q]);
  }
  if (lost) atomicAdd(g.lost + row, lost);
  uint8_t *o = out + ((uint64_t)blockIdx.x * nch + ch) * (kHcDigits * 1024) + lane * 16;
#pragma unroll
  for (uint32_t i = 0; i < kHcDigits; i++) *(uint4 *)(o + 1024 * i) = make_uint4(d[0][i], d[1][i], d[2][i], d[3][i]);
  const bool low = __any((d[0][0] | d[1][0] | d[2][0] | d[3][0]) != 0u) != 0;
  if (lane == 0) out[(uint64_t)gridDim.x * nch * (kHcDigits * 1024) + (uint64_t)blockIdx.x * nch + ch] = low ? 1 : 0;
}

// A row's or token's part of the bound: 2-norm (rounded up), the same in units of its values' least lsb (infinite when bits
// were lost), the sum of its lost bits, and a power of two above its largest value. wide: its digits are not used.
struct Side {
  double norm, units, lost, top;
};
// What side_of reads of n consecutive rows or tokens from i on, all in flight together (left to the compiler, a side's lsb is
// read only once its lost bits are known to be none, and each side is waited for before the next one's loads: the up
// product 69 us instead of 61 at 1000 tokens of H 2560, lr 320). n 4: i a multiple of 4, the arrays 16-byte aligned.
template <uint32_t n>
struct SideRaw {
  uint32_t norm[n][2], lsb[n], exp[n], lost[n];
  __device__ __forceinline__ void load(const double *nm, const int *l, const HcGrid &g, uint32_t i) {
    if constexpr (n == 4) {
      *(uint4 *)&norm[0] = *(const uint4 *)(nm + i), *(uint4 *)&norm[2] = *(const uint4 *)(nm + i + 2);
      *(uint4 *)lsb = *(const uint4 *)(l + i), *(uint4 *)exp = *(const uint4 *)(g.exp + i), *(uint4 *)lost = *(const uint4 *)(g.lost + i);
    } else {
      *(uint2 *)&norm[0] = *(const uint2 *)(nm + i), lsb[0] = l[i], exp[0] = g.exp[i], lost[0] = g.lost[i];
    }
  }
  __device__ __forceinline__ void arrived() {
#pragma unroll
    for (uint32_t k = 0; k < n; k++)
      asm volatile("" : "+v"(norm[k][0]), "+v"(norm[k][1]), "+v"(lsb[k]), "+v"(exp[k]), "+v"(lost[k]));
  }
  __device__ __forceinline__ Side side(uint32_t k, bool wide) const {
    const uint32_t m = wide ? 0u : lost[k];
    const int e = max((int)exp[k], 1);
    const double r = __hiloint2double((int)norm[k][1], (int)norm[k][0]);
    return {r, m ? __builtin_inf() : ldexp(r, -(int)lsb[k]), ldexp((double)m, e - 172), ldexp(1.0, e - 126)};
  }
};
__device__ __forceinline__ Side side_of(const double *norm, const int *lsb, const HcGrid &g, uint32_t i, bool wide) {
  SideRaw<1> r;
  r.load(norm, lsb, g, i);
  r.arrived();
  return r.side(0, wide);
}

// Whether the sum v of a row's and a token's bf16 products rounds to fp32 as the fixed order's does. Exact: no bits lost,
// every product is a multiple of the two least lsbs' product and sum|p| <= r.norm t.norm is below 2^53 of it, so
// every partial sum of any order is representable and both give the exact sum (the product of r.units and t.units rounds
// by 2^-53, which the norms' rounding up covers). Otherwise bounded: the two fp64 values
// are within bnd, and every value in [v - bnd, v + bnd] rounds to the same fp32.
__device__ __forceinline__ bool certain(double v, const Side &r, const Side &t, double bound_k) {
  if (r.units * t.units < 0x1p53) return true;
  const double bnd = bound_k * (r.norm * t.norm) + (r.lost * t.top + r.top * t.lost);
  const float f = (float)v;
  return (float)(v - bnd) == f && (float)(v + bnd) == f;
}

// Whether a wave's 32 rows and 32 tokens take wide_products: their lost bits would leave more than about 3% of the sums
// open. A sum is about r.norm t.norm / sqrt(K), half its fp32 unit 2^-25 of that; limit is 2^-30 / sqrt(K), against the
// lost term over the norms. A normal row of 10240 loses bits in one value of 0.8% of the rows, 4 to 8 times less than the limit.
__device__ __forceinline__ bool tile_is_wide(const double *rn, const double *tn, const HcGrid &gr, const HcGrid &gt,
                                             uint32_t M, uint32_t N, uint32_t m0, uint32_t n0, double limit) {
  const uint32_t lane = lane_of(), f32 = lane % 32;
  const bool row = lane < 32;  // lanes 0-31 the rows, 32-63 the tokens
  const uint32_t i = row ? min(m0 + f32, M - 1) : min(n0 + f32, N - 1);
  const uint32_t n = (row ? gr.lost : gt.lost)[i];
  if (!__any(n != 0u)) return false;
  const int e = max((row ? gr.exp : gt.exp)[i], 1);
  const double norm = (row ? rn : tn)[i];
  // (Both far inside fp32's range; a zero row has neither part.)
  float lost = norm == 0.0 ? 0.0f : (float)(ldexp((double)n, e - 172) / norm), top = norm == 0.0 ? 0.0f : (float)(ldexp(1.0, e - 126) / norm);
#pragma unroll
  for (int o = 16; o > 0; o >>= 1) lost = fmaxf(lost, __shfl_xor(lost, o, 64)), top = fmaxf(top, __shfl_xor(top, o, 64));
  const float other = __shfl_xor(top, 32, 64);
  return __any((double)lost * other > limit) != 0;
}

// sum of s[i] 256^i, rounded to fp64 once: a part has at most 4096 values, so |s[6]| <= 2^24, |s[5]| <= 2^26, |s[4]| <= 2^27,
// |s[3]| and |s[2]| < 2^28, |s[1]| <= 2^27, |s[0]| <= 2^26, and every step but the last is exact.
__device__ __forceinline__ double diagonals(const int s[kDiagonals]) {
  const double p = __builtin_fma((double)s[6], 256.0, (double)s[5]), q = __builtin_fma((double)s[4], 256.0, (double)s[3]);
  const double r = __builtin_fma((double)s[2], 65536.0, __builtin_fma((double)s[1], 256.0, (double)s[0]));
  return __builtin_fma(__builtin_fma(p, 65536.0, q), 0x1p24, r);
}

// The sums of a wave's 32 rows and 32 tokens over K range kb .. ke from the bf16 values (rows of A0's first M0, then A1's) on
// the fp64 matrix cores. Lane l (g = l / 16) holds values 8 g .. 8 g + 7 of a 32-value step of both operands, step m of the
// matrix instruction its m'th (the order of a sum is free here: the bound covers any); the A operand's lane c takes row
// 4 (c % 4) + c / 4, so that v[i][j][q] is digit_products' element. Each kGroupK values' chain starts from zero and is added
// to the total.
__device__ __forceinline__ void wide_products(const uint16_t *A0, uint32_t M0, const uint16_t *A1, uint32_t M,
                                              const uint16_t *B, uint32_t N, uint32_t K, uint32_t kb, uint32_t ke,
                                              uint32_t m0, uint32_t n0, double (&v)[2][2][4]) {
  const uint32_t lane = lane_of(), g = lane / 16, c16 = lane % 16;
  const uint16_t *ar[2], *br[2];
#pragma unroll
  for (int f = 0; f < 2; f++) {
    const uint32_t row = min(m0 + 16 * f + 4 * (c16 % 4) + c16 / 4, M - 1), tok = min(n0 + 16 * f + c16, N - 1);
    ar[f] = row < M0 ? A0 + (uint64_t)row * K : A1 + (uint64_t)(row - M0) * K;
    br[f] = B + (uint64_t)tok * K;
  }
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int q = 0; q < 4; q++) v[i][j][q] = 0.0;
  for (uint32_t kg = kb; kg < ke; kg += kGroupK) {
    v4d_t acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int j = 0; j < 2; j++) acc[i][j] = v4d_t{0.0, 0.0, 0.0, 0.0};
    const uint32_t kge = min(ke, kg + kGroupK);
    for (uint32_t kc = kg; kc < kge; kc += 32) {
      const uint32_t k = kc + 8 * g;
      const bool ok = k < kge;  // (K is a multiple of 8: a lane's eight values are all in or all out)
      uint32_t a[2][4], b[2][4];
#pragma unroll
      for (int f = 0; f < 2; f++) {
        const uint4 x = ok ? *(const uint4 *)(ar[f] + k) : make_uint4(0u, 0u, 0u, 0u);
        const uint4 y = ok ? *(const uint4 *)(br[f] + k) : make_uint4(0u, 0u, 0u, 0u);
        a[f][0] = x.x, a[f][1] = x.y, a[f][2] = x.z, a[f][3] = x.w;
        b[f][0] = y.x, b[f][1] = y.y, b[f][2] = y.z, b[f][3] = y.w;
      }
#pragma unroll
      for (int m = 0; m < 8; m++) {
        double ad[2], bd[2];
#pragma unroll
        for (int f = 0; f < 2; f++) {
          ad[f] = m % 2 ? bf16_hi(a[f][m / 2]) : bf16_lo(a[f][m / 2]);
          bd[f] = m % 2 ? bf16_hi(b[f][m / 2]) : bf16_lo(b[f][m / 2]);
        }
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
          for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ad[i], bd[j], acc[i][j], 0, 0, 0);
      }
    }
    // (The f64 form's result layout: element q of lane l is A lane 4 q + l / 16's row, B lane l % 16's token.)
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int q = 0; q < 4; q++) v[i][j][q] = __dadd_rn(v[i][j][q], acc[i][j][q]);
  }
}

// The same from the digits of part `split` (cs of nch 64-value chunks): each sum exact in 32-bit diagonals, rounded once.
// v[i][j][q]: row m0 + 16 i + 4 g + q, token n0 + 16 j + c16 (g = lane / 16, c16 = lane % 16); i1, j1: 0 where the second
// tile lies wholly past the rows or tokens (the first's operands are repeated and its sums dropped).
__device__ __forceinline__ void digit_products(const uint8_t *A, uint32_t M, const uint8_t *B, uint32_t N, uint32_t nch,
                                               uint32_t split, uint32_t cs, uint32_t m0, uint32_t n0, uint32_t i1,
                                               uint32_t j1, const HcGrid &gr, const HcGrid &gt, double (&v)[2][2][4]) {
  const uint32_t lane = lane_of(), g = lane / 16, c16 = lane % 16;
  const uint64_t tile = (uint64_t)nch * (kHcDigits * 1024), first = (uint64_t)split * cs * (kHcDigits * 1024) + lane * 16;
  const uint8_t *ap[2] = {A + m0 / 16 * tile + first, A + (m0 / 16 + i1) * tile + first};
  const uint8_t *bp[2] = {B + n0 / 16 * tile + first, B + (n0 / 16 + j1) * tile + first};
  v4i_t acc[2][2][kDiagonals];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (uint32_t d = 0; d < kDiagonals; d++) acc[i][j][d] = v4i_t{0, 0, 0, 0};
  v4i_t a[2][kHcDigits], b[2][kHcDigits];
  // Bit c: chunk c's lowest digits are not all zero (a part has at most 64 chunks). The bytes are read beside the first
  // chunk's other digits.
  uint64_t al[2], bl[2];
  const auto low_digits = [&](uint32_t c, v4i_t (&to)[2][kHcDigits], const uint8_t *const (&from)[2], const uint64_t (&low)[2]) {
#pragma unroll
    for (int f = 0; f < 2; f++)
      if ((low[f] >> c) & 1) to[f][0] = *(const v4i_t *)(from[f] + c * kHcDigits * 1024);
  };
  const auto load = [&](uint32_t c, v4i_t (&to)[2][kHcDigits], const uint8_t *const (&from)[2]) {
#pragma unroll
    for (int f = 0; f < 2; f++)
#pragma unroll
      for (uint32_t d = 1; d < kHcDigits; d++) to[f][d] = *(const v4i_t *)(from[f] + (c * kHcDigits + d) * 1024);
  };
  {
    const uint8_t *af = A + ((M + 15) / 16) * tile + split * cs, *bf = B + ((N + 15) / 16) * tile + split * cs;
    const uint32_t c = min(lane, cs - 1);
    const uint8_t f0 = af[(uint64_t)(m0 / 16) * nch + c], f1 = af[(uint64_t)(m0 / 16 + i1) * nch + c];
    const uint8_t f2 = bf[(uint64_t)(n0 / 16) * nch + c], f3 = bf[(uint64_t)(n0 / 16 + j1) * nch + c];
    load(0, a, ap), load(0, b, bp);
    al[0] = __ballot(f0), al[1] = __ballot(f1), bl[0] = __ballot(f2), bl[1] = __ballot(f3);
  }
#pragma unroll
  for (int f = 0; f < 2; f++) a[f][0] = b[f][0] = v4i_t{0, 0, 0, 0};
  low_digits(0, a, ap, al), low_digits(0, b, bp, bl);
  for (uint32_t c = 0; c < cs; c++) {
    v4i_t na[2][kHcDigits], nb[2][kHcDigits];
#pragma unroll
    for (int f = 0; f < 2; f++) na[f][0] = nb[f][0] = v4i_t{0, 0, 0, 0};
    const uint32_t next = min(c + 1, cs - 1);
    low_digits(next, na, ap, al), low_digits(next, nb, bp, bl);
    load(next, na, ap), load(next, nb, bp);
#pragma unroll
    for (uint32_t da = 1; da < kHcDigits; da++)
#pragma unroll
      for (uint32_t db = 1; db < kHcDigits; db++)
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
          for (int j = 0; j < 2; j++)
            acc[i][j][da + db] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[i][da], b[j][db], acc[i][j][da + db], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 2; i++)
      if ((al[i] >> c) & 1)
#pragma unroll
        for (uint32_t db = 0; db < kHcDigits; db++)
#pragma unroll
          for (int j = 0; j < 2; j++)
            acc[i][j][db] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[i][0], b[j][db], acc[i][j][db], 0, 0, 0);  // (b[j][0] may be zeros)
#pragma unroll
    for (int j = 0; j < 2; j++)
      if ((bl[j] >> c) & 1)
#pragma unroll
        for (uint32_t da = 1; da < kHcDigits; da++)
#pragma unroll
          for (int i = 0; i < 2; i++)
            acc[i][j][da] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[i][da], b[j][0], acc[i][j][da], 0, 0, 0);
#pragma unroll
    for (int f = 0; f < 2; f++)
#pragma unroll
      for (uint32_t d = 0; d < kHcDigits; d++) a[f][d] = na[f][d], b[f][d] = nb[f][d];
  }
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const uint32_t row = min(m0 + 16 * i + 4 * g, M - 4);  // (M is a multiple of 4)
    int er[4];
#pragma unroll
    for (int q = 0; q < 4; q++) er[q] = max(gr.exp[row + q], 1);
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const int et = max(gt.exp[min(n0 + 16 * j + c16, N - 1)], 1) - 312;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        int s[kDiagonals];
#pragma unroll
        for (uint32_t d = 0; d < kDiagonals; d++) s[d] = acc[i][j][d][q];
        v[i][j][q] = ldexp(diagonals(s), er[q] + et);
      }
    }
  }
}

// C = A B^T over the digits of the rows (M of them, A) and of the tokens (N, B), nch 64-value chunks in blockIdx.x % nsplit
// parts of cs. A work-group takes 64 rows x 64 tokens, wave w rows 32 (w & 1) .. and tokens 32 (w >> 1) .., as 2 x 2 tiles
// of 16 x 16, whose digit products of one weight share an accumulator (a part has at most 4096 values: 2^28).
// The lowest digit is nonzero only for values 2^15 and more below their row's largest (about one in 5000 of a normal
// row's): a fragment whose lowest digits are all zero skips their load and products, which leaves 9 of 16 in most chunks.
// The operands come straight from L2 in the matrix cores' order, the next chunk's while this one's products run.
// A part keeps to one XCD (nsplit 8), so that each L2 reads one part of both operands; without parts the XCD
// takes every eighth row tile.
// A wave whose rows or tokens lost too many bits (tile_is_wide) takes their bf16 values (A0's first M0 rows, then A1's; Bb; K a
// row) on the fp64 matrix cores. With the digits for those too, nearly every sum of such a token was left open, and the
// fixed-order kernels took most of the step: 1000 tokens of H 2560 with two channels 3000 times the others, the whole
// step 2.0 ms (3.7 with W_down eight times as large), 0.70 (0.80) with this, 0.96 with all products in fp64; 0.58 on normal
// values either way.
// kUp: one part; the sums are certified here (rows' and tokens' sides) and written as fp32 to out32 (N x M), an open one's
// (token, row) to the list open (pf_hc_up_fix writes it). Otherwise the part's fp64 sums go to part (nsplit x N x M), and
// whether a 32 x 32 tile was wide to wide_map (token tiles x row tiles).
// T 1000, H 2560, lr 320 (2 x 3.3 G products): down 49 us (5 more with the lowest digits always loaded) and up 61, where the
// fp64 matrix cores took 162 and 141.
template <bool kUp>
__global__ void __launch_bounds__(kHcWG, 2) pf_hc_gemm(const uint8_t *A, uint32_t M, const uint8_t *B, uint32_t N,
                                                       const uint16_t *A0, uint32_t M0, const uint16_t *A1,
                                                       const uint16_t *Bb, uint32_t K, uint32_t nch, uint32_t nsplit,
                                                       double *part, float *out32, uint8_t *wide_map, const double *rn,
                                                       const double *tn, const int *rl, const int *tl, HcGrid gr,
                                                       HcGrid gt, double limit, double bound_digits, double bound_wide,
                                                       uint32_t *open, uint32_t *cnt) {
  const uint32_t nmt = (M + 63) / 64, split = blockIdx.x % nsplit, item = blockIdx.x / nsplit;
  const uint32_t mt = item % nmt, nt = item / nmt, cs = nch / nsplit;
  const uint32_t lane = lane_of(), w = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane / 16, c16 = lane % 16;
  const uint32_t m0 = 64 * mt + 32 * (w & 1), n0 = 64 * nt + 32 * (w >> 1);
  // 16 x 16 tiles wholly past the rows or the tokens are skipped: a wave with none returns (the kernel has no barrier),
  // the others repeat their first tile's operands and drop its sums.
  if (m0 >= M || n0 >= N) return;
  const uint32_t i1 = m0 + 16 < M ? 1u : 0u, j1 = n0 + 16 < N ? 1u : 0u;
  const bool wide = tile_is_wide(rn, tn, gr, gt, M, N, m0, n0, limit);
  if (!kUp && split == 0 && lane == 0) wide_map[n0 / 32 * ((M + 31) / 32) + m0 / 32] = wide ? 1 : 0;
  const double bound_k = wide ? bound_wide : bound_digits;
  double v[2][2][4];
  if (wide)
    wide_products(A0, M0, A1, M, Bb, N, K, 64 * split * cs, min(K, 64 * (split + 1) * cs), m0, n0, v);
  else
    digit_products(A, M, B, N, nch, split, cs, m0, n0, i1, j1, gr, gt, v);
  SideRaw<4> rr[2];
  SideRaw<1> tr[2];
  if constexpr (kUp) {
#pragma unroll
    for (uint32_t f = 0; f < 2; f++)
      rr[f].load(rn, rl, gr, min(m0 + 16 * f + 4 * g, M - 4)), tr[f].load(tn, tl, gt, min(n0 + 16 * f + c16, N - 1));
#pragma unroll
    for (uint32_t f = 0; f < 2; f++) rr[f].arrived(), tr[f].arrived();
  }
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const uint32_t row = m0 + 16 * i + 4 * g;
    if (row >= M) continue;
    Side rs[4];
    if constexpr (kUp)
#pragma unroll
      for (int q = 0; q < 4; q++) rs[q] = rr[i].side(q, wide);
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const uint32_t tok = n0 + 16 * j + c16;
      if (tok >= N) continue;
      if constexpr (kUp) {
        const Side ts = tr[j].side(0, wide);
        *(float4 *)(out32 + (uint64_t)tok * M + row) =
            make_float4((float)v[i][j][0], (float)v[i][j][1], (float)v[i][j][2], (float)v[i][j][3]);
#pragma unroll
        for (int q = 0; q < 4; q++)
          if (!certain(v[i][j][q], rs[q], ts, bound_k)) {  // open: pf_hc_up_fix writes it
            const uint32_t at = atomicAdd(cnt, 1u);
            open[2 * at] = tok, open[2 * at + 1] = row + q;
          }
      } else {
        double *o = part + ((uint64_t)split * N + tok) * M + row;
        *(double2 *)o = make_double2(v[i][j][0], v[i][j][1]), *(double2 *)(o + 2) = make_double2(v[i][j][2], v[i][j][3]);
      }
    }
  }
}

// Token t's down sums (rows < lr of W_down, then the 4 of W_inject): the splits added in order, certified against the
// fixed order (certain), rounded to fp32 into raw (T x (lr + 4)); an open one's (t, row) goes to the list (its
// raw entry is written by pf_hc_down_fix). force_open sends all.
__global__ void __launch_bounds__(kHcWG) pf_hc_down_fin(const double *part, uint32_t T, uint32_t M, uint32_t nsplit,
                                                        const double *rn, const double *tn, const int *rl,
                                                        const int *tl, HcGrid gr, HcGrid gt, const uint8_t *wide_map,
                                                        double bound_digits, double bound_wide, bool force_open,
                                                        float *raw, uint32_t *open, uint32_t *cnt) {
  const uint32_t t = blockIdx.x;
  for (uint32_t row = threadIdx.x; row < M; row += kHcWG) {
    double v = 0.0;
    for (uint32_t s = 0; s < nsplit; s++) v = __dadd_rn(v, part[((uint64_t)s * T + t) * M + row]);
    const bool wide = wide_map[t / 32 * ((M + 31) / 32) + row / 32] != 0;
    if (!force_open && certain(v, side_of(rn, rl, gr, row, wide), side_of(tn, tl, gt, t, wide), wide ? bound_wide : bound_digits)) {
      raw[(uint64_t)t * M + row] = (float)v;
    } else {
      const uint32_t at = atomicAdd(cnt, 1u);
      open[2 * at] = t, open[2 * at + 1] = row;
    }
  }
}

// The open down sums in the decode kernel's fixed order (bf16_dot for one row and one token, restated for one wave):
// 512-value chunks c; lane l's eight values 8 l .. 8 l + 7 a fused chain from zero; a lane row r (16 lanes) as
// ((P0 + P7) + (P3 + P4)) + ((P1 + P6) + (P2 + P5)), P_m = a_m + a_(15 - m); slot 4 (c mod 4) + r takes the chunks'
// sums in chunk order; the 16 slots added in order from zero. A work-group an entry, wave q the chunks q, q + 4, ..: what
// bounds it is one entry's chunk chain (K = 10240, 1000 tokens: 9.5 us, one wave an entry 24).
__global__ void __launch_bounds__(kHcWG) pf_hc_down_fix(const uint16_t *w_down, const uint16_t *w_inj, uint32_t lr,
                                                        uint32_t K, const uint16_t *nb, const uint32_t *open,
                                                        const uint32_t *cnt, float *raw) {
  __shared__ double slots[16];  // slot 4 q + r
  const uint32_t lane = lane_of(), r = lane / 16, q = threadIdx.x >> 6, M = lr + kHcStreams4;
  for (uint32_t e = blockIdx.x; e < *cnt; e += gridDim.x) {
    const uint32_t t = open[2 * e], row = open[2 * e + 1];
    const uint16_t *wr = row < lr ? w_down + (uint64_t)row * K : w_inj + (uint64_t)(row - lr) * K;
    const uint16_t *xr = nb + (uint64_t)t * K;
    double slot = 0.0;
    for (uint32_t c = q; c < K / 512; c += 4) {
      const uint32_t k0 = 512 * c + 8 * lane;
      const uint4 wq = *(const uint4 *)(wr + k0), xq = *(const uint4 *)(xr + k0);
      const uint32_t ww[4] = {wq.x, wq.y, wq.z, wq.w}, xw[4] = {xq.x, xq.y, xq.z, xq.w};
      double a = 0.0;
#pragma unroll
      for (int k = 0; k < 8; k++)
        a = __builtin_fma((k & 1) ? bf16_hi(ww[k / 2]) : bf16_lo(ww[k / 2]), (k & 1) ? bf16_hi(xw[k / 2]) : bf16_lo(xw[k / 2]), a);
      const double P = __dadd_rn(a, __shfl_xor(a, 15, 64));  // lanes m < 8 of a row: P_m
      double p[8];
#pragma unroll
      for (int j = 0; j < 8; j++) p[j] = __shfl(P, (int)(16 * r + j), 64);
      const double S = __dadd_rn(__dadd_rn(__dadd_rn(p[0], p[7]), __dadd_rn(p[3], p[4])),
                                 __dadd_rn(__dadd_rn(p[1], p[6]), __dadd_rn(p[2], p[5])));
      slot = c < 4 ? S : __dadd_rn(slot, S);
    }
    if (lane % 16 == 0) slots[4 * q + r] = slot;
    __syncthreads();
    if (threadIdx.x == 0) {
      double s = 0.0;
      for (uint32_t i = 0; i < 16; i++) s = __dadd_rn(s, slots[i]);
      raw[(uint64_t)t * M + row] = (float)s;
    }
    __syncthreads();
  }
}

// The open up sums in the fixed order: a k-order chain over the lr values of W_up's row against bf16(l) of the token,
// one fused step a term from zero. One wave an entry: the wave brings the row and l into its LDS, lane 0 runs the
// chain from there.
__global__ void __launch_bounds__(kHcWG) pf_hc_up_fix(const uint16_t *w_up, uint32_t lr, uint32_t M, const uint16_t *lb,
                                                      const uint32_t *open, const uint32_t *cnt, float *out32) {
  __shared__ __align__(16) float ws[kHcWG / 64][512], xs[kHcWG / 64][512];
  const uint32_t lane = lane_of(), wv = threadIdx.x >> 6, nw = gridDim.x * (kHcWG / 64);
  for (uint32_t e = blockIdx.x * (kHcWG / 64) + wv; e < *cnt; e += nw) {
    const uint32_t t = open[2 * e], row = open[2 * e + 1];
    const uint16_t *wr = w_up + (uint64_t)row * lr;
    const uint16_t *xr = lb + (uint64_t)t * lr;
    for (uint32_t k = lane; k < lr; k += 64) {
      ws[wv][k] = __uint_as_float((uint32_t)wr[k] << 16);
      xs[wv][k] = __uint_as_float((uint32_t)xr[k] << 16);
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_wave_barrier();
    if (lane == 0) {
      double c = 0.0;
      for (uint32_t k = 0; k < lr; k += 4) {
        const float4 w4 = *(const float4 *)&ws[wv][k], x4 = *(const float4 *)&xs[wv][k];
        c = __builtin_fma((double)w4.x, (double)x4.x, c);
        c = __builtin_fma((double)w4.y, (double)x4.y, c);
        c = __builtin_fma((double)w4.z, (double)x4.z, c);
        c = __builtin_fma((double)w4.w, (double)x4.w, c);
      }
      out32[(uint64_t)t * M + row] = (float)c;
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// Token t: l = silu(v / 4) for W_down's rows (the quarter exact; z / (1 + e^-z)) as bf16 bits (the up GEMM's operand),
// the inject logits for W_inject's, and the 2-norm (rounded up), least lsb exponent and largest exponent field of bf16(l).
__global__ void __launch_bounds__(kHcWG) pf_hc_down_epi(const float *raw, uint32_t lr, uint16_t *lb, float *inj,
                                                        double *ln, int *llsb, HcGrid l) {
  __shared__ uint64_t tab[32];
  __shared__ double red[4];
  __shared__ int redi[4];
  int lsb = 1 << 20, top = 0;
  if (threadIdx.x < 32) tab[threadIdx.x] = kExp2Tab[threadIdx.x];
  __syncthreads();
  const uint32_t t = blockIdx.x, M = lr + kHcStreams4;
  double sq = 0.0;
  for (uint32_t j = threadIdx.x; j < M; j += kHcWG) {
    const float v = raw[(uint64_t)t * M + j];
    if (j < lr) {
      const float z = __fmul_rn(v, 0.25f);
      const float o = __fdiv_rn(z, __fadd_rn(1.0f, expf_libm(-z, tab)));
      const float bo = round_bf16(o);
      lb[(uint64_t)t * lr + j] = (uint16_t)(__float_as_uint(bo) >> 16);
      const double b = (double)bo;
      sq = __builtin_fma(b, b, sq);
      lsb = min(lsb, bf16_lsb_of(bo));
      top = max(top, (int)((__float_as_uint(bo) >> 23) & 0xffu));
    } else {
      inj[(uint64_t)t * kHcStreams4 + j - lr] = v;
    }
  }
  sq = wg_sum(sq, red);
  lsb = wg_min(lsb, redi);
  top = -wg_min(-top, redi);
  if (threadIdx.x == 0) l.exp[t] = top;
  if (threadIdx.x == 0) ln[t] = sqrt(sq) * (1.0 + 0x1p-30), llsb[t] = lsb;
}

// x[t][i] = (sum over s in order of n_s[i] sigma(a_s[i])) / 4 with n_s[i] = (R_s[i] sc_s) gamma_s[i] (pf_hc_norm's
// product), a thread two consecutive values (H is a multiple of 512, so a work-group's 512 values are one token's);
// every load issued before the first is used.
__global__ void __launch_bounds__(kHcWG) pf_hc_mix(const float *R, const float *gamma, const float *sc, const float *a,
                                                   uint32_t T, uint32_t H, float *x) {
  __shared__ uint64_t tab[32];
  if (threadIdx.x < 32) tab[threadIdx.x] = kExp2Tab[threadIdx.x];
  __syncthreads();
  const uint64_t e = ((uint64_t)blockIdx.x * kHcWG + threadIdx.x) * 2;
  if (e >= (uint64_t)T * H) return;
  const uint32_t t = (uint32_t)(e / H), i = (uint32_t)(e % H);
  float2 nv[kHcStreams4], av[kHcStreams4], gv[kHcStreams4];
  float scale[kHcStreams4];
#pragma unroll
  for (uint32_t s = 0; s < kHcStreams4; s++) {
    const uint64_t o = ((uint64_t)t * kHcStreams4 + s) * H + i;
    nv[s] = *(const float2 *)(R + o), av[s] = *(const float2 *)(a + o), gv[s] = *(const float2 *)(gamma + s * H + i);
    scale[s] = sc[t * kHcStreams4 + s];
  }
  float2 acc = make_float2(0.0f, 0.0f);
#pragma unroll
  for (uint32_t s = 0; s < kHcStreams4; s++) {
    nv[s].x = __fmul_rn(__fmul_rn(nv[s].x, scale[s]), gv[s].x);
    nv[s].y = __fmul_rn(__fmul_rn(nv[s].y, scale[s]), gv[s].y);
    acc.x = __fadd_rn(acc.x, __fmul_rn(nv[s].x, sigmoid_libm(av[s].x, tab)));
    acc.y = __fadd_rn(acc.y, __fmul_rn(nv[s].y, sigmoid_libm(av[s].y, tab)));
  }
  *(float2 *)(x + e) = make_float2(__fmul_rn(acc.x, 0.25f), __fmul_rn(acc.y, 0.25f));
}

// R_s[i] += 2 sigma(inject_s / 4) y[i], a thread two consecutive values of a token (a work-group's 512 values are one
// token's: H is a multiple of 512), the four stream weights worked out once a work-group.
__global__ void __launch_bounds__(kHcWG) pf_hc_post(float *R, const float *y, const float *inj, uint32_t T,
                                                    uint32_t H) {
  __shared__ uint64_t tab[32];
  __shared__ float ws[kHcStreams4];
  if (threadIdx.x < 32) tab[threadIdx.x] = kExp2Tab[threadIdx.x];
  __syncthreads();
  const uint64_t e0 = (uint64_t)blockIdx.x * kHcWG * 2, e = e0 + 2 * threadIdx.x;
  if (e0 >= (uint64_t)T * H) return;
  const uint32_t t = (uint32_t)(e0 / H), i = (uint32_t)(e % H);
  if (threadIdx.x < kHcStreams4)
    ws[threadIdx.x] = __fmul_rn(2.0f, sigmoid_libm(__fmul_rn(inj[(uint64_t)t * kHcStreams4 + threadIdx.x], 0.25f), tab));
  const float2 yv = *(const float2 *)(y + e);
  float2 rv[kHcStreams4];
#pragma unroll
  for (uint32_t s = 0; s < kHcStreams4; s++) rv[s] = *(const float2 *)(R + ((uint64_t)t * kHcStreams4 + s) * H + i);
  __syncthreads();
#pragma unroll
  for (uint32_t s = 0; s < kHcStreams4; s++) {
    const float w = ws[s];
    *(float2 *)(R + ((uint64_t)t * kHcStreams4 + s) * H + i) =
        make_float2(__fadd_rn(rv[s].x, __fmul_rn(w, yv.x)), __fadd_rn(rv[s].y, __fmul_rn(w, yv.y)));
  }
}

}  // namespace

hipError_t prefill_hc_pre(const HcShape &S, const HcLayer &L, const HcBufs &b, const float *R, bool force_open,
                          hipStream_t st) {
  const uint32_t H = S.H, lr = S.lr, T = S.T, D = kHcStreams4 * H, Md = lr + kHcStreams4;
  const uint32_t nd = D / 64, nu = (lr + 63) / 64, tiles = (T + 15) / 16;
  pf_hc_norm<<<T, kHcStreams4 * kHcWG, 0, st>>>(R, L.gamma, H, b.sc, b.nb, b.nn, b.nlsb, b.ng, b.lg, b.cnt);
  pf_hc_digits<<<dim3(tiles, (nd + 3) / 4), kHcWG, 0, st>>>(b.nb, T, nullptr, T, D, b.ng, b.nd);
  // The down GEMM: K = 4H in kHcDownSplit parts. Roundings on a sum's path: here one a part (wide: at most kGroupK of a
  // matrix-core chain and one a group's total) and one a part's addition; in the fixed order 8 (chain) + 1 + 3 (tree) +
  // K / 2048 (the slot's chunks) + 16 (the slots); doubled, and 2^-53 each.
  const double nd_ref = kHcDownSplit + 28.0 + D / 2048.0, bd = 2.0 * (1.0 + nd_ref) * 0x1p-53;
  const double bdw = 2.0 * (kGroupK + D / kHcDownSplit / kGroupK + 1.0 + nd_ref) * 0x1p-53;
  pf_hc_gemm<false><<<(Md + 63) / 64 * ((T + 63) / 64) * kHcDownSplit, kHcWG, 0, st>>>(
      L.dig_down, Md, b.nd, T, L.w_down, lr, L.w_inj, b.nb, D, nd, kHcDownSplit, b.part, nullptr, b.wide, L.row_norm, b.nn,
      nullptr, nullptr, L.grid, b.ng, 0x1p-30 / sqrt((double)D), 0.0, 0.0, nullptr, nullptr);
  pf_hc_down_fin<<<T, kHcWG, 0, st>>>(b.part, T, Md, kHcDownSplit, L.row_norm, b.nn, L.row_lsb, b.nlsb, L.grid, b.ng, b.wide,
                                      bd, bdw, force_open, b.raw, b.open, b.cnt);
  pf_hc_down_fix<<<1024, kHcWG, 0, st>>>(L.w_down, L.w_inj, lr, D, b.nb, b.open, b.cnt, b.raw);
  pf_hc_down_epi<<<T, kHcWG, 0, st>>>(b.raw, lr, b.lb, b.inj, b.ln, b.llsb, b.lg);
  // The up GEMM: 4H rows of W_up against bf16(l), K = lr; the fixed order is a k chain of lr terms.
  pf_hc_digits<<<dim3(tiles, (nu + 3) / 4), kHcWG, 0, st>>>(b.lb, T, nullptr, T, lr, b.lg, b.ld);
  const double bu = 2.0 * (1.0 + 1.0 + lr) * 0x1p-53, buw = 2.0 * (kGroupK + lr / kGroupK + 1.0 + lr) * 0x1p-53;
  const HcGrid gu{L.grid.exp + Md, L.grid.lost + Md};
  pf_hc_gemm<true><<<(D + 63) / 64 * ((T + 63) / 64), kHcWG, 0, st>>>(
      L.dig_up, D, b.ld, T, L.w_up, D, nullptr, b.lb, lr, nu, 1, nullptr, b.a, nullptr, L.row_norm + Md, b.ln,
      L.row_lsb + Md, b.llsb, gu, b.lg, 0x1p-30 / sqrt((double)lr), bu, buw, b.open_up, b.cnt + 1);
  pf_hc_up_fix<<<256, kHcWG, 0, st>>>(L.w_up, lr, D, b.lb, b.open_up, b.cnt + 1, b.a);
  const uint64_t nx = (uint64_t)T * H;
  pf_hc_mix<<<(uint32_t)((nx + 2 * kHcWG - 1) / (2 * kHcWG)), kHcWG, 0, st>>>(R, L.gamma, b.sc, b.a, T, H, b.x);
  return hipGetLastError();
}

hipError_t prefill_hc_load(uint32_t H, uint32_t lr, const HcLayer &L, uint8_t *dig_down, uint8_t *dig_up, hipStream_t st) {
  const uint32_t D = kHcStreams4 * H, Md = lr + kHcStreams4;
  pf_hc_digits<<<dim3((Md + 15) / 16, (D / 64 + 3) / 4), kHcWG, 0, st>>>(L.w_down, lr, L.w_inj, Md, D, L.grid, dig_down);
  pf_hc_digits<<<dim3(D / 16, ((lr + 63) / 64 + 3) / 4), kHcWG, 0, st>>>(L.w_up, D, nullptr, D, lr,
                                                                         HcGrid{L.grid.exp + Md, L.grid.lost + Md}, dig_up);
  return hipGetLastError();
}

hipError_t prefill_hc_post(const HcShape &S, const HcBufs &b, float *R, const float *y, hipStream_t st) {
  const uint64_t nx = (uint64_t)S.T * S.H;
  pf_hc_post<<<(uint32_t)((nx + 2 * kHcWG - 1) / (2 * kHcWG)), kHcWG, 0, st>>>(R, y, b.inj, S.T, S.H);
  return hipGetLastError();
}

}  // namespace c0ven
