// INT8-weight projections of fp32 activations on the int8 matrix cores.
//
// A row of activations becomes fixed-point numbers of 30 bits and a sign under
// the row's own power of two, x = 2^ex * I with |I| <= 2^30, and each I four
// signed base-256 digits: I = d0 + 2^8 d1 + 2^16 d2 + 2^24 d3. The dot product
// with an int8 weight row is then four int8 dot products with exact int32 sums
// (|sum| <= 2^14 in_dim, in_dim at most 65536), put together in fp32 at the end:
//   y = (s0 + 2^8 s1 + 2^16 s2 + 2^24 s3) * 2^ex * row_scale.
// The only roundings are the row's fixed point (at most 2^-30 of its largest
// element, 64 times finer than fp32's rounding of that element) and the last few
// fp32 operations, against one per product for an fp32 accumulator. The int8
// matrix cores run at twice the bf16 rate, so four digits cost two bf16
// products where the three-way bf16 split costs three, and neither operand is
// converted in the GEMM: weights and digits go from memory to LDS to the
// matrix cores as they are. The digits take the bytes of the fp32 row.
//
// Wide rows. The fixed step is one for the whole row, so an element far below
// the largest keeps fewer than fp32's 24 bits, and an output whose weights are 0
// at the few largest elements would be off by more than an fp32 sum. The writers
// of digit rows therefore mark (when asked, kWideRow) each row whose largest
// magnitude is above kWideRange times its mean magnitude, or which holds an
// infinity and no NaN; the GEMMs then multiply that row in fp32 precision from its
// floats (wide_rows below), in the token tiles that hold such a row alone. For
// an unmarked row, leaving out its largest element leaves a row whose 2-norm is
// at least max (cols / kWideRange - 1) / sqrt(cols), so the fixed point's error
// in a dot product with the rest is at most about
//   2^-29 / sqrt(12) kWideRange / (1 - kWideRange / cols) = 8e-8 (1024 columns)
// of the product's size, at or below that of an fp32 accumulation.
#include "common.hpp"

namespace qasr {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int kDigits = 4;
constexpr int kDigitBits = 30;          // |I| <= 2^30
constexpr int kBadRow = -0x40000000;    // exponent of a row with an infinity (unless marked wide) or NaN: NaN outputs
constexpr int kWideRow = -0x40000001;   // exponent of a row that the GEMMs take from its floats
constexpr float kWideRange = 128.0f;    // largest over mean magnitude from which a row is wide

// Which rows of x_norm the norm writes, and whether it marks wide rows.
enum DigitWide { kNoWide = 0, kWideAllNorm = 1, kWideOwnNorm = 2 };

// One workgroup per row of up to 1024 NV floats: h = x (+ delta, the sum of
// `parts` slices [rows][cols] in slice order, written back to x), with NORM the
// RMSNorm (h * rinv) * gain of it (kernels/mod.rs:897-918) and optionally that
// row itself, then the row's digits and exponent.
struct DigitArgs {
  int8_t* digits;  // [4][rows][cols]
  int32_t* exps;   // [rows]
  float* x;
  const float* delta;  // nullable
  const float* gain;   // NORM
  float* x_norm;       // nullable
  int rows, cols, parts;
  float eps;
  int wide;            // DigitWide; kWideOwnNorm: x_norm gets the wide rows alone
  float wide_sum;      // kWideRange / cols: times a row's sum of magnitudes, the line
};

// The largest of `big` and the sum of `sum` over a workgroup of 256, in one pass
// through LDS.
QASR_DEV void block_max_sum(float& big, float& sum, float (&lds)[2][256 / kWave]) {
  big = wave_max(big);
  sum = wave_sum(sum);
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  if (lane == 0) {
    lds[0][w] = big;
    lds[1][w] = sum;
  }
  __syncthreads();
  big = lds[0][0];
  sum = lds[1][0];
#pragma unroll
  for (int i = 1; i < 256 / kWave; ++i) {
    big = fmaxf(big, lds[0][i]);
    sum += lds[1][i];
  }
}

template <int NV, bool NORM>
__global__ __launch_bounds__(256) void digit_rows_kernel(DigitArgs a) {
  __shared__ float red[2][256 / kWave];
  const int row = blockIdx.x, n4 = a.cols >> 2;
  float* xr = a.x + (size_t)row * a.cols;
  float4 v[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = threadIdx.x + 256 * i;
    v[i] = c < n4 ? ld4(xr, c) : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  if (a.delta) {
    const float* dr = a.delta + (size_t)row * a.cols;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = threadIdx.x + 256 * i;
      if (c < n4) {
        float4 d = ld4(dr, c);
        for (int p = 1; p < a.parts; ++p) {  // uniform
          const float4 e = ld4(dr + (size_t)p * a.rows * a.cols, c);
          d.x += e.x; d.y += e.y; d.z += e.z; d.w += e.w;
        }
        v[i].x += d.x; v[i].y += d.y; v[i].z += d.z; v[i].w += d.w;
        st4(xr, c, v[i]);
      }
    }
  }
  if constexpr (NORM) {
    float4 g[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = threadIdx.x + 256 * i;
      g[i] = c < n4 ? ld4(a.gain, c) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      ss += v[i].x * v[i].x;
      ss += v[i].y * v[i].y;
      ss += v[i].z * v[i].z;
      ss += v[i].w * v[i].w;
    }
    ss = block_sum<256>(ss, red[0]);
    const float rinv = 1.0f / sqrtf(ss / (float)a.cols + a.eps);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = threadIdx.x + 256 * i;
      v[i].x = (v[i].x * rinv) * g[i].x;
      v[i].y = (v[i].y * rinv) * g[i].y;
      v[i].z = (v[i].z * rinv) * g[i].z;
      v[i].w = (v[i].w * rinv) * g[i].w;
      if (a.x_norm && a.wide != kWideOwnNorm && c < n4) st4(a.x_norm + (size_t)row * a.cols, c, v[i]);
    }
  }
  // the largest magnitude; an infinity or NaN counts as infinity
  auto mag = [](float f) {
    const float m = fabsf(f);
    return m <= 3.402823466e38f ? m : __builtin_inff();
  };
  float big = 0.0f, sum = 0.0f;  // of the magnitudes
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    big = fmaxf(big, fmaxf(fmaxf(mag(v[i].x), mag(v[i].y)), fmaxf(mag(v[i].z), mag(v[i].w))));
    sum += (fabsf(v[i].x) + fabsf(v[i].y)) + (fabsf(v[i].z) + fabsf(v[i].w));
  }
  block_max_sum(big, sum, red);
  const bool bad = big == __builtin_inff();
  // The sum is infinite for a row with an infinity and for one of floats so large
  // that it overflows (marked too: its range is not known), NaN only for a row with
  // a NaN, whose outputs are NaN whatever the weights: not worth the floats.
  const bool wide = a.wide && (sum == __builtin_inff() || big > sum * a.wide_sum) && sum == sum;
  const int up = bad ? 0 : kDigitBits - __builtin_amdgcn_frexp_expf(big);  // big < 2^exp (0 for a row of zeros)
  if (threadIdx.x == 0) a.exps[row] = wide ? kWideRow : bad ? kBadRow : -up;
  // byte d of (I + 0x00808080) ^ 0x00808080 is digit d: adding 128 to the lower
  // three bytes carries into the next one where a digit is negative
  auto digits_of = [&](float f) {
    const int q = bad ? 0 : (int)__builtin_rintf(ldexpf(f, up));
    return (unsigned)(q + 0x00808080) ^ 0x00808080u;
  };
  const size_t plane = (size_t)a.rows * a.cols;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = threadIdx.x + 256 * i;
    if (c >= n4) continue;
    const unsigned e0 = digits_of(v[i].x), e1 = digits_of(v[i].y), e2 = digits_of(v[i].z), e3 = digits_of(v[i].w);
    // 4 x 4 byte transpose
    const unsigned l01 = __builtin_amdgcn_perm(e1, e0, 0x05010400u), l23 = __builtin_amdgcn_perm(e3, e2, 0x05010400u);
    const unsigned h01 = __builtin_amdgcn_perm(e1, e0, 0x07030602u), h23 = __builtin_amdgcn_perm(e3, e2, 0x07030602u);
    int8_t* out = a.digits + (size_t)row * a.cols + 4 * c;
    *reinterpret_cast<unsigned*>(out) = __builtin_amdgcn_perm(l23, l01, 0x05040100u);
    *reinterpret_cast<unsigned*>(out + plane) = __builtin_amdgcn_perm(l23, l01, 0x07060302u);
    *reinterpret_cast<unsigned*>(out + 2 * plane) = __builtin_amdgcn_perm(h23, h01, 0x05040100u);
    *reinterpret_cast<unsigned*>(out + 3 * plane) = __builtin_amdgcn_perm(h23, h01, 0x07060302u);
  }
  if constexpr (NORM) {
    if (a.wide == kWideOwnNorm && wide) {
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int c = threadIdx.x + 256 * i;
        if (c < n4) st4(a.x_norm + (size_t)row * a.cols, c, v[i]);
      }
    }
  }
}

template <bool NORM>
bool launch_digit_rows(const DigitArgs& a, hipStream_t st) {
  const unsigned g = (unsigned)a.rows;
  switch ((a.cols + 1023) / 1024) {
    case 1: digit_rows_kernel<1, NORM><<<g, 256, 0, st>>>(a); return true;
    case 2: digit_rows_kernel<2, NORM><<<g, 256, 0, st>>>(a); return true;
    case 3: digit_rows_kernel<3, NORM><<<g, 256, 0, st>>>(a); return true;
    case 4: digit_rows_kernel<4, NORM><<<g, 256, 0, st>>>(a); return true;
    case 5:
    case 6: digit_rows_kernel<6, NORM><<<g, 256, 0, st>>>(a); return true;
    case 7:
    case 8: digit_rows_kernel<8, NORM><<<g, 256, 0, st>>>(a); return true;
    default: return false;
  }
}

enum DigitEpi { kDgPlain = 0, kDgResidual = 1, kDgSwiglu = 2, kDgSwigluLibm = 3, kDgHeads = 4 };

// kDgHeads: the matrices are q, k and v, every 128-row tile is one head, and
// token t sits at position start_pos + t: per-head RMSNorm + NeoX RoPE of the q
// and k heads (decoder.rs:799-804), q to y, the k and v rows to the caches
// (:805-810). The entry point has checked that every position lies inside both.
struct DigitHeads {
  float* k_cache;
  float* v_cache;
  const float* q_norm_w;
  const float* k_norm_w;
  const float* cos_tab;
  const float* sin_tab;
  long long start_pos;
  float eps;
};

struct DigitGemm {
  float* y[3];
  const int8_t* w[3];   // [N][K]
  const float* s[3];
  int N[3];
  unsigned bx_begin[4];
  int n;
  const int8_t* digits;  // [4][T][K]
  const int32_t* exps;
  const float* x;        // [T][K], read for rows marked kWideRow; null: such rows give NaN
  int T, K;
  int parts;             // K cut over this many workgroups: part p writes y + p * T * N (kDgPlain)
  unsigned cols, rows, split_cols;  // the tile grid, and how the XCDs share it
  DigitHeads heads;
};

// The K groups' double buffers, or their output tiles after the loop.
template <int BN, int BT, int BK, int KW>
constexpr size_t digit_gemm_tile_bytes() {
  constexpr size_t stages = (size_t)KW * 2 * (BN + kDigits * BT) * BK;
  constexpr size_t tiles = (size_t)KW * BT * (BN + 4) * sizeof(float);
  return stages > tiles ? stages : tiles;
}

// acc[i] = the dot products of a 32-token block's wide rows with MI 32-row weight
// blocks over nk (a multiple of 64) of K, with the sums of the bf16 split
// (int8.hip): an int8 weight is exact in bf16, an fp32 activation is
// hi + mid + lo exactly, and the products are summed in fp32. The operands come
// straight from memory (L2), a 64-wide chunk ahead: of every 32 of K, lane (r, g)
// loads 16 weights of row r and 16 floats of a token, the first 8 of each for one
// matrix instruction and the rest for the next (the same permutation of K for
// both). xp and wp[i] point at the lane's first ones; lanes of other tokens pass
// a wide one's xp, so that no load is conditional, and their columns mean
// nothing. An infinity or NaN travels as in fp32: hi alone carries an infinity.
// What a launch costs without, with one and with only wide rows, and the bf16
// split on the same product (us): 64 tokens [2048 -> 12288] 14, 34, 51 and 20;
// 77 [3072 -> 1024] 9, 17, 23 and 13; 8 [2048 -> 151936] 63, 140, 150 and 131.
// Each wave converts its own operands and shares nothing through LDS, which is
// what the split's launches are faster by where every row is wide.
template <int MI>
QASR_DEV void wide_rows(v16f (&acc)[MI], const int8_t* const (&wp)[MI], const float* xp, int nk) {
  v16f low[MI];
#pragma unroll
  for (int i = 0; i < MI; ++i) acc[i] = low[i] = v16f{};
  struct Chunk {
    v4i w[MI][2];
    v4f x[2][4];
  };
  auto load = [&](Chunk& c, int k) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int i = 0; i < MI; ++i) c.w[i][h] = *reinterpret_cast<const v4i*>(wp[i] + k + 32 * h);
#pragma unroll
      for (int q = 0; q < 4; ++q) c.x[h][q] = *reinterpret_cast<const v4f*>(xp + k + 32 * h + 4 * q);
    }
  };
  auto multiply = [&](const Chunk& c) {
#pragma unroll
    for (int h = 0; h < 4; ++h) {  // 16 of K: half h % 2 of the lane's 16 of 32-block h / 2
      v4u b[3];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        float e[2], r1[2], r2[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          e[j] = c.x[h >> 1][2 * (h & 1) + (p >> 1)][2 * (p & 1) + j];
          r1[j] = fabsf(e[j]) == __builtin_inff() ? 0.0f : e[j] - bf16_trunc(e[j]);
          r2[j] = r1[j] - bf16_trunc(r1[j]);  // at most 8 significant bits
        }
        b[0][p] = bf16_pair(e[0], e[1]);
        b[1][p] = bf16_pair(r1[0], r1[1]);
        b[2][p] = bf16_pair(r2[0], r2[1]);
      }
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const int w0 = c.w[i][h >> 1][2 * (h & 1)], w1 = c.w[i][h >> 1][2 * (h & 1) + 1];
        const v8bf a = __builtin_bit_cast(v8bf, v4u{bf16_pair_i8(w0, 0), bf16_pair_i8(w0, 2), bf16_pair_i8(w1, 0),
                                                    bf16_pair_i8(w1, 2)});
        acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, __builtin_bit_cast(v8bf, b[0]), acc[i], 0, 0, 0);
        low[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, __builtin_bit_cast(v8bf, b[1]), low[i], 0, 0, 0);
        low[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, __builtin_bit_cast(v8bf, b[2]), low[i], 0, 0, 0);
      }
    }
  };
  Chunk c[2];
  load(c[0], 0);
  for (int k = 0; k < nk; k += 128) {
    load(c[1], min(k + 64, nk - 64));  // past the end: the last chunk again, not multiplied
    __builtin_amdgcn_sched_barrier(0);
    multiply(c[0]);
    if (k + 64 < nk) {  // uniform
      load(c[0], min(k + 128, nk - 64));
      __builtin_amdgcn_sched_barrier(0);
      multiply(c[1]);
    }
  }
#pragma unroll
  for (int i = 0; i < MI; ++i) acc[i] += low[i];
}

// One BN x BT output tile (BT tokens, so 4 BT digit columns) per workgroup.
// KW groups of waves take a K range each and meet in the epilogue; a group's
// waves are a (BN / 32 MI) x (BT / 32) grid, each MI x 4 blocks of 32 x 32: a
// lane ends up with the four digit sums of its (row, token) pairs. BK bytes of
// K per chunk, two LDS buffers; while chunk c is multiplied, each k step also
// stores a share of chunk c + 1 (in registers since the step before the last
// barrier) into the other buffer and issues the loads of chunk c + 2 in their
// place: a load has a whole chunk's products to arrive in, and LDS writes and
// address work hide under the matrix pipe. 16-byte slots are XOR-swizzled by
// row so that a fragment read touches every bank once.
template <int BN, int BT, int MI, int BK, int KW, int EPI>
__global__ __launch_bounds__(64 * KW * (BN / (32 * MI)) * (BT / 32), 2) void digit_gemm_kernel(DigitGemm a) {
  constexpr int WR = BN / (32 * MI), WC = BT / 32;
  constexpr int NTG = 64 * WR * WC;            // threads of a K group
  constexpr int NT = NTG * KW;
  constexpr int SL = BK / 16;                  // 16-byte slots of a row
  constexpr int ROWS = BN + kDigits * BT;
  constexpr int U = ROWS * SL / NTG;           // staged slots per thread
  constexpr int RPU = NTG / SL;                // rows per staging step
  constexpr int UW = BN / RPU;                 // the steps that stage weights
  constexpr int KS = BK / 32;
  constexpr int STAGE = ROWS * BK;
  constexpr int PART = (U + KS - 1) / KS;
  constexpr size_t TILE_BYTES = digit_gemm_tile_bytes<BN, BT, BK, KW>();
  static_assert(BN % RPU == 0 && (kDigits * BT) % RPU == 0 && U * NTG == ROWS * SL, "whole staging steps");
  static_assert(SL == 8 || SL == 4, "the swizzle");
  static_assert(BN <= NT, "one scale per thread");
  // the 16 rows that a quarter of a fragment read touches fall on 16 slots of a 256-byte bank line
  auto swizzled = [](int row, int slot) { return SL == 8 ? slot ^ ((row >> 1) & 7) : slot ^ ((row >> 2) & 3); };
  extern __shared__ __align__(16) int8_t dg_lds[];

  unsigned bx, by;
  const unsigned part = EPI == kDgPlain ? blockIdx.x / (a.cols * a.rows) : 0;
  const unsigned block = blockIdx.x - part * a.cols * a.rows;
  if (a.split_cols == 0) {
    bx = block % a.cols;
    by = block / a.cols;
  } else {
    const unsigned xcd = block % 8, slot = block / 8;
    const unsigned ca = a.cols / a.split_cols, rb = a.rows / (8 / a.split_cols);
    bx = (xcd % a.split_cols) * ca + slot % ca;
    by = (xcd / a.split_cols) * rb + slot / ca;
  }
  float* y = a.y[0];
  const int8_t* w = a.w[0];
  const float* scales = a.s[0];
  int N = a.N[0];
  unsigned bx0 = 0;
  [[maybe_unused]] int mat = 0;
#pragma unroll
  for (int m = 1; m < 3; ++m)
    if (m < a.n && bx >= a.bx_begin[m]) {
      y = a.y[m];
      w = a.w[m];
      scales = a.s[m];
      N = a.N[m];
      bx0 = a.bx_begin[m];
      mat = m;
    }
  const int n0 = (int)(bx - bx0) * BN, t0 = (int)by * BT;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int kg = wave / (WR * WC), wv = wave % (WR * WC);
  const int wr = wv % WR, wc = wv / WR;
  const int r = lane & 31, g = lane >> 5;
  const int gt = (int)threadIdx.x - kg * NTG;  // thread of its group
  const int nch = a.K / (BK * KW * a.parts);
  if constexpr (EPI == kDgPlain) y += (size_t)part * a.T * N;
  int8_t* buf = dg_lds + kg * 2 * STAGE;

  // row of the digit block of a token tile: 128 (t / 32) + 32 d + t % 32
  const int8_t* src[U];
  int dst[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int row = u * RPU + gt / SL, slot = gt % SL;
    const size_t k = (size_t)((int)part * KW + kg) * nch * BK + 16 * slot;
    if (u < UW) {
      src[u] = w + (size_t)min(n0 + row, N - 1) * a.K + k;  // rows and tokens past the end re-read the last one
    } else {
      const int xr = row - BN;
      const int t = min(t0 + 32 * (xr >> 7) + (xr & 31), a.T - 1), d = (xr >> 5) & 3;
      src[u] = a.digits + ((size_t)d * a.T + t) * a.K + k;
    }
    dst[u] = row * BK + 16 * swizzled(row, slot);
  }
  // row scales and token exponents of the tile, for the epilogue
  float* sc_lds = reinterpret_cast<float*>(dg_lds + TILE_BYTES);
  int* ex_lds = reinterpret_cast<int*>(sc_lds + BN);
  if ((int)threadIdx.x < BN) sc_lds[threadIdx.x] = scales[min(n0 + (int)threadIdx.x, N - 1)];
  if ((int)threadIdx.x < BT) ex_lds[threadIdx.x] = a.exps[min(t0 + (int)threadIdx.x, a.T - 1)];
  const int t_wave = min(t0 + 32 * wc + r, a.T - 1);
  int e_wave;  // of this lane's token, looked at after the loop
  v4i st[U];
  {
    v4i first[U];
#pragma unroll
    for (int u = 0; u < U; ++u) first[u] = *reinterpret_cast<const v4i*>(src[u]);
    const int k = min(1, nch - 1) * BK;
#pragma unroll
    for (int u = 0; u < U; ++u) st[u] = *reinterpret_cast<const v4i*>(src[u] + k);
    e_wave = a.exps[t_wave];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u) *reinterpret_cast<v4i*>(buf + dst[u]) = first[u];
  }
  v16i acc[MI][kDigits];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int d = 0; d < kDigits; ++d) acc[i][d] = v16i{};
  lds_barrier();

  auto frag = [&](const int8_t* b, int row, int s) {
    return *reinterpret_cast<const v4i*>(b + row * BK + 16 * swizzled(row, 2 * s + g));
  };
  auto read_step = [&](const int8_t* b, int s, v4i (&fa)[MI], v4i (&fb)[kDigits]) {
#pragma unroll
    for (int i = 0; i < MI; ++i) fa[i] = frag(b, 32 * (MI * wr + i) + r, s);
#pragma unroll
    for (int d = 0; d < kDigits; ++d) fb[d] = frag(b, BN + 128 * wc + 32 * d + r, s);
  };
  for (int c = 0; c < nch; ++c) {
    const int8_t* cur = buf + (c & 1) * STAGE;
    int8_t* nxt = buf + ((c + 1) & 1) * STAGE;
    const int k2 = min(c + 2, nch - 1) * BK;  // past the end: the last chunk again, into the idle buffer
    v4i fa[2][MI], fb[2][kDigits];
    read_step(cur, 0, fa[0], fb[0]);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      if (s + 1 < KS) read_step(cur, s + 1, fa[(s + 1) & 1], fb[(s + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int d = 0; d < kDigits; ++d)
          acc[i][d] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[s & 1][i], fb[s & 1][d], acc[i][d], 0, 0, 0);
#pragma unroll
      for (int u = PART * s; u < (PART * (s + 1) < U ? PART * (s + 1) : U); ++u) {
        *reinterpret_cast<v4i*>(nxt + dst[u]) = st[u];
        st[u] = *reinterpret_cast<const v4i*>(src[u] + k2);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    lds_barrier();
  }

  // The groups' tiles go through LDS, [KW][BT][BN + 4] floats, so that the
  // output rows are read and written in whole lines.
  constexpr int PITCH = BN + 4;
  float* tile = reinterpret_cast<float*>(dg_lds);
  {
    float* mine = tile + ((size_t)kg * BT + 32 * wc + r) * PITCH;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float f[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int e = 4 * q + v;
          f[v] = __builtin_fmaf((float)acc[i][1][e], 256.0f, (float)acc[i][0][e]);
          f[v] = __builtin_fmaf((float)acc[i][2][e], 65536.0f, f[v]);
          f[v] = __builtin_fmaf((float)acc[i][3][e], 16777216.0f, f[v]);
        }
        *reinterpret_cast<float4*>(mine + 32 * (MI * wr + i) + 8 * q + 4 * g) = make_float4(f[0], f[1], f[2], f[3]);
      }
    // This wave's wide rows again, from the floats: its own part of the tile, its own part of K.
    const unsigned wide_tokens = a.x ? (unsigned)__ballot(e_wave == kWideRow) : 0u;
    if (wide_tokens) {
      const size_t k = (size_t)((int)part * KW + kg) * nch * BK + 16 * g;
      const int8_t* wp[MI];
#pragma unroll
      for (int i = 0; i < MI; ++i) wp[i] = w + (size_t)min(n0 + 32 * (MI * wr + i) + r, N - 1) * a.K + k;
      const bool wide = wide_tokens >> r & 1;
      const int t = wide ? t_wave : min(t0 + 32 * wc + __builtin_ctz(wide_tokens), a.T - 1);
      v16f f[MI];
      wide_rows<MI>(f, wp, a.x + (size_t)t * a.K + k, nch * BK);
      if (wide) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            *reinterpret_cast<float4*>(mine + 32 * (MI * wr + i) + 8 * q + 4 * g) =
                make_float4(f[i][4 * q], f[i][4 * q + 1], f[i][4 * q + 2], f[i][4 * q + 3]);
      }
    }
  }
  __syncthreads();
  // a token's power of two (a wide row's floats have none), and a sum of products times it
  auto power = [&](int tt) { return ex_lds[tt] == kWideRow && a.x ? 0 : ex_lds[tt]; };
  auto powered = [](float v, int ex) { return ex <= kBadRow ? qnan() : ldexpf(v, ex); };
  if constexpr (EPI == kDgHeads) {
    // 16 lanes a head: lane `sub` holds dims 4 sub.. and 64 + 4 sub..
    constexpr int L = 16, PER = NT / L;
    static_assert(BN == 128 && BT % PER == 0, "one head per tile");
    const DigitHeads& he = a.heads;
    const int sub = threadIdx.x % L;
    const float* gain = mat == 0 ? he.q_norm_w : he.k_norm_w;
    const float4 w1 = ld4(gain, sub), w2 = ld4(gain + 64, sub);
#pragma unroll
    for (int p = 0; p < BT / PER; ++p) {
      const int tt = p * PER + threadIdx.x / L, t = t0 + tt;
      const size_t pos = (size_t)(he.start_pos + min(t, a.T - 1)), trow = pos * 128;
      const float4 c1 = ld4(he.cos_tab + trow, sub), c2 = ld4(he.cos_tab + trow + 64, sub);
      const float4 s1 = ld4(he.sin_tab + trow, sub), s2 = ld4(he.sin_tab + trow + 64, sub);
      const int ex = power(tt);
      auto value = [&](int c) {
        float4 f = *reinterpret_cast<const float4*>(tile + (size_t)tt * PITCH + c);
#pragma unroll
        for (int k = 1; k < KW; ++k) {
          const float4 q = *reinterpret_cast<const float4*>(tile + ((size_t)k * BT + tt) * PITCH + c);
          f.x += q.x; f.y += q.y; f.z += q.z; f.w += q.w;
        }
        const float4 sc = *reinterpret_cast<const float4*>(sc_lds + c);
        return make_float4(powered(f.x * sc.x, ex), powered(f.y * sc.y, ex), powered(f.z * sc.z, ex),
                           powered(f.w * sc.w, ex));
      };
      float4 x1 = value(4 * sub), x2 = value(64 + 4 * sub);
      if (mat != 2) head_norm_rope<128, true, true>(x1, x2, w1, w2, c1, c2, s1, s2, true, he.eps);
      if (t >= a.T) continue;
      float* row = mat == 0 ? y + (size_t)t * N : (mat == 1 ? he.k_cache : he.v_cache) + pos * N;
      st4(row + n0, sub, x1);
      st4(row + n0 + 64, sub, x2);
    }
    return;
  }
  constexpr int C4 = BN / 4, IT = BT * C4 / NT;
  static_assert(IT * NT == BT * C4 && (NT % C4 == 0 || C4 % NT == 0), "whole passes over the tile");
  [[maybe_unused]] float4 h[IT];
  if constexpr (EPI == kDgResidual) {
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      const int it = (int)threadIdx.x + NT * i, n = n0 + 4 * (it % C4), t = t0 + it / C4;
      h[i] = ld4(y + (size_t)min(t, a.T - 1) * N + min(n, N - 4), 0);
    }
  }
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int it = (int)threadIdx.x + NT * i;
    const int tt = it / C4, c = 4 * (it % C4), n = n0 + c, t = t0 + tt;
    float4 f = *reinterpret_cast<const float4*>(tile + (size_t)tt * PITCH + c);
#pragma unroll
    for (int k = 1; k < KW; ++k) {
      const float4 p = *reinterpret_cast<const float4*>(tile + ((size_t)k * BT + tt) * PITCH + c);
      f.x += p.x; f.y += p.y; f.z += p.z; f.w += p.w;
    }
    const float4 sc = *reinterpret_cast<const float4*>(sc_lds + c);
    const int ex = power(tt);
    float res[4] = {f.x * sc.x, f.y * sc.y, f.z * sc.z, f.w * sc.w};
#pragma unroll
    for (int v = 0; v < 4; ++v) res[v] = powered(res[v], ex);
    if (t >= a.T || n >= N) continue;
    if constexpr (EPI == kDgSwiglu || EPI == kDgSwigluLibm) {
      const int inter = N >> 1, j = n >> 1, fast_end = EPI == kDgSwiglu ? inter & ~7 : 0;
      *reinterpret_cast<float2*>(y + (size_t)t * inter + j) =
          make_float2(swiglu_ref(res[0], res[1], j < fast_end), swiglu_ref(res[2], res[3], j + 1 < fast_end));
    } else {
      if constexpr (EPI == kDgResidual) {
        res[0] = h[i].x + res[0];
        res[1] = h[i].y + res[1];
        res[2] = h[i].z + res[2];
        res[3] = h[i].w + res[3];
      }
      st4(y + (size_t)t * N + n, 0, make_float4(res[0], res[1], res[2], res[3]));
    }
  }
}

template <int BN, int BT, int MI, int BK, int KW, int EPI>
bool run_digit_gemm(DigitGemm a, hipStream_t st) {
  constexpr size_t lds = digit_gemm_tile_bytes<BN, BT, BK, KW>() + (BN + BT) * 4;
  static_assert(lds <= 163840, "LDS of a CU");
  if (a.K % (BK * KW * a.parts) != 0) return false;
  if (!raise_lds_limit<&digit_gemm_kernel<BN, BT, MI, BK, KW, EPI>>(lds)) return false;
  unsigned c = 0;
  for (int m = 0; m < a.n; ++m) {
    a.bx_begin[m] = c;
    c += (unsigned)((a.N[m] + BN - 1) / BN);
  }
  for (int m = a.n; m <= 3; ++m) a.bx_begin[m] = c;
  a.cols = c;
  a.rows = (unsigned)((a.T + BT - 1) / BT);
  constexpr unsigned kThreads = 64 * KW * (BN / (32 * MI)) * (BT / 32);
  if (!exact_grid_ok((size_t)a.cols * a.rows * (size_t)a.parts * kThreads)) return false;
  // the XCD map that reads least: cols / s weight blocks and rows / (8 / s) token blocks each
  a.split_cols = 0;
  double best = 0;
  for (unsigned s = 1; s <= 8; s *= 2) {
    if (a.cols % s || a.rows % (8 / s)) continue;
    const double cost = (double)(a.cols / s) * BN + (double)(a.rows / (8 / s)) * BT * kDigits;
    if (a.split_cols == 0 || cost < best) {
      a.split_cols = s;
      best = cost;
    }
  }
  digit_gemm_kernel<BN, BT, MI, BK, KW, EPI>
      <<<a.cols * a.rows * (unsigned)a.parts, kThreads, lds, st>>>(a);
  return true;
}

// Tile choice by a cost fitted to measured times (us; K' = in_dim / 1024,
// n tiles on 256 CUs, weights and digits in L2 or HBM as a layer finds them):
//   256 x 64, one workgroup a CU   2.5 + ceil(n / 256) (5.2 + 12.7 K')
//   128 x 32, two a CU             5   + max(1, n / 256) 5.2 K'
//   64 x 32, K over 4 wave groups  2.5 + ceil(n / 256) (2.6 + 3.6 K')
//   32 x 32, K over 4 waves        3.5 + 1.8 K' up to n = 256, then 3.5 + n / 256 3.6 K'
// A CU holds one 32 x 32 workgroup (82 KB of LDS): 256 tiles are one round, 257 two.
// That tile measured at 64 tokens and K' = 1, 2 and 6: 64 tiles 5.7, 7.3 and 14.0 us,
// 256 7.0, 9.1 and 21.6, 320 10.7, 14.7 and 35.8, 512 11.9, 16.1 and 44.4 (64 x 32 on
// the same products, half the tiles: 6.3, 8.4, 17.5; 6.6, 8.8, 21.9; 6.9, 9.1, 22.9;
// 7.9, 10.8, 26.1).
// Measured on one MI355X against the bf16 three-way split kernels (int8.hip)
// for the same product: 1473 tokens [2048 -> 12288] 163 us against 242 (1.8e15
// int8 operations a second, 74% of what the same matrix instructions reach
// alone), [6144 -> 2048] 85 against 142, [2048 -> 4096] 62 against 88; 512
// tokens [1024 -> 6144] 20 against 25; 64 tokens [2048 -> 12288] 13.7 against
// 20.4, [2048 -> 151936] 115 against 162; 11 tokens [1024 -> 151936] 33 against
// 72. Error against 64 bits 3.7e-8 to 5.7e-8 where theirs is 8e-8 to 8e-7.
template <int EPI>
bool launch_digit_gemm(const DigitGemm& a, hipStream_t st) {
  if constexpr (EPI == kDgHeads) {
    return run_digit_gemm<128, 32, 1, 128, 1, EPI>(a, st);
  } else {
    auto tiles = [&](int bn, int bt) {
      long long c = 0;
      for (int m = 0; m < a.n; ++m) c += (a.N[m] + bn - 1) / bn;
      return (double)(c * ((a.T + bt - 1) / bt) * a.parts) / 256.0;
    };
    const double k = a.K / (1024.0 * a.parts);
    const double t32 = tiles(32, 32), t64 = tiles(64, 32), t128 = tiles(128, 32), t256 = tiles(256, 64);
    const double c256 = 2.5 + ceil(t256) * (5.2 + 12.7 * k);
    const double c128 = 5.0 + (t128 > 1.0 ? t128 : 1.0) * 5.2 * k;
    const double c64 = 2.5 + ceil(t64) * (2.6 + 3.6 * k);
    const double c32 = 3.5 + (t32 > 1.0 ? t32 : 0.5) * 3.6 * k;
    const double small = c32 < c64 ? c32 : c64, large = c128 < c256 ? c128 : c256;
    if (small < large)
      return c32 < c64 ? run_digit_gemm<32, 32, 1, 64, 4, EPI>(a, st) : run_digit_gemm<64, 32, 1, 64, 4, EPI>(a, st);
    return c128 < c256 ? run_digit_gemm<128, 32, 1, 128, 1, EPI>(a, st)
                       : run_digit_gemm<256, 64, 2, 128, 1, EPI>(a, st);
  }
}

// Parts of K for a projection whose 32 x 32 tiles leave CUs idle (a few streams'
// o and down projections): as many, up to 4, as still give each CU at most one
// workgroup of at least 512 of K. Their slices are added by the norm that reads
// them (qasr_add_rms_norm_digits_f32), so no launch is added.
size_t digit_parts(size_t T, size_t K, size_t N) {
  const size_t tiles = ((N + 31) / 32) * ((T + 31) / 32);
  size_t p = 1;
  while (p < 4 && 2 * p * tiles <= 256 && K % (512 * p) == 0 && K / (2 * p) >= 512) p *= 2;
  return p;
}

int digit_gemm_checks(size_t T, size_t K, const int8_t* digits, const int32_t* exps, const float* x,
                      const char* what) {
  QASR_REQUIRE(digits && exps, std::string(what) + ": null pointer");
  size_t n;
  QASR_REQUIRE(T <= 0xffffffu && K <= 65536 && mul_ok(T, 4 * K, &n), std::string(what) + ": size too large");
  if (K == 0 || K % 256 != 0 || !aligned16(digits) || !aligned4(exps) || !aligned16(x))
    return fail(QASR_ERR_UNSUPPORTED,
                std::string(what) + ": in_dim must be a multiple of 256, digits and x 16-byte aligned");
  return QASR_OK;
}

int digit_mat_checks(const float* y, const int8_t* w, const float* s, size_t N, size_t T, size_t K,
                     const char* what) {
  QASR_REQUIRE(y && w && s, std::string(what) + ": null pointer");
  size_t n;
  QASR_REQUIRE(N <= 0x3fffffffu && mul_ok(N, K, &n) && mul_ok(T, N, &n), std::string(what) + ": size too large");
  if (N == 0 || N % 4 != 0 || !aligned16(y) || !aligned16(w) || !aligned4(s))
    return fail(QASR_ERR_UNSUPPORTED,
                std::string(what) + ": out_dim must be a multiple of 4, outputs and weights 16-byte aligned");
  return QASR_OK;
}

}  // namespace
}  // namespace qasr

using namespace qasr;

static int digit_rows(int8_t* digits, int32_t* exps, const float* x, size_t rows, size_t cols, DigitWide wide,
                      void* stream) {
  if (rows == 0) return QASR_OK;
  QASR_REQUIRE(digits && exps && x, "digit_rows: null pointer");
  QASR_REQUIRE(rows < kMaxRows, "digit_rows: too many rows");
  if (cols == 0 || cols % 4 != 0 || cols > 8192 || !aligned16(x) || !aligned16(digits) || !aligned4(exps))
    return fail(QASR_ERR_UNSUPPORTED, "digit_rows: cols must be a multiple of 4 up to 8192, buffers 16-byte aligned");
  const DigitArgs a{digits, exps, const_cast<float*>(x), nullptr, nullptr, nullptr, (int)rows, (int)cols, 1, 0.0f,
                    wide, kWideRange / (float)cols};
  if (!launch_digit_rows<false>(a, as_stream(stream)))
    return fail(QASR_ERR_UNSUPPORTED, "digit_rows: no kernel for this row length");
  return launch_status("digit_rows");
}

extern "C" int qasr_digit_rows_f32(int8_t* digits, int32_t* exps, const float* x, size_t rows, size_t cols,
                                   void* stream) {
  return digit_rows(digits, exps, x, rows, cols, kNoWide, stream);
}

extern "C" int qasr_digit_rows_wide_f32(int8_t* digits, int32_t* exps, const float* x, size_t rows, size_t cols,
                                        void* stream) {
  return digit_rows(digits, exps, x, rows, cols, kWideAllNorm, stream);
}

static int add_rms_norm_digits(float* x, const float* delta, size_t delta_parts, const float* weight, float* x_norm,
                               DigitWide wide, int8_t* digits, int32_t* exps, size_t rows, size_t cols, float eps,
                               void* stream) {
  if (rows == 0) return QASR_OK;
  QASR_REQUIRE(x && weight && digits && exps && (x_norm || wide == kNoWide), "add_rms_norm_digits: null pointer");
  QASR_REQUIRE(rows < kMaxRows && delta_parts >= 1 && delta_parts <= 4,
               "add_rms_norm_digits: too many rows, or not 1 to 4 slices of delta");
  if (cols == 0 || cols % 4 != 0 || cols > 8192 || !aligned16(x) || !aligned16(delta) || !aligned16(weight) ||
      !aligned16(x_norm) || !aligned16(digits) || !aligned4(exps))
    return fail(QASR_ERR_UNSUPPORTED,
                "add_rms_norm_digits: cols must be a multiple of 4 up to 8192, buffers 16-byte aligned");
  const DigitArgs a{digits, exps, x, delta, weight, x_norm, (int)rows, (int)cols, (int)delta_parts, eps, wide,
                    kWideRange / (float)cols};
  if (!launch_digit_rows<true>(a, as_stream(stream)))
    return fail(QASR_ERR_UNSUPPORTED, "add_rms_norm_digits: no kernel for this row length");
  return launch_status("add_rms_norm_digits");
}

extern "C" int qasr_add_rms_norm_digits_f32(float* x, const float* delta, size_t delta_parts, const float* weight,
                                            float* x_norm, int8_t* digits, int32_t* exps, size_t rows, size_t cols,
                                            float eps, void* stream) {
  return add_rms_norm_digits(x, delta, delta_parts, weight, x_norm, kNoWide, digits, exps, rows, cols, eps, stream);
}

extern "C" int qasr_add_rms_norm_digits_wide_f32(float* x, const float* delta, size_t delta_parts,
                                                 const float* weight, float* x_norm, size_t all_rows,
                                                 int8_t* digits, int32_t* exps, size_t rows, size_t cols, float eps,
                                                 void* stream) {
  return add_rms_norm_digits(x, delta, delta_parts, weight, x_norm, all_rows ? kWideAllNorm : kWideOwnNorm, digits,
                             exps, rows, cols, eps, stream);
}

extern "C" int qasr_linear_digits_wide_int8_f32(size_t n_mats, float* const* ys, const int8_t* const* ws,
                                                const float* const* scales, const size_t* out_dims,
                                                const int8_t* digits, const int32_t* exps, const float* x,
                                                size_t seq, size_t in_dim, size_t residual, size_t parts,
                                                void* stream) {
  if (seq == 0 || n_mats == 0) return QASR_OK;
  QASR_REQUIRE(n_mats <= 3 && ys && ws && scales && out_dims, "linear_digits: 1 to 3 matrices");
  QASR_REQUIRE(parts >= 1 && parts <= 4 && (parts == 1 || !residual),
               "linear_digits: 1 to 4 parts, and only one with a residual");
  int rc = digit_gemm_checks(seq, in_dim, digits, exps, x, "linear_digits");
  if (rc != QASR_OK) return rc;
  DigitGemm a{};
  a.n = (int)n_mats;
  for (size_t m = 0; m < n_mats; ++m) {
    rc = digit_mat_checks(ys[m], ws[m], scales[m], out_dims[m], parts * seq, in_dim, "linear_digits");
    if (rc != QASR_OK) return rc;
    a.y[m] = ys[m];
    a.w[m] = ws[m];
    a.s[m] = scales[m];
    a.N[m] = (int)out_dims[m];
  }
  a.digits = digits;
  a.exps = exps;
  a.x = x;
  a.T = (int)seq;
  a.K = (int)in_dim;
  a.parts = (int)parts;
  const bool ok = residual ? launch_digit_gemm<kDgResidual>(a, as_stream(stream))
                           : launch_digit_gemm<kDgPlain>(a, as_stream(stream));
  if (!ok) return fail(QASR_ERR_UNSUPPORTED, "linear_digits: no kernel for this shape");
  return launch_status("linear_digits");
}

extern "C" int qasr_linear_digits_int8_f32(size_t n_mats, float* const* ys, const int8_t* const* ws,
                                           const float* const* scales, const size_t* out_dims,
                                           const int8_t* digits, const int32_t* exps, size_t seq, size_t in_dim,
                                           size_t residual, size_t parts, void* stream) {
  return qasr_linear_digits_wide_int8_f32(n_mats, ys, ws, scales, out_dims, digits, exps, nullptr, seq, in_dim,
                                          residual, parts, stream);
}

extern "C" size_t qasr_linear_digits_parts(size_t seq, size_t in_dim, size_t out_dim) {
  if (seq == 0 || seq > 0xffffffu || out_dim > 0x3fffffffu) return 1;
  return digit_parts(seq, in_dim, out_dim);
}

extern "C" int qasr_gate_up_swiglu_digits_wide_int8_f32(float* out, const int8_t* w_gate_up, const float* scales,
                                                        const int8_t* digits, const int32_t* exps, const float* x,
                                                        size_t seq, size_t in_dim, size_t inter, size_t prefill,
                                                        void* stream) {
  if (seq == 0 || inter == 0) return QASR_OK;
  int rc = digit_gemm_checks(seq, in_dim, digits, exps, x, "gate_up_swiglu_digits");
  if (rc != QASR_OK) return rc;
  rc = digit_mat_checks(out, w_gate_up, scales, 2 * inter, seq, in_dim, "gate_up_swiglu_digits");
  if (rc != QASR_OK) return rc;
  DigitGemm a{};
  a.n = 1;
  a.y[0] = out;
  a.w[0] = w_gate_up;
  a.s[0] = scales;
  a.N[0] = (int)(2 * inter);
  a.digits = digits;
  a.exps = exps;
  a.x = x;
  a.T = (int)seq;
  a.K = (int)in_dim;
  a.parts = 1;
  const bool ok = prefill ? launch_digit_gemm<kDgSwiglu>(a, as_stream(stream))
                          : launch_digit_gemm<kDgSwigluLibm>(a, as_stream(stream));
  if (!ok) return fail(QASR_ERR_UNSUPPORTED, "gate_up_swiglu_digits: no kernel for this shape");
  return launch_status("gate_up_swiglu_digits");
}

extern "C" int qasr_gate_up_swiglu_digits_int8_f32(float* out, const int8_t* w_gate_up, const float* scales,
                                                   const int8_t* digits, const int32_t* exps, size_t seq,
                                                   size_t in_dim, size_t inter, size_t prefill, void* stream) {
  return qasr_gate_up_swiglu_digits_wide_int8_f32(out, w_gate_up, scales, digits, exps, nullptr, seq, in_dim, inter,
                                                  prefill, stream);
}

extern "C" int qasr_qkv_heads_digits_wide_int8_f32(
    float* q, float* k_cache, float* v_cache, size_t cache_rows, const int8_t* wq, const float* sq, const int8_t* wk,
    const float* sk, const int8_t* wv, const float* sv, const int8_t* digits, const int32_t* exps, const float* x,
    size_t seq, size_t in_dim, size_t n_heads, size_t n_kv_heads, size_t head_dim, const float* q_norm_w,
    const float* k_norm_w, const float* cos_tab, const float* sin_tab, size_t table_rows, size_t start_pos, float eps,
    void* stream) {
  if (seq == 0 || n_heads == 0) return QASR_OK;
  const char* what = "qkv_heads_digits";
  QASR_REQUIRE(q_norm_w && k_norm_w && cos_tab && sin_tab, "qkv_heads_digits: null pointer");
  QASR_REQUIRE(seq <= 0xffffffu, "qkv_heads_digits: size too large");
  QASR_REQUIRE(n_kv_heads > 0 && n_heads <= 65536 && n_kv_heads <= 65536 && start_pos < 0x40000000u &&
                   table_rows < 0x40000000u && cache_rows < 0x40000000u,
               "qkv_heads_digits: bad sizes");
  QASR_REQUIRE(start_pos + seq <= table_rows && start_pos + seq <= cache_rows,
               "qkv_heads_digits: rows start_pos..start_pos+seq exceed the cache or the RoPE table");
  if (head_dim != 128 || !aligned16(q_norm_w) || !aligned16(k_norm_w) || !aligned16(cos_tab) || !aligned16(sin_tab))
    return fail(QASR_ERR_UNSUPPORTED, "qkv_heads_digits: head_dim must be 128, tables and gains 16-byte aligned");
  int rc = digit_gemm_checks(seq, in_dim, digits, exps, x, what);
  if (rc != QASR_OK) return rc;
  size_t n;
  QASR_REQUIRE(mul_ok(cache_rows, n_kv_heads * 128, &n), "qkv_heads_digits: size overflows");
  DigitGemm a{};
  a.n = 3;
  float* ys[3] = {q, k_cache, v_cache};
  const int8_t* ws[3] = {wq, wk, wv};
  const float* ss[3] = {sq, sk, sv};
  for (int m = 0; m < 3; ++m) {
    const size_t N = (m == 0 ? n_heads : n_kv_heads) * 128;
    rc = digit_mat_checks(ys[m], ws[m], ss[m], N, seq, in_dim, what);
    if (rc != QASR_OK) return rc;
    a.y[m] = ys[m];
    a.w[m] = ws[m];
    a.s[m] = ss[m];
    a.N[m] = (int)N;
  }
  a.digits = digits;
  a.exps = exps;
  a.x = x;
  a.T = (int)seq;
  a.K = (int)in_dim;
  a.parts = 1;
  a.heads = {k_cache, v_cache, q_norm_w, k_norm_w, cos_tab, sin_tab, (long long)start_pos, eps};
  if (!launch_digit_gemm<kDgHeads>(a, as_stream(stream)))
    return fail(QASR_ERR_UNSUPPORTED, "qkv_heads_digits: no kernel for this shape");
  return launch_status(what);
}

extern "C" int qasr_qkv_heads_digits_int8_f32(float* q, float* k_cache, float* v_cache, size_t cache_rows,
                                              const int8_t* wq, const float* sq, const int8_t* wk, const float* sk,
                                              const int8_t* wv, const float* sv, const int8_t* digits,
                                              const int32_t* exps, size_t seq, size_t in_dim, size_t n_heads,
                                              size_t n_kv_heads, size_t head_dim, const float* q_norm_w,
                                              const float* k_norm_w, const float* cos_tab, const float* sin_tab,
                                              size_t table_rows, size_t start_pos, float eps, void* stream) {
  return qasr_qkv_heads_digits_wide_int8_f32(q, k_cache, v_cache, cache_rows, wq, sq, wk, sk, wv, sv, digits, exps,
                                             nullptr, seq, in_dim, n_heads, n_kv_heads, head_dim, q_norm_w, k_norm_w,
                                             cos_tab, sin_tab, table_rows, start_pos, eps, stream);
}
