// fmx_attn.hip -- scaled dot-product attention of forwards with several
// tokens per sequence (prefill, chunks that continue a context), after
// rope_cache_kernel: causal, over the KV cache
// (mx::fast::scaled_dot_product_attention, server/src/model.cpp:879-882).
//
//   attn_tile_kernel  head sizes 64 and 128: tiles of 16 query rows against
//                     tiles of 16 keys on the matrix cores
//   attn_kernel       other head sizes and the smallest calls: one workgroup
//                     per (token, head)
//
// Both form the same sums in the same order, so a row has the same bits on
// either.
//
// Single-token forwards: attn_split_kernel (fmx_model.hip).
#include <algorithm>

#include "fmx_dev.hpp"
#include "fmx_model_kernels.hpp"

namespace fmx {

namespace {

// ------------------------------------------------------------------ one row

// The row of (token t = b * L + l, q head h), by one workgroup: keys
// 0 .. p of kv head g = h / (nh / nkv), p = offset(b) + l (causal).
//   s_j = scale * sum_d q_d k_jd   (fp32, d in order: exact bf16 products)
//   e_j = exp(s_j - max s)         (fp64, the deterministic exp)
//   out_d = sum_j e_j v_jd / sum_j e_j, both sums in fp64 over four
//           contiguous quarters of the keys (keys in order within a quarter,
//           fma), the quarter sums added in order; rounded once to bf16
// Scores: a thread per key; the weighted sum: wave w takes quarter w, its
// lanes pairs of dimensions. s_at: attn_row_lds(max_seq) bytes of LDS.
constexpr int kAttnThreads = 256;
constexpr int kAttnWaves = kAttnThreads / kWave;
constexpr int kAttnBatch = 32;  // keys whose value words are loaded together
constexpr int64_t kLdsBytes = 160 * 1024;  // per CU

size_t attn_row_lds(int64_t max_seq) {
  return static_cast<size_t>(align_up(max_seq * 12, 8) + 8 * kAttnWaves * (kAttnMaxHd + 1) +
                             4 * (kAttnMaxHd + kAttnWaves));
}

template <int PAIRS>
__device__ __attribute__((always_inline)) void attn_row(const AttnArgs& a, int t, int h, uint8_t* s_at) {
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  double* s_e = reinterpret_cast<double*>(s_at);
  float* s_s = reinterpret_cast<float*>(s_at + static_cast<size_t>(a.max_seq) * 8);
  double(*s_num)[kAttnMaxHd] = reinterpret_cast<double(*)[kAttnMaxHd]>(s_at + align_up(a.max_seq * 12, 8));
  double* s_den = &s_num[kAttnWaves][0];
  float* s_q = reinterpret_cast<float*>(s_den + kAttnWaves);
  float* s_max = s_q + kAttnMaxHd;
  const int b = t / a.L, l = t - b * a.L;
  const int p = token_pos(a.offs, a.off, b, l, a.max_seq);
  const int nk = p + 1;
  const int rep = a.nh / a.nkv, g = h / rep;
  const int64_t cbase = (cache_slot(a.slots, a.n_slots, b) * a.nkv + g) * a.max_seq * a.hd;
  uint16_t* kb = a.kc + cbase;
  uint16_t* vb = a.vc + cbase;
  const uint16_t* qrow = a.q + (static_cast<int64_t>(t) * a.nh + h) * a.hd;
  for (int d = tid; d < a.hd; d += kAttnThreads) s_q[d] = bf16_to_f32(qrow[d]);
  __syncthreads();

  // this wave's quarter of the keys for the weighted sum below; its first
  // kAttnBatch value words are loaded now, so that their latency overlaps
  // the scores
  const int quarter = (nk + kAttnWaves - 1) / kAttnWaves;
  const int j0 = min(wave * quarter, nk), j1 = min(j0 + quarter, nk);
  const int npair = a.hd / 2;
  const int jg = j1;
  // lanes past the head's pairs read pair 0 (in bounds) and discard it
  uint32_t vv[kAttnBatch][PAIRS];
  int prl[PAIRS];
#pragma unroll
  for (int i = 0; i < PAIRS; ++i) prl[i] = (lane + kWave * i) < npair ? lane + kWave * i : 0;
  auto load_values = [&](int jb) {
#pragma unroll
    for (int u = 0; u < kAttnBatch; ++u) {
      const uint32_t* vr = reinterpret_cast<const uint32_t*>(vb + static_cast<int64_t>(min(jb + u, jg - 1)) * a.hd);
#pragma unroll
      for (int i = 0; i < PAIRS; ++i) vv[u][i] = vr[prl[i]];
    }
  };
  if (j0 < jg) load_values(j0);

  // scores, a thread per key
  float m = -__builtin_huge_valf();
  for (int jk = tid; jk < nk; jk += kAttnThreads) {
    // the key row's chunks are loaded 16 at a time, then used in order
    float acc = 0.0f;
    const u32x4_t* kr = reinterpret_cast<const u32x4_t*>(kb + static_cast<int64_t>(jk) * a.hd);
    const int nch = a.hd / 8;
    for (int c0 = 0; c0 < nch; c0 += 16) {
      u32x4_t kv[16];
#pragma unroll
      for (int c = 0; c < 16; ++c) kv[c] = kr[min(c0 + c, nch - 1)];
#pragma unroll
      for (int c = 0; c < 16; ++c) {
        if (c0 + c < nch) {
#pragma unroll
          for (int mm = 0; mm < 4; ++mm) {
            acc = __builtin_fmaf(s_q[8 * (c0 + c) + 2 * mm], bf16_to_f32(kv[c][mm] & 0xffffu), acc);
            acc = __builtin_fmaf(s_q[8 * (c0 + c) + 2 * mm + 1], bf16_to_f32(kv[c][mm] >> 16), acc);
          }
        }
      }
    }
    const float sc = acc * a.scale;
    s_s[jk] = sc;
    m = fmaxf(m, sc);
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
  if (lane == 0) s_max[wave] = m;
  __syncthreads();
  m = s_max[0];
#pragma unroll
  for (int w = 1; w < kAttnWaves; ++w) m = fmaxf(m, s_max[w]);
  for (int jk = tid; jk < nk; jk += kAttnThreads)
    s_e[jk] = exp_det(static_cast<double>(s_s[jk]) - static_cast<double>(m));
  __syncthreads();

  // weighted sum: wave w over keys [j0, j1), lane over dimension pairs
  // (2 pr, 2 pr + 1), pr = lane + 64 i; the value words of kAttnBatch keys
  // are loaded together, then used in key order
  double num[PAIRS][2], den = 0.0;
#pragma unroll
  for (int i = 0; i < PAIRS; ++i) num[i][0] = num[i][1] = 0.0;
  for (int jb = j0; jb < jg; jb += kAttnBatch) {
    if (jb != j0) load_values(jb);
#pragma unroll
    for (int u = 0; u < kAttnBatch; ++u) {
      if (jb + u < jg) {
        const double e = s_e[jb + u];
        den += e;
#pragma unroll
        for (int i = 0; i < PAIRS; ++i) {
          num[i][0] = __builtin_fma(e, static_cast<double>(bf16_to_f32(vv[u][i] & 0xffffu)), num[i][0]);
          num[i][1] = __builtin_fma(e, static_cast<double>(bf16_to_f32(vv[u][i] >> 16)), num[i][1]);
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < PAIRS; ++i) {
    const int pr = lane + kWave * i;
    if (pr < npair) {
      s_num[wave][2 * pr] = num[i][0];
      s_num[wave][2 * pr + 1] = num[i][1];
    }
  }
  if (lane == 0) s_den[wave] = den;
  __syncthreads();

  bool ovf = false;
  for (int d = tid; d < a.hd; d += kAttnThreads) {
    double nsum = s_num[0][d], dsum = s_den[0];
#pragma unroll
    for (int w = 1; w < kAttnWaves; ++w) {
      nsum += s_num[w][d];
      dsum += s_den[w];
    }
    const uint16_t o = f64_to_bf16(nsum / dsum);
    const int64_t oc = static_cast<int64_t>(h) * a.hd + d;
    a.out[static_cast<int64_t>(t) * a.ldo + oc] = o;
    if (a.outh) {
      ovf = ovf || bf16_f16_overflow(o);
      a.outh[static_cast<int64_t>(t) * a.ldo + ((oc & ~7) | p8_slot(oc & 7))] =
          static_cast<uint16_t>(bf16_to_f16_bits(o));
    }
  }
  if (a.outh && __ballot(ovf) && lane == 0) atomicOr(a.flag, 1u);
}

template <int PAIRS>
__global__ __launch_bounds__(kAttnThreads) void attn_kernel(AttnArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t s_at[];
  attn_row<PAIRS>(a, blockIdx.x, blockIdx.y, s_at);
}

// ------------------------------------------------------------------ tiles

// One workgroup per (16 query rows of one sequence, q head): the sums of
// attn_row, bit for bit, on the matrix cores, whose fp32 and fp64 products
// over K = 4 add their terms one after the other, each a fused multiply-add
// (measured against fma chains, subnormal results among them):
//   scores S^T = K Q^T by v_mfma_f32_16x16x4_f32, dimensions in order, then
//     times scale;
//   weights by exp_det's steps;
//   sums O^T += V^T P^T by v_mfma_f64_16x16x4_f64, keys in order, den by
//     v_mfma_f64_4x4x4_4b_f64 with ones.
// Wave w has quarter w of the keys, as in attn_row. The rows' quarters begin
// up to 12 keys apart: the wave runs over the keys of any of its rows, and
// the weight of a key outside a row's own quarter is 0, which leaves the
// row's sums as they are.
//
// The weights need the row's largest score first. A pass of bf16 products
// (v_mfma_f32_16x16x32_bf16, an eighth of the score steps' time) finds the
// key that has it, whose score is then formed like all others; the second
// pass checks that no score is larger, and the tile is done again behind a
// pass of fp32 scores where one is (a near tie that the bf16 products' order
// of summation decided otherwise).
//
// Row 4j + r of a 16-key score tile is key 4r + j, so lane (i16, j) ends up
// with query i16 and key 4r + j in register r: the B operand of step r of the
// value products as it stands. Nothing passes through LDS but the maxima and
// the quarter sums at the end: a lane loads 16 bytes of a key (chunk 4i + j
// of its 8-dimension chunks), pairs dimensions d and d + 4 and exchanges the
// pairs with the three other lanes of the key (4 x 4 transposes by
// v_permlane32_swap and v_permlane16_swap), which leaves it dimension 4s + j
// of every step s. Values: DT dimensions DT i16 + dt of a key per lane, so
// row i16 of dimension tile dt.
//
// A row that is not finite at the end (inf or NaN in the keys or values its
// tile read, those beyond its own position included) is computed again by
// attn_row.
//
// Bound by the matrix cores' fp64 and fp32 rates (58 and 155 TFLOP/s,
// measured): one sequence of 3001 tokens, 16 heads of 128, 18.4 GFLOP of
// each, 433 us, took 697-751 us (averages on several boxes; the row kernel
// 3300-3440). Without the exps it was 75 us less, without the loads 75,
// without the value products 260; the rest is the scores, whose operands'
// preparation (2 VALU instructions per step, 3 with the exchange) is not
// hidden behind the fp32 products. With the first pass in fp32 870-890 us.
// 1024 tokens 119 us (495 as rows), 512 tokens behind 1024 cached ones 138
// us (552). Two key tiles at a time, or the next tile's score steps between
// the value products, gave nothing: two waves per SIMD cover the chains.
constexpr int kTileRows = 16;

// exp_det of r <= 0 or NaN without branches, so that several run side by
// side (r > 0: some value)
__device__ inline double exp_neg(double r) {
  const double e = exp_steps(r, fmax(rint(r * kExpLog2e), -1000.0));
  return r < -690.0 ? 0.0 : e;
}

typedef double f64x4_t __attribute__((ext_vector_type(4)));

template <int HD>
struct AttnTile {
  static constexpr int NI = HD / 32;       // 16-byte loads of a lane per key tile
  static constexpr int NC = HD / 8;        // 8-dimension chunks: two score steps each
  static constexpr int DT = HD / 16;       // 16-dimension tiles
  static constexpr int kRow = HD + 2;      // doubles of a row's sums: dimensions, den, (padding)
  static constexpr int kLds = kAttnWaves * kTileRows * kRow * 8;
};

// Raw chunks 4i + j of a row to its dimension pairs (8c + j, 8c + 4 + j),
// c = 0 .. NC - 1, j = lane / 16.
template <int NI>
__device__ inline void attn_pairs(const u32x4_t (&raw)[NI], uint32_t (&pr)[4 * NI]) {
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    // bytes 0, 1 of the first word below, bytes 4, 5: 2, 3 of the second
    uint32_t r0 = __builtin_amdgcn_perm(raw[i][2], raw[i][0], 0x05040100u);
    uint32_t r1 = __builtin_amdgcn_perm(raw[i][2], raw[i][0], 0x07060302u);
    uint32_t r2 = __builtin_amdgcn_perm(raw[i][3], raw[i][1], 0x05040100u);
    uint32_t r3 = __builtin_amdgcn_perm(raw[i][3], raw[i][1], 0x07060302u);
    const auto a = __builtin_amdgcn_permlane32_swap(r0, r2, false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(r1, r3, false, false);
    const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
    const auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    pr[4 * i] = c[0];
    pr[4 * i + 1] = c[1];
    pr[4 * i + 2] = d[0];
    pr[4 * i + 3] = d[1];
  }
}

__device__ inline float pair_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ inline float pair_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

template <int HD>
__global__ __launch_bounds__(kAttnThreads) __attribute__((amdgpu_waves_per_eu(2)))
void attn_tile_kernel(AttnArgs a, int B, int n_tiles) {
  using T = AttnTile<HD>;
  constexpr int NI = T::NI, NC = T::NC, DT = T::DT;
  extern __shared__ __attribute__((aligned(16))) uint8_t s_at[];
  __shared__ uint32_t s_bad[kTileRows];
  __shared__ float s_max[kAttnWaves][kTileRows];
  __shared__ int s_key[kAttnWaves][kTileRows];
  __shared__ uint32_t s_over[kAttnWaves];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i16 = lane & 15, j = lane >> 4;
  // block -> (row tile, sequence, head): the heads of one kv group sit 8 or
  // nkv blocks apart, so where nkv is a multiple of the 8 XCDs a group's
  // keys and values are read into one L2; the last rows, which see the most
  // keys, go first
  const int nhb = a.nh * B;
  const int tile = n_tiles - 1 - static_cast<int>(blockIdx.x) / nhb;
  const int bh = static_cast<int>(blockIdx.x) % nhb;
  const int b = bh / a.nh, hi = bh - b * a.nh;
  const int g = hi % a.nkv, h = g * (a.nh / a.nkv) + hi / a.nkv;
  const int l0 = tile * kTileRows;
  const int l = min(l0 + i16, a.L - 1);  // rows past the sequence repeat its last
  const int p = token_pos(a.offs, a.off, b, l, a.max_seq);
  const int p_lo = token_pos(a.offs, a.off, b, l0, a.max_seq);
  const int p_hi = token_pos(a.offs, a.off, b, min(l0 + kTileRows - 1, a.L - 1), a.max_seq);
  const int64_t cbase = (cache_slot(a.slots, a.n_slots, b) * a.nkv + g) * a.max_seq * HD;
  const uint16_t* kb = a.kc + cbase;
  const uint16_t* vb = a.vc + cbase;

  auto load_key = [&](u32x4_t (&raw)[NI], int key) {
    const uint16_t* src = kb + static_cast<int64_t>(key) * HD + 8 * j;
#pragma unroll
    for (int i = 0; i < NI; ++i) raw[i] = *reinterpret_cast<const u32x4_t*>(src + 32 * i);
  };
  // keys key0 .. key0 + 15 (past the last key: that key again)
  const int krow = 4 * (i16 & 3) + (i16 >> 2);
  auto load_keys = [&](u32x4_t (&raw)[NI], int key0) { load_key(raw, min(key0 + krow, p_hi)); };
  uint32_t vw[4][DT / 2];
  auto load_values = [&](int key0) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const uint16_t* src = vb + static_cast<int64_t>(min(key0 + 4 * r + j, p_hi)) * HD + DT * i16;
      if constexpr (DT == 8) {
        const u32x4_t w = *reinterpret_cast<const u32x4_t*>(src);
#pragma unroll
        for (int q = 0; q < 4; ++q) vw[r][q] = w[q];
      } else {
        const u32x2_t w = *reinterpret_cast<const u32x2_t*>(src);
#pragma unroll
        for (int q = 0; q < 2; ++q) vw[r][q] = w[q];
      }
    }
  };

  u32x4_t raw[NI], qr[NI];
  load_keys(raw, wave * 16);
  const uint16_t* qrow = a.q + ((static_cast<int64_t>(b) * a.L + l) * a.nh + h) * HD + 8 * j;
#pragma unroll
  for (int i = 0; i < NI; ++i) qr[i] = *reinterpret_cast<const u32x4_t*>(qrow + 32 * i);
  float Q[2 * NC];  // query i16, dimensions 4s + j
  {
    uint32_t qp[4 * NI];
    attn_pairs<NI>(qr, qp);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      Q[2 * c] = pair_lo(qp[c]);
      Q[2 * c + 1] = pair_hi(qp[c]);
    }
  }
  auto scores = [&](const u32x4_t (&r)[NI]) {
    uint32_t kp[4 * NI];
    attn_pairs<NI>(r, kp);
    f32x4_t S = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      S = __builtin_amdgcn_mfma_f32_16x16x4f32(pair_lo(kp[c]), Q[2 * c], S, 0, 0, 0);
      S = __builtin_amdgcn_mfma_f32_16x16x4f32(pair_hi(kp[c]), Q[2 * c + 1], S, 0, 0, 0);
    }
    return S;
  };

  // this wave's quarter: row i16's keys [j0, j1), any row's [k_lo, k_hi),
  // every row's [full_lo, full_hi)
  const int quarter = (p + kAttnWaves) / kAttnWaves;
  const int j0 = min(wave * quarter, p + 1), j1 = min(j0 + quarter, p + 1);
  auto row_min = [](int v) {
#pragma unroll
    for (int o = 8; o >= 1; o >>= 1) v = min(v, __shfl_xor(v, o));
    return __builtin_amdgcn_readfirstlane(v);
  };
  const int k_lo = row_min(j0), k_hi = -row_min(-j1);
  const int full_lo = -row_min(-j0), full_hi = row_min(j1);

  double* s_o = reinterpret_cast<double*>(s_at);
  for (bool exact = false;; exact = true) {
    // 1. each row's largest score; the waves take every fourth key tile
    float m = -__builtin_huge_valf();
    if (!exact) {
      // that of the key whose bf16 products sum up largest
      int mk = 0;
      for (int key0 = wave * 16; key0 <= p_hi; key0 += 16 * kAttnWaves) {
        f32x4_t S = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < NI; ++i)
          S = mfma_bf16(__builtin_bit_cast(bf16x8_t, raw[i]), __builtin_bit_cast(bf16x8_t, qr[i]), S);
        load_keys(raw, key0 + 16 * kAttnWaves);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int key = key0 + 4 * r + j;
          const bool up = S[r] > m && key <= p;
          m = up ? S[r] : m;
          mk = up ? key : mk;
        }
      }
#pragma unroll
      for (int o = 16; o <= 32; o *= 2) {
        const float om = __shfl_xor(m, o);
        const int ok = __shfl_xor(mk, o);
        mk = om > m ? ok : mk;
        m = fmaxf(m, om);
      }
      if (j == 0) {
        s_max[wave][i16] = m;
        s_key[wave][i16] = mk;
      }
      lds_barrier();
      m = s_max[0][i16];
      mk = s_key[0][i16];
#pragma unroll
      for (int w = 1; w < kAttnWaves; ++w) {
        mk = s_max[w][i16] > m ? s_key[w][i16] : mk;
        m = fmaxf(m, s_max[w][i16]);
      }
      // a tile of the rows' keys: row i16's score is on its diagonal
      load_key(raw, mk);
      const f32x4_t S = scores(raw);
      m = i16 >> 2 == j ? (i16 & 2 ? (i16 & 1 ? S[3] : S[2]) : (i16 & 1 ? S[1] : S[0])) * a.scale
                        : -__builtin_huge_valf();
      m = fmaxf(m, __shfl_xor(m, 16));
      m = fmaxf(m, __shfl_xor(m, 32));
    } else {
      for (int key0 = wave * 16; key0 <= p_hi; key0 += 16 * kAttnWaves) {
        load_keys(raw, key0);
        const f32x4_t S = scores(raw);
#pragma unroll
        for (int r = 0; r < 4; ++r) m = fmaxf(m, key0 + 4 * r + j > p ? -__builtin_huge_valf() : S[r] * a.scale);
      }
      m = fmaxf(m, __shfl_xor(m, 16));
      m = fmaxf(m, __shfl_xor(m, 32));
      if (j == 0) s_max[wave][i16] = m;
      lds_barrier();
#pragma unroll
      for (int w = 0; w < kAttnWaves; ++w) m = fmaxf(m, s_max[w][i16]);
    }

    // 2. the wave's quarter
    load_keys(raw, k_lo);
    load_values(k_lo);
    const double md = static_cast<double>(m);
    float seen = m;
    f64x4_t acc[DT];
    double den = 0.0;
#pragma unroll
    for (int d = 0; d < DT; ++d) acc[d] = f64x4_t{0.0, 0.0, 0.0, 0.0};
    for (int key0 = k_lo; key0 < k_hi; key0 += 16) {
      f32x4_t S = scores(raw);
      load_keys(raw, key0 + 16);
#pragma unroll
      for (int r = 0; r < 4; ++r) S[r] *= a.scale;
      double e[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) e[r] = exp_neg(static_cast<double>(S[r]) - md);
      if (key0 < full_lo || key0 + 16 > full_hi) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int key = key0 + 4 * r + j;
          const bool own = key >= j0 && key < j1;
          e[r] = own ? e[r] : 0.0;
          S[r] = own ? S[r] : m;
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) seen = fmaxf(seen, S[r]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        den = __builtin_amdgcn_mfma_f64_4x4x4f64(1.0, e[r], den, 0, 0, 0);
#pragma unroll
        for (int d = 0; d < DT; ++d) {
          const uint32_t w = vw[r][d / 2];
          acc[d] = __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(d & 1 ? pair_hi(w) : pair_lo(w)), e[r],
                                                        acc[d], 0, 0, 0);
        }
      }
      load_values(key0 + 16);
    }
    double* mine = s_o + (wave * kTileRows + i16) * T::kRow;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int d = 0; d < DT; ++d) mine[DT * (j + 4 * r) + d] = acc[d][r];
    if (j == 0) mine[HD] = den;
    const bool over = __ballot(seen > m) != 0;
    if (lane == 0) s_over[wave] = over;
    lds_barrier();
    if (exact || !(s_over[0] | s_over[1] | s_over[2] | s_over[3])) break;
  }

  // 3. the quarter sums, added in order; thread (row, c): dimensions 8c .. 8c + 7
  const int row = tid >> 4, c = tid & 15;
  const double* s = s_o + row * T::kRow;
  constexpr int W = kTileRows * T::kRow;
  const double dn = ((s[HD] + s[W + HD]) + s[2 * W + HD]) + s[3 * W + HD];
  double n[8];
  bool bad = !(dn < __builtin_huge_val());
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int d = min(8 * c, HD - 8) + e;
    n[e] = ((s[d] + s[W + d]) + s[2 * W + d]) + s[3 * W + d];
    bad |= !(fabs(n[e]) < __builtin_huge_val());
  }
  bad = ((__ballot(bad) >> (lane & 48)) & 0xffffull) != 0;
  if (c == 0) s_bad[row] = bad && l0 + row < a.L;
  bool ovf = false;
  if (!bad && l0 + row < a.L && c < NC) {
    const int64_t ob = (static_cast<int64_t>(b) * a.L + l0 + row) * a.ldo + static_cast<int64_t>(h) * HD + 8 * c;
    u32x4_t v;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[e] = f64_to_bf16(n[2 * e] / dn) | (static_cast<uint32_t>(f64_to_bf16(n[2 * e + 1] / dn)) << 16);
    *reinterpret_cast<u32x4_t*>(a.out + ob) = v;
    if (a.outh) *reinterpret_cast<u32x4_t*>(a.outh + ob) = bf16_chunk_to_f16_p8(v, ovf);
  }
  if (a.outh && __ballot(ovf) && lane == 0) atomicOr(a.flag, 1u);

  __syncthreads();
  for (int r = 0; r < kTileRows; ++r)
    if (s_bad[r]) {
      attn_row<1>(a, b * a.L + l0 + r, h, s_at);
      __syncthreads();
    }
}

template <int HD>
hipError_t launch_tiles(const AttnArgs& a, int B, hipStream_t stream) {
  const int n_tiles = (a.L + kTileRows - 1) / kTileRows;
  const size_t lds = std::max<size_t>(AttnTile<HD>::kLds, attn_row_lds(a.max_seq));
  hipLaunchKernelGGL((attn_tile_kernel<HD>), dim3(n_tiles * a.nh * B), dim3(kAttnThreads), lds, stream, a, B, n_tiles);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_attn_prefill(const AttnArgs& a, int T, hipStream_t stream) {
  if (T == 0) return hipSuccess;
  const int B = T / a.L;
  if (a.hd == 64 || a.hd == 128) {
    // Few rows run as rows: a tile's four waves walk a quarter of the keys
    // each, a row has four waves of its own. The line is where the row
    // kernel's workgroups no longer run at the same time (three per CU by
    // registers, fewer by LDS), for head size 64, whose tiles take 0.6 of the
    // time, a third of that (us, rows / tiles, at keys 0 / 256 / 1024 / 3000
    // before the call: 32 tokens x 16 heads of 128 7 / 14, 19 / 26, 48 / 59,
    // 119 / 143; 48 x 16 8 / 15, 22 / 26, 62 / 60, 161 / 146; 64 x 16 13 / 15,
    // 31 / 26, 82 / 60, 206 / 146; heads of 64, 8 x 16 6 / 10, 13 / 16, 32 /
    // 36, 78 / 85; 24 x 16 7 / 10, 16 / 16, 43 / 36, 108 / 87). Over few keys
    // rows are faster up to two rounds of them, one round for head size 64
    // (96 x 16 of 128 at 0 / 32 / 64 keys before the call 16 / 17, 18 / 18,
    // 22 / 20; 48 x 16 of 64 at 0 / 64 / 128 8 / 11, 10 / 13, 13 / 15; 64 x 16
    // 12 / 12, 14 / 13, 19 / 14).
    // Rows are also faster where a tile has only two of them, over few keys
    // three (96 sequences x 16 heads of 128 over 100 / 500 / 2000 keys, 2 rows
    // 38 / 60, 139 / 154, 519 / 537; 3 rows 54 / 60, 189 / 151, 720 / 529;
    // heads of 64, 2 rows 32 / 42, 97 / 91, 374 / 319).
    const bool hd128 = a.hd == 128;
    const int64_t n = static_cast<int64_t>(T) * a.nh;
    const int64_t tiles = static_cast<int64_t>((a.L + kTileRows - 1) / kTileRows) * a.nh * B;
    const int64_t resident = 256 * std::min<int64_t>(3, kLdsBytes / attn_row_lds(a.max_seq));
    // With the offsets on the device the keys are not known here and taken to
    // be few (40 tokens x 16 heads of 128 in a cache of 4096, rows / tiles: 60
    // keys 11 / 14, 540 43 / 33, 2040 126 / 96).
    const bool few_keys = a.offs || a.off + a.L <= (hd128 ? 128 : 192);
    const int64_t most = hd128 ? (few_keys ? 2 * resident : resident) : (few_keys ? resident : resident / 3);
    const int per_tile = (hd128 ? 3 : 2) + (few_keys ? 1 : 0);  // rows that take a tile's time
    if (n > most && n >= per_tile * tiles) return hd128 ? launch_tiles<128>(a, B, stream) : launch_tiles<64>(a, B, stream);
  }
  const dim3 grid(T, a.nh);
  const size_t lds = attn_row_lds(a.max_seq);
  if (a.hd <= 128)
    hipLaunchKernelGGL((attn_kernel<1>), grid, dim3(kAttnThreads), lds, stream, a);
  else
    hipLaunchKernelGGL((attn_kernel<2>), grid, dim3(kAttnThreads), lds, stream, a);
  return hipGetLastError();
}

}  // namespace fmx
