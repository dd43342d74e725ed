// fmx_attn.hip -- scaled dot-product attention of forwards with several
// tokens per sequence (prefill, chunks that continue a context), after
// rope_cache_kernel: causal, over the KV cache
// (mx::fast::scaled_dot_product_attention, server/src/model.cpp:879-882).
//
//   attn_mfma_kernel  head sizes 64 and 128: tiles of query rows against
//                     blocks of keys on the matrix cores
//   attn_kernel       other head sizes and the smallest calls: one workgroup
//                     per (token, head)
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

// ------------------------------------------------------------------ MFMA tiles

// One workgroup per (64 / KW query rows of one sequence, q head): four waves
// in groups of KW that share 16 rows, each wave with keys of its own (KW 1:
// every wave its own 16 rows and all keys; KW 4: the waves' sums are added
// at the end). Blocks of KB keys and values stream through a two-stage LDS
// ring by LDS DMA, 16-byte chunks XOR-swizzled by row.
//
// Scores come out transposed, S^T = K Q^T (v_mfma_f32_16x16x32_bf16, exact
// products, fp32 sums): lane (i16, j) holds query i16 against keys 4j + r of
// each 16-key tile, which is the B operand of O^T = V^T P^T as it stands;
// V^T comes from the row-major values by the transposing LDS read
// (ds_read_b64_tr_b16: 4 keys x 16 dimensions per 16 lanes).
//
// The softmax weights keep their 24 bits: p = hi + mid + lo, three bf16
// values cut from its fp32 pattern, three MFMAs. fp32 sums run over at most
// kFoldKeys keys and are then added to fp64 sums (as the row kernel's), one
// division and one rounding at the end. The running maximum moves only when
// a score exceeds it by more than 2^8 in weight, which the sums have the
// range for.
//
// A row that is not finite at the end (inf or NaN in the keys or values its
// tile read, those beyond its own position included, or an overflow of the
// fp32 sums) is computed again by attn_row.
//
// Bound: per 16 rows x 64 keys x 128 dimensions a wave issues 64 MFMAs (48
// of them the weights' three parts) and about 200 VALU instructions, on two
// waves per SIMD (241 VGPRs, half of a CU's LDS per workgroup). 16 heads of
// 128, one sequence of 3001 tokens: 113 us (18.4 GFLOP causal, 3750 us as
// rows), 1024 tokens 37 us (519), 512 tokens behind 1024 cached ones 47 us
// (570).
constexpr int kFoldKeys = 256;
constexpr float kMaxSlack = 8.0f;

typedef short i16x4_t __attribute__((ext_vector_type(4)));

template <int HD, int KW>
struct AttnTile {
  static constexpr int kRows = 64 / KW;              // query rows per workgroup
  static constexpr int kKeysWave = KW == 1 ? 64 : 32;  // keys per wave and block
  static constexpr int kKeys = kKeysWave * KW;       // keys per block
  static constexpr int kStage = kKeys * HD * 2 * 2;  // a block's keys and values
  static constexpr int kMerge = KW == 1 ? 0 : KW * 16 * (HD + 2) * 8;
  static constexpr int kLds = 2 * kStage > kMerge ? 2 * kStage : kMerge;
};

template <int HD>
__device__ inline bf16x8_t attn_vt(const uint8_t* sv, int key, int dt, int i16, int j) {
  // dimensions 16 dt + i16 of keys key + 4 j + (0..3) and key + 16 + 4 j + (0..3)
  constexpr int CH = HD / 8;
  union {
    i16x4_t h[2];
    bf16x8_t v;
  } u;
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int row = key + 16 * t + 4 * j + (i16 >> 2);
    const uint8_t* p = sv + row * (HD * 2) + (((2 * dt + ((i16 >> 1) & 1)) ^ (2 * (row & (CH / 2 - 1)))) << 4) +
                       (i16 & 1) * 8;
    u.h[t] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4_t*)p);
  }
  return u.v;
}

// words holding the high halves of two fp32 patterns
__device__ inline uint32_t high_halves(float lo, float hi) {
  return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}

template <int HD, int KW>
__global__ __launch_bounds__(kAttnThreads) __attribute__((amdgpu_waves_per_eu(KW == 1 ? 2 : 1)))
void attn_mfma_kernel(AttnArgs a, int B, int n_tiles) {
  using T = AttnTile<HD, KW>;
  constexpr int CH = HD / 8, RB = HD * 2, NQ = HD / 32, ND = HD / 16, NT = T::kKeysWave / 16;
  constexpr int RPP = 1024 / RB;                       // rows per 1 KB LDS DMA piece
  constexpr int PW = T::kKeys / RPP / kAttnWaves;      // pieces per wave, of keys and of values
  constexpr int kFold = kFoldKeys / T::kKeysWave;      // blocks between folds
  extern __shared__ __attribute__((aligned(16))) uint8_t s_at[];
  __shared__ uint32_t s_bad[T::kRows];

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
  const int l0 = tile * T::kRows;
  const int lw = l0 + (KW == 1 ? 16 * wave : 0);
  const int l = min(lw + i16, a.L - 1);                // rows past the sequence repeat its last
  const int p = token_pos(a.offs, a.off, b, l, a.max_seq);
  const int p_lo = token_pos(a.offs, a.off, b, min(lw, a.L - 1), a.max_seq);
  const int p_wave = token_pos(a.offs, a.off, b, min(lw + 15, a.L - 1), a.max_seq);
  const int p_hi = token_pos(a.offs, a.off, b, min(l0 + T::kRows - 1, a.L - 1), a.max_seq);
  const int64_t cbase = (cache_slot(a.slots, a.n_slots, b) * a.nkv + g) * a.max_seq * HD;
  const uint16_t* kb = a.kc + cbase;
  const uint16_t* vb = a.vc + cbase;

  // the wave's 16 rotated query rows, B operands
  bf16x8_t Q[NQ];
  const uint16_t* qrow = a.q + ((static_cast<int64_t>(b) * a.L + l) * a.nh + h) * HD + 8 * j;
#pragma unroll
  for (int q = 0; q < NQ; ++q) Q[q] = *reinterpret_cast<const bf16x8_t*>(qrow + 32 * q);

  auto issue = [&](int key0, uint8_t* st) {
#pragma unroll
    for (int pc = 0; pc < PW; ++pc) {
      const int piece = pc * kAttnWaves + wave;
      const int row = piece * RPP + lane / CH, c = lane % CH;
      const int64_t src = static_cast<int64_t>(min(key0 + row, p_hi)) * HD;  // past the last key: that key again
      __builtin_amdgcn_global_load_lds(static_cast<const void*>(kb + src + 8 * (c ^ (row & (CH - 1)))),
                                       (__attribute__((address_space(3))) void*)(st + piece * 1024), 16, 0, 0);
      __builtin_amdgcn_global_load_lds(static_cast<const void*>(vb + src + 8 * (c ^ (2 * (row & (CH / 2 - 1))))),
                                       (__attribute__((address_space(3))) void*)(st + T::kStage / 2 + piece * 1024),
                                       16, 0, 0);
    }
  };

  f32x4_t acc[ND];
  double o[ND][4], den = 0.0;
  float m = -__builtin_huge_valf();
#pragma unroll
  for (int d = 0; d < ND; ++d) {
    acc[d] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r) o[d][r] = 0.0;
  }
  // scores in units of log 2: the weights are powers of two
  const float cs = a.scale * 1.4426950408889634f;
  const int nb = p_hi / T::kKeys + 1;
  const int kw = KW == 1 ? 0 : wave * T::kKeysWave;  // the wave's keys within a block
  issue(0, s_at);
  for (int blk = 0; blk < nb; ++blk) {
    // this wave's pieces of the block have landed; behind the barrier every
    // wave's have, and every wave's reads of the other stage are done
    wait_vmcnt0();
    lds_barrier();
    if (blk + 1 < nb) issue((blk + 1) * T::kKeys, s_at + ((blk + 1) & 1) * T::kStage);
    const uint8_t* sk = s_at + (blk & 1) * T::kStage;
    const uint8_t* sv = sk + T::kStage / 2;
    const int key0 = blk * T::kKeys + kw;
    if (key0 <= p_wave) {
      f32x4_t S[NT];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        S[nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        const int row = kw + 16 * nt + i16;
#pragma unroll
        for (int q = 0; q < NQ; ++q)
          S[nt] = mfma_bf16(*reinterpret_cast<const bf16x8_t*>(sk + row * RB + (((4 * q + j) ^ (row & (CH - 1))) << 4)),
                            Q[q], S[nt]);
      }
      const bool diag = key0 + T::kKeysWave - 1 > p_lo;
      float mx = -__builtin_huge_valf();
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float x = S[nt][r] * cs;
          mx = fmaxf(mx, diag && key0 + 16 * nt + 4 * j + r > p ? -__builtin_huge_valf() : x);
        }
      if (__ballot(mx > m + kMaxSlack)) {
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float mn = fmaxf(m, mx);
        // the same factor on both sums, so its rounding cancels
        const float f = mn == m ? 1.0f : __builtin_amdgcn_exp2f(m - mn);
        m = mn;
        den *= static_cast<double>(f);
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            acc[d][r] *= f;
            o[d][r] *= static_cast<double>(f);
          }
      }
      float ds = 0.0f;
      u32x4_t P[NT / 2][3];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        float w[4], w2[4], w3[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          w[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(S[nt][r], cs, -m));
          if (diag && key0 + 16 * nt + 4 * j + r > p) w[r] = 0.0f;
          ds += w[r];
          w2[r] = w[r] - __uint_as_float(__float_as_uint(w[r]) & 0xffff0000u);
          w3[r] = w2[r] - __uint_as_float(__float_as_uint(w2[r]) & 0xffff0000u);
        }
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          P[nt / 2][0][2 * (nt & 1) + c] = high_halves(w[2 * c], w[2 * c + 1]);
          P[nt / 2][1][2 * (nt & 1) + c] = high_halves(w2[2 * c], w2[2 * c + 1]);
          P[nt / 2][2][2 * (nt & 1) + c] = high_halves(w3[2 * c], w3[2 * c + 1]);
        }
      }
      den += static_cast<double>(ds);
#pragma unroll
      for (int ks = 0; ks < NT / 2; ++ks)
#pragma unroll
        for (int d = 0; d < ND; ++d) {
          const bf16x8_t V = attn_vt<HD>(sv, kw + 32 * ks, d, i16, j);
#pragma unroll
          for (int c = 2; c >= 0; --c) acc[d] = mfma_bf16(V, __builtin_bit_cast(bf16x8_t, P[ks][c]), acc[d]);
        }
    }
    if (blk % kFold == kFold - 1 || blk == nb - 1) {
#pragma unroll
      for (int d = 0; d < ND; ++d) {
#pragma unroll
        for (int r = 0; r < 4; ++r) o[d][r] += static_cast<double>(acc[d][r]);
        acc[d] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
    }
  }
  den += __shfl_xor(den, 16);
  den += __shfl_xor(den, 32);

  bool ovf = false;
  if constexpr (KW == 1) {
    // lane (i16, j): row i16, dimensions 16 d + 4 j + r
    const double inv = 1.0 / den;
    bool bad = !(den < __builtin_huge_val());
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int r = 0; r < 4; ++r) bad |= !(fabs(o[d][r]) < __builtin_huge_val());
    const uint64_t bm = __ballot(bad) >> i16;
    bad = (bm & 0x0001000100010001ull) != 0;
    if (j == 0) s_bad[16 * wave + i16] = bad && lw + i16 < a.L;
    const bool store = !bad && lw + i16 < a.L;
    const int64_t ob = (static_cast<int64_t>(b) * a.L + l) * a.ldo + static_cast<int64_t>(h) * HD;
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      uint16_t v[4], vh[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        v[r] = f64_to_bf16(o[d][r] * inv);
        ovf |= store && bf16_f16_overflow(v[r]);
        vh[r] = static_cast<uint16_t>(bf16_to_f16_bits(v[r]));
      }
      // P8 words pair element e with e + 4: the lane with the chunk's
      // elements 0..3 writes words 0 and 1, its neighbour 2 and 3
      const bool up = j & 1;
      const uint32_t give = up ? vh[0] | (vh[1] << 16) : vh[2] | (vh[3] << 16);
      const uint32_t got = __shfl_xor(give, 16);
      const u32x2_t wh = up ? u32x2_t{(got & 0xffffu) | (static_cast<uint32_t>(vh[2]) << 16),
                                      (got >> 16) | (static_cast<uint32_t>(vh[3]) << 16)}
                            : u32x2_t{vh[0] | (got << 16), vh[1] | (got & 0xffff0000u)};
      if (store) {
        *reinterpret_cast<u32x2_t*>(a.out + ob + 16 * d + 4 * j) =
            u32x2_t{v[0] | (static_cast<uint32_t>(v[1]) << 16), v[2] | (static_cast<uint32_t>(v[3]) << 16)};
        if (a.outh) *reinterpret_cast<u32x2_t*>(a.outh + ob + 16 * d + 4 * j) = wh;
      }
    }
  } else {
    // the waves' sums through LDS; thread (row, c): dimensions 8c .. 8c + 7
    double* s_o = reinterpret_cast<double*>(s_at);
    __syncthreads();  // the last block's reads
    double* mine = s_o + (wave * 16 + i16) * (HD + 2);
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int r = 0; r < 4; ++r) mine[16 * d + 4 * j + r] = o[d][r];
    if (j == 0) {
      mine[HD] = den;
      mine[HD + 1] = static_cast<double>(m);
    }
    __syncthreads();
    const int row = tid >> 4, c = tid & 15;
    double M = -__builtin_huge_val(), n[8], dn = 0.0;
#pragma unroll
    for (int e = 0; e < 8; ++e) n[e] = 0.0;
#pragma unroll
    for (int w = 0; w < KW; ++w) M = fmax(M, s_o[(w * 16 + row) * (HD + 2) + HD + 1]);
#pragma unroll
    for (int w = 0; w < KW; ++w) {
      const double* s = s_o + (w * 16 + row) * (HD + 2);
      // a wave without keys for the row: m = -inf, f = 0
      const double f = static_cast<double>(__builtin_amdgcn_exp2f(static_cast<float>(s[HD + 1] - M)));
      dn = __builtin_fma(s[HD], f, dn);
#pragma unroll
      for (int e = 0; e < 8; ++e) n[e] = __builtin_fma(s[min(8 * c, HD - 8) + e], f, n[e]);
    }
    bool bad = !(dn < __builtin_huge_val());
#pragma unroll
    for (int e = 0; e < 8; ++e) bad |= !(fabs(n[e]) < __builtin_huge_val());
    bad = ((__ballot(bad) >> (lane & 48)) & 0xffffull) != 0;
    if (c == 0) s_bad[row] = bad && l0 + row < a.L;
    if (!bad && l0 + row < a.L && c < CH) {
      const double inv = 1.0 / dn;
      const int64_t ob = (static_cast<int64_t>(b) * a.L + l0 + row) * a.ldo + static_cast<int64_t>(h) * HD + 8 * c;
      u32x4_t v;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[e] = f64_to_bf16(n[2 * e] * inv) | (static_cast<uint32_t>(f64_to_bf16(n[2 * e + 1] * inv)) << 16);
      *reinterpret_cast<u32x4_t*>(a.out + ob) = v;
      if (a.outh) *reinterpret_cast<u32x4_t*>(a.outh + ob) = bf16_chunk_to_f16_p8(v, ovf);
    }
  }
  if (a.outh && __ballot(ovf) && lane == 0) atomicOr(a.flag, 1u);

  __syncthreads();
  for (int r = 0; r < T::kRows; ++r)
    if (s_bad[r]) {
      attn_row<1>(a, b * a.L + l0 + r, h, s_at);
      __syncthreads();
    }
}

template <int HD, int KW>
hipError_t launch_mfma(const AttnArgs& a, int B, hipStream_t stream) {
  using T = AttnTile<HD, KW>;
  const int n_tiles = (a.L + T::kRows - 1) / T::kRows;
  const size_t lds = std::max<size_t>(T::kLds, attn_row_lds(a.max_seq));
  hipLaunchKernelGGL((attn_mfma_kernel<HD, KW>), dim3(n_tiles * a.nh * B), dim3(kAttnThreads), lds, stream, a, B,
                     n_tiles);
  return hipGetLastError();
}

}  // namespace

constexpr int64_t kRowsMax = 512;
constexpr int kRowsMaxKeys = 64;
constexpr int64_t kWideTiles = 128;

hipError_t launch_attn_prefill(const AttnArgs& a, int T, hipStream_t stream) {
  if (T == 0) return hipSuccess;
  const int B = T / a.L;
  if (a.hd == 64 || a.hd == 128) {
    // Few rows over few keys run as rows: a tile's fixed part (its code,
    // the merge of the waves' sums) is then most of its time (24 tokens x 16
    // heads 5.8 us as rows, 8.7 as tiles; 64 x 16 already 12.4 and 9.2).
    // 64-row tiles from half a chip of them; below that 16-row tiles with
    // the keys over the four waves (400 tokens x 16 heads, 112 tiles of 64:
    // 20.4 us against 22.2; 512, 128 tiles: 22.8 / 23.7; 700, 176 tiles:
    // 35.6 / 28.8; 100 tokens behind 1400: 25.9 / 45.4).
    const bool rows = static_cast<int64_t>(T) * a.nh <= kRowsMax && !a.offs && a.off + a.L <= kRowsMaxKeys;
    const bool wide = static_cast<int64_t>((a.L + 63) / 64) * a.nh * B >= kWideTiles;
    if (!rows) {
      if (a.hd == 128) return wide ? launch_mfma<128, 1>(a, B, stream) : launch_mfma<128, 4>(a, B, stream);
      return wide ? launch_mfma<64, 1>(a, B, stream) : launch_mfma<64, 4>(a, B, stream);
    }
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
