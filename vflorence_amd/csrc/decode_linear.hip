// Decode-step linear layers on the matrix cores (gfx950), 16-bit inputs and output,
// fp32 sums:
//
//   y[m][n] = sum_k x[m][k] * w[n][k] + bias[n]        (w: nn.Linear's [out, in])
//
// for the few hundred token rows of a decode step times the decoder's projection
// weights (vflorence/models/bart.py:111,114,142,146: the fused q|k|v, the attention
// output and the cross-attention query projections).  Each step streams every weight
// from HBM once (a decoder's weights exceed the last-level cache), so the time goes to
// memory round trips, not arithmetic: a GEMM that walks K in a loop pays one round
// trip per K step.  Here a workgroup owns an output tile (32 features x 32 tokens; others
// by size, see pick_tile) and splits K over its 8 waves.  Each wave loads the operands of
// up to 4 K steps of 32 in one batch, so K <= 1024 costs one round trip; a longer K range is
// walked in batches of 2 steps with the next batch in flight while one is multiplied (a 32 x 16
// tile: up to 16 steps in one batch, K <= 4096, then batches of 4).  The waves' partial tiles
// are summed through LDS in the order of a 3-level tree (waves w and w + 4 first, then (s0 +
// s2) + (s1 + s3)), and the waves then add the bias and store a 16 x 16 quarter each.
//
// Operand order.  The product per 32-wide K step is mfma_f32_16x16x32 with A = 16
// weight rows (features) and B = 16 token rows, giving D[feature][token]; a lane's four
// D registers are four consecutive features of one token -- one 8-byte store.  Lane l
// holds row l % 16 and k = 8 (l / 16) .. +7 of both operands, so neighbouring lanes read
// rows 2 KB apart.  Loaded that way, every 16-byte chunk is a separate cache access.
// The operands are therefore brought in contiguously instead:
// - The weight is re-laid out once (vfl_pack_linear_weight) into 1 KB blocks of 16
//   rows x 32 k, each stored in lane order: block (r, c) holds, for lane l, row
//   16 r + l % 16 and k = 32 c + 8 (l / 16) .. +7 at byte 16 l.  One wave load is then
//   one contiguous KB.  Rows are padded with zeros to a multiple of 32.
// - Activation rows are read as 64-byte runs (lanes 4 i .. 4 i + 3 take row i) and
//   moved into operand order with ds_bpermute (lane l takes lane 4 (l % 16) + l / 16).
//   Activations that one call produces for another can skip that: the feed-forward
//   block (bart.py:192-201, fc2(gelu(fc1(h)))) runs fc1 with the exact GELU in its
//   epilogue and its output written in the packed layout (token rows as the weight's
//   rows), which fc2 then reads as one contiguous KB per wave load.
#include "common.h"
#include "mfma_ops.h"

namespace vfl {

constexpr int LIN_WAVES = 8;   // waves splitting K
constexpr int LIN_TILE = 32;   // features and tokens per workgroup
constexpr int LIN_BATCH = 4;   // K steps whose operands are loaded together
constexpr int LIN_PIPE_BATCH = 2;  // the same when two batches are in flight
constexpr int LIN_K_MULTIPLE = 32 * LIN_WAVES;
constexpr int LIN_BLOCK = 16 * 32;  // elements of one packed 16-row x 32-k weight block

__host__ __device__ constexpr int64_t packed_rows(int64_t out_features) {
  return (out_features + LIN_TILE - 1) / LIN_TILE * LIN_TILE;
}

// One thread per 16-byte chunk of the packed weight: chunk t is lane t % 64 of block
// t / 64 = (row block r, k block c).
__global__ __launch_bounds__(256) void pack_linear_weight_kernel(
    const uint16_t *__restrict__ w, int64_t ldw, int N, int K, uint16_t *__restrict__ packed,
    int64_t chunks) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= chunks) return;
  const int l = (int)(t & 63);
  const int64_t blk = t >> 6;
  const int ks = K / 32;
  const int64_t r = blk / ks;
  const int c = (int)(blk % ks);
  const int64_t row = 16 * r + (l & 15);
  uint4 v = make_uint4(0, 0, 0, 0);
  if (row < N) v = *reinterpret_cast<const uint4 *>(w + row * ldw + 32 * c + 8 * (l >> 4));
  *reinterpret_cast<uint4 *>(packed + t * 8) = v;
}

// Element offset of (row m, column k) in a packed [rows][K] array (weight or activation).
__device__ __forceinline__ int64_t packed_offset(int m, int k, int K) {
  return ((int64_t)(m / 16) * (K / 32) + k / 32) * LIN_BLOCK + (16 * ((k % 32) / 8) + m % 16) * 8 +
         k % 8;
}

// torch's exact GELU (x / 2 * (1 + erf(x / sqrt(2)))) in fp32 on a value already rounded to
// the element type, as the separate activation kernel would see it.
template <int DT> __device__ __forceinline__ float gelu_of_stored(float v) {
  const float x = Mfma<DT>::widen(Mfma<DT>::narrow(v));
  return x * 0.5f * (1.0f + erff(x * 0.70710678118654752440f));
}

// Deferred LayerNorm across the decoder's projections.  BART's sublayers end in
// h' = LN(h + y) (post-LN, bart.py:259-261); a separate residual + LayerNorm launch per
// sublayer costs ~5 us in a decode step's graph, more than its bytes.  Instead:
// - the sublayer's output projection (LIN_RESIDUAL) stores the pre-norm sum
//   v = round(round(acc + bias) + h) -- the value the LayerNorm kernel normalizes -- and,
//   per row and 32-feature tile, the tile's mean and sum of squared deviations;
// - the projections that read h' (LIN_NORM_IN) multiply v itself, with LayerNorm's
//   weight folded into their packed weight (W' = W diag(gamma), rounded) and its bias
//   into theirs (b' = b + W beta), and finish in the epilogue:
//   y = rstd_r (acc - mean_r u[n]) + b'[n] with u[n] = sum_k W'[n][k];
// - the residual of the next sublayer is h' itself, normalized element by element in
//   that sublayer's output projection (or by vfl_layer_norm_apply).
// A row's mean and 1/std combine its T tiles: mean = sum_t m_t / T,
// M2 = sum_t M2_t + 32 sum_t (m_t - mean)^2, rstd = 1 / sqrt(M2 / (32 T) + eps).
constexpr int LIN_PLAIN = 0, LIN_NORM_IN = 1, LIN_RESIDUAL = 2;
constexpr int LIN_STAT_TILE = 32;   // features per statistics tile

struct LinNorm {
  const float2 *x_stats;  // LIN_NORM_IN: [rows][K / 32] of x
  const float *u, *fbias; // LIN_NORM_IN: [N] fp32
  float eps;
  bool vec4;              // LIN_NORM_IN: u and fbias 16-byte aligned
  const uint16_t *res;    // LIN_RESIDUAL: h, [rows][N] with row stride res_stride
  int64_t res_stride;
  const float2 *res_stats;  // null: h is plain; else h = LN(res) with these statistics
  const uint16_t *res_gamma, *res_beta;
  float res_eps;
  float2 *y_stats;        // LIN_RESIDUAL: [rows][N / 32] of the stored v
};

// The workgroup's rows' means and 1/stds from their T tiles' (mean, M2) at
// st[row * T + t]: thread (row r = tid / TPR, j = tid % TPR) takes tiles j, j + 16, ... and,
// where 8 threads share a row, j + 8, j + 24, ...; the threads of a row (within one DPP row
// of a wave) combine them in an order that does not depend on TPR.
// Requested after the main loop, so the loads' latency overlaps the partial-tile
// reduction; results in s_ms[r] = (mean, rstd) before the reduction's last barrier.
template <int TPR> struct RowStatLoads {
  static_assert(TPR == 16 || TPR == 8, "16 partial sums per row");
  static constexpr int H = 16 / TPR;
  float2 p[H][2];
  __device__ __forceinline__ void issue(const float2 *st, int T, int m0, int M) {
    const int r = (int)threadIdx.x / TPR, j0 = (int)threadIdx.x % TPR;
    const float2 *row = st + (int64_t)min(m0 + r, M - 1) * T;
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int t = j0 + TPR * h + 16 * i;
        p[h][i] = t < T ? row[t] : make_float2(0.f, 0.f);
      }
  }
  __device__ __forceinline__ static float total(const float (&s)[H]) {
    float x = group_sum<TPR>(s[0]);
    if constexpr (H == 2) x += group_sum<TPR>(s[1]);
    return x;
  }
  __device__ __forceinline__ void finish(const float2 *st, int T, int m0, int M, float eps,
                                         float2 *s_ms) {
    const int r = (int)threadIdx.x / TPR, j0 = (int)threadIdx.x % TPR;
    const float2 *row = st + (int64_t)min(m0 + r, M - 1) * T;
    float s[H], m2[H];
#pragma unroll
    for (int h = 0; h < H; ++h) {
      s[h] = p[h][0].x + p[h][1].x;
      for (int t = j0 + TPR * h + 32; t < T; t += 16) s[h] += row[t].x;
    }
    const float mean = total(s) / (float)T;
#pragma unroll
    for (int h = 0; h < H; ++h) {
      const int j = j0 + TPR * h;
      m2[h] = 0.f;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if (j + 16 * i < T) {
          const float d = p[h][i].x - mean;
          m2[h] += p[h][i].y + (float)LIN_STAT_TILE * d * d;
        }
      }
      for (int t = j + 32; t < T; t += 16) {
        const float2 v = row[t];
        const float d = v.x - mean;
        m2[h] += v.y + (float)LIN_STAT_TILE * d * d;
      }
    }
    const float q = total(m2);
    if (j0 == 0) s_ms[r] = make_float2(mean, rsqrtf(q / (float)(LIN_STAT_TILE * T) + eps));
  }
};

template <int DT> __device__ __forceinline__ float round_elem(float v) {
  return Mfma<DT>::widen(Mfma<DT>::narrow(v));
}

// The sum of the waves' partial tiles of quarter q, in the order of a 3-level tree: waves
// w and w + 4 first (SUM4: already added, four sums left), then (s0 + s2) + (s1 + s3).
template <int SUB, bool SUM4>
__device__ __forceinline__ floatx4_t sum_partials(const floatx4_t *s_part, int q, int lane) {
  auto s = [&](int w) {
    const floatx4_t v = s_part[(w * SUB + q) * 64 + lane];
    if constexpr (SUM4) return v;
    else return v + s_part[((w + 4) * SUB + q) * 64 + lane];
  };
  return (s(0) + s(2)) + (s(1) + s(3));
}

// LIN_RESIDUAL's epilogue inputs and epilogue.  Finishing wave w < TT * FT / 2 takes token
// quarter w % TT and a pair of feature quarters (32 features from n0), so each lane holds 8
// of a row's 32 statistics-tile features (4 of each quarter: n0 + 16 f + 4 (lane / 16) ..
// +3) and their statistics need only the 4 lanes of the row (rows_sum4), no LDS exchange.
struct ResidualIn {
  float b[2][4], r[2][4], g[2][4], be[2][4];  // bias, residual (or its pre-norm sum), LN's
  uint2 raw[2];                               // the residual's 8 values as loaded
  // The residual itself, requested with the operands (its 4 registers are the only ones
  // held through the products).
  __device__ __forceinline__ void issue_residual(const LinNorm &nrm, int lane, int m, int n0,
                                                 int M) {
    const int64_t row = min(m, M - 1);
#pragma unroll
    for (int f = 0; f < 2; ++f)  // n + 3 < N: N is a multiple of 32
      raw[f] = *reinterpret_cast<const uint2 *>(nrm.res + row * nrm.res_stride + n0 + 16 * f +
                                                4 * (lane >> 4));
  }
  template <int DT>
  __device__ __forceinline__ void issue(const uint16_t *bias, const LinNorm &nrm, int lane,
                                        int n0) {
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      const int n = n0 + 16 * f + 4 * (lane >> 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) b[f][j] = bias ? Mfma<DT>::widen(bias[n + j]) : 0.f;
      unpack4<DT>(raw[f], r[f]);
      if (nrm.res_stats) {
        unpack4<DT>(*reinterpret_cast<const uint2 *>(nrm.res_gamma + n), g[f]);
        unpack4<DT>(*reinterpret_cast<const uint2 *>(nrm.res_beta + n), be[f]);
      }
    }
  }
  template <int DT> __device__ __forceinline__ static void unpack4(uint2 w, float (&o)[4]) {
    o[0] = Mfma<DT>::widen_lo(w.x);
    o[1] = Mfma<DT>::widen_hi(w.x);
    o[2] = Mfma<DT>::widen_lo(w.y);
    o[3] = Mfma<DT>::widen_hi(w.y);
  }
};

// The values are rounded where the separate projection store and LayerNorm kernel round
// them: y, the normalized residual, v.
template <int DT, int FT, int TT, bool SUM4>
__device__ __forceinline__ void residual_epilogue(const floatx4_t *s_part, int wv, int lane,
                                                  int m0, int n0, int M, int N,
                                                  const ResidualIn &in, const float2 *s_ms,
                                                  uint16_t *y, int64_t ldy, const LinNorm &nrm) {
  const int t = wv % TT, pair = wv / TT;
  const int r = 16 * t + (lane & 15);  // the workgroup's row
  const int m = m0 + r;
  float mean = 0.f, rstd = 1.f;
  if (nrm.res_stats) {
    mean = s_ms[r].x;
    rstd = s_ms[r].y;
  }
  float o[2][4];
#pragma unroll
  for (int f = 0; f < 2; ++f) {
    const floatx4_t v =
        sum_partials<FT * TT, SUM4>(s_part, (2 * pair + f) * TT + t, lane);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float yj = round_elem<DT>(v[j] + in.b[f][j]);
      const float hj = nrm.res_stats
                           ? round_elem<DT>((in.r[f][j] - mean) * rstd * in.g[f][j] + in.be[f][j])
                           : in.r[f][j];
      o[f][j] = round_elem<DT>(yj + hj);
    }
  }
  // The tile row's mean over the lane's 8 values and the row's 4 lanes, then the sum of
  // squared deviations from it, in a fixed order.
  const float tmean =
      rows_sum4(((o[0][0] + o[0][1]) + (o[0][2] + o[0][3])) +
                ((o[1][0] + o[1][1]) + (o[1][2] + o[1][3]))) / (float)LIN_STAT_TILE;
  float dd = 0.f;
#pragma unroll
  for (int f = 0; f < 2; ++f)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float d = o[f][j] - tmean;
      dd = fmaf(d, d, dd);
    }
  const float m2 = rows_sum4(dd);
  if (m >= M) return;
#pragma unroll
  for (int f = 0; f < 2; ++f)
    *reinterpret_cast<uint2 *>(y + (int64_t)m * ldy + n0 + 16 * f + 4 * (lane >> 4)) =
        make_uint2(Mfma<DT>::narrow2(o[f][0], o[f][1]), Mfma<DT>::narrow2(o[f][2], o[f][3]));
  if (lane < 16)
    nrm.y_stats[(int64_t)m * (N / LIN_STAT_TILE) + n0 / LIN_STAT_TILE] = make_float2(tmean, m2);
}

// XP: x is packed (no ds_bpermute); GELU: exact GELU after the bias; YP: y is written
// packed (rows padded to 32; padding rows are left unwritten); B: K steps whose operands
// are loaded together; PIPE: two such batches, double-buffered; WR: the weight is in its own
// row-major layout, read as the activation rows are;
// MODE: LIN_PLAIN, LIN_NORM_IN (x is a pre-norm sum, nrm.x_stats its statistics) or
// LIN_RESIDUAL (y = v and nrm.y_stats, as described above).  FT x TT: 16-feature x 16-token
// quarters of the output tile (the rule is at pick_tile).
template <int DT, bool XP, bool GELU, bool YP, bool PIPE, int MODE, int FT, int TT, int B,
          bool WR>
__global__ __launch_bounds__(64 * LIN_WAVES) void decode_linear_kernel(
    const uint16_t *__restrict__ x, int64_t ldx, const uint16_t *__restrict__ wp,
    const uint16_t *__restrict__ bias, uint16_t *__restrict__ y, int64_t ldy, int M, int N,
    int K, bool vec_store, LinNorm nrm) {
  static_assert(MODE != LIN_RESIDUAL || (!GELU && !YP), "the residual epilogue stores v");
  static_assert(MODE != LIN_NORM_IN || !XP, "a pre-norm x is stored row by row");
  static_assert(!XP || TT <= 2, "packed activations are padded to 32 rows");
  constexpr int SUB = FT * TT;  // 16 x 16 quarters of the tile
  // The tiles up to 32 x 32 hand the partial tiles over in two halves (8 or 16 KB); the larger
  // ones, one on a CU by their registers (157 to 256; 32 x 32: up to 124, two on a CU), all at
  // once (64 or 128 KB, one barrier), and every wave finishes QPW quarters.
  constexpr bool HALVES = SUB < LIN_WAVES;
  constexpr int QPW = HALVES ? 1 : SUB / LIN_WAVES;
  static_assert(TT % QPW == 0, "a wave's quarters share their features");
  // Partial tiles of four (eight) waves, each in the MFMA result order (16 bytes per lane).
  __shared__ floatx4_t s_part[(HALVES ? LIN_WAVES / 2 : LIN_WAVES) * SUB * 64];

  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int n0 = blockIdx.x * (16 * FT), m0 = blockIdx.y * (16 * TT);
  const int ks = K / 32;
  // This wave's K steps: wv, wv + 8, ... where it loads them all at once (the waves then
  // read neighbouring KBs and the two halves of a row's 128-byte lines together: 512 rows,
  // 1024 to 1024, 6.0 against 7.1 us; 256 rows, 1024 to 4096, 10.0 against 10.5), a
  // contiguous range of a longer K, walked in batches (4096 to 1024: 10.3 against 10.6).
  constexpr bool SPREAD = !PIPE && B == LIN_BATCH;
  constexpr int KSTEP = SPREAD ? LIN_WAVES : 1;
  const int steps = ks / LIN_WAVES;
  const int k0 = SPREAD ? wv : wv * steps;
  // byte address of the lane whose 64-byte run holds this lane's operand chunk
  const int src = 4 * (4 * (lane & 15) + (lane >> 4));

  // Packed weight blocks of this wave's first K step; activation runs (rows past M read
  // the last row; their results are dropped).
  const uint16_t *wblk[FT];
  const uint16_t *xrow[TT];
#pragma unroll
  for (int f = 0; f < FT; ++f)
    wblk[f] = WR ? wp + (int64_t)(n0 + 16 * f + (lane >> 2)) * K + 32 * k0 + 8 * (lane & 3)
                 : wp + ((int64_t)(n0 / 16 + f) * ks + k0) * LIN_BLOCK + lane * 8;
#pragma unroll
  for (int t = 0; t < TT; ++t)
    xrow[t] = XP ? x + ((int64_t)(m0 / 16 + t) * ks + k0) * LIN_BLOCK + lane * 8
                 : x + (int64_t)min(m0 + 16 * t + (lane >> 2), M - 1) * ldx + 32 * k0 +
                       8 * (lane & 3);
  constexpr int WSTEP = KSTEP * (WR ? 32 : LIN_BLOCK), XSTEP = KSTEP * (XP ? LIN_BLOCK : 32);

  // Quarter q of the tile is features 16 (q / TT) + 4 (lane / 16) .. +3 of token
  // 16 (q % TT) + lane % 16; wave w finishes quarters QPW w .. +QPW - 1.  Their bias is
  // requested now, with the operands, so that no load is left for after the reduction.
  const bool finisher = QPW * wv < SUB;
  const int qf = QPW * wv / TT, qt = QPW * wv % TT;
  const int qn = n0 + 16 * qf + 4 * (lane >> 4);
  float bv[4] = {0.f, 0.f, 0.f, 0.f};
  if (bias && finisher && MODE == LIN_PLAIN) {
#pragma unroll
    for (int j = 0; j < 4; ++j) bv[j] = qn + j < N ? Mfma<DT>::widen(bias[qn + j]) : 0.f;
  }
  // The epilogue inputs requested before the operands so that they have landed when
  // the products have (loads complete in order): the rows' tile statistics (two per
  // thread) and, for LIN_NORM_IN's finishing lanes (features qn .. qn + 3), u and b'.
  constexpr int TPR = TT > 2 ? 8 : 16;  // threads per row of statistics
  __shared__ float2 s_ms[MODE == LIN_PLAIN ? 1 : 64 * LIN_WAVES / TPR];
  RowStatLoads<TPR> rsl;
  const float2 *row_st = nullptr;
  int row_t = 0;
  float fa[4] = {0.f, 0.f, 0.f, 0.f}, fb[4] = {0.f, 0.f, 0.f, 0.f};  // LIN_NORM_IN: u, b'
  if constexpr (MODE == LIN_NORM_IN) {
    row_st = nrm.x_stats;
    row_t = K / LIN_STAT_TILE;
    if (finisher) {
      if (qn + 3 < N && nrm.vec4) {  // one 16-byte load each
        const float4 a = *reinterpret_cast<const float4 *>(nrm.u + qn);
        const float4 b = *reinterpret_cast<const float4 *>(nrm.fbias + qn);
        fa[0] = a.x, fa[1] = a.y, fa[2] = a.z, fa[3] = a.w;
        fb[0] = b.x, fb[1] = b.y, fb[2] = b.z, fb[3] = b.w;
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          fa[j] = qn + j < N ? nrm.u[qn + j] : 0.f;
          fb[j] = qn + j < N ? nrm.fbias[qn + j] : 0.f;
        }
      }
    }
  }
  if constexpr (MODE == LIN_RESIDUAL) {
    row_st = nrm.res_stats;  // null: a plain residual
    row_t = N / LIN_STAT_TILE;
  }
  if (MODE != LIN_PLAIN && row_st) rsl.issue(row_st, row_t, m0, M);
  // The residual too, for one batch of K steps (a 1024-deep output projection: 6.2
  // against 6.3 us); a longer, double-buffered K loop ran 0.1 us slower with it here.
  ResidualIn rin;
  const bool res_finisher = wv < TT * FT / 2;
  const int res_m = m0 + 16 * (wv % TT) + (lane & 15), res_n = n0 + 32 * (wv / TT);
  if constexpr (MODE == LIN_RESIDUAL && !PIPE) {
    if (res_finisher) rin.issue_residual(nrm, lane, res_m, res_n, M);
  }

  floatx4_t acc[FT][TT];
#pragma unroll
  for (int f = 0; f < FT; ++f)
#pragma unroll
    for (int t = 0; t < TT; ++t) acc[f][t] = floatx4_t{0.f, 0.f, 0.f, 0.f};

  auto load = [&](uint4 (&a)[B][FT], uint4 (&b)[B][TT], int s0) {
#pragma unroll
    for (int g = 0; g < B; ++g) {
      if (s0 + g < steps) {
#pragma unroll
        for (int f = 0; f < FT; ++f)
          a[g][f] = *reinterpret_cast<const uint4 *>(wblk[f] + WSTEP * (s0 + g));
#pragma unroll
        for (int t = 0; t < TT; ++t)
          b[g][t] = *reinterpret_cast<const uint4 *>(xrow[t] + XSTEP * (s0 + g));
      }
    }
  };
  auto to_operand = [&](uint4 &v) {  // a 64-byte row run in operand order
    v.x = __builtin_amdgcn_ds_bpermute(src, (int)v.x);
    v.y = __builtin_amdgcn_ds_bpermute(src, (int)v.y);
    v.z = __builtin_amdgcn_ds_bpermute(src, (int)v.z);
    v.w = __builtin_amdgcn_ds_bpermute(src, (int)v.w);
  };
  auto multiply = [&](uint4 (&a)[B][FT], uint4 (&b)[B][TT], int s0) {
#pragma unroll
    for (int g = 0; g < B; ++g) {
      if (s0 + g < steps) {
#pragma unroll
        for (int t = 0; t < TT && !XP; ++t) to_operand(b[g][t]);
#pragma unroll
        for (int f = 0; f < FT && WR; ++f) to_operand(a[g][f]);
#pragma unroll
        for (int f = 0; f < FT; ++f)
#pragma unroll
          for (int t = 0; t < TT; ++t) acc[f][t] = Mfma<DT>::qk(a[g][f], b[g][t], acc[f][t]);
      }
    }
  };
  if constexpr (PIPE) {
    uint4 a0[B][FT], b0[B][TT], a1[B][FT], b1[B][TT];
    load(a0, b0, 0);
    for (int s0 = 0; s0 < steps; s0 += 2 * B) {
      if (s0 + B < steps) load(a1, b1, s0 + B);
      multiply(a0, b0, s0);
      if (s0 + 2 * B < steps) load(a0, b0, s0 + 2 * B);
      if (s0 + B < steps) multiply(a1, b1, s0 + B);
    }
  } else {
    for (int s0 = 0; s0 < steps; s0 += B) {
      uint4 a[B][FT], b[B][TT];
      load(a, b, s0);
      multiply(a, b, s0);
    }
  }

  // LIN_RESIDUAL's per-feature inputs, requested now so that they overlap the reduction
  // below (with them before the operands, a 1024-wide output projection ran 0.3 us
  // slower).
  if constexpr (MODE == LIN_RESIDUAL) {
    if (res_finisher) {
      if constexpr (PIPE) rin.issue_residual(nrm, lane, res_m, res_n, M);
      rin.issue<DT>(bias, nrm, lane, res_n);
    }
  }

  // Sum the waves' partial tiles.  Halves: waves 4..7 hand theirs to waves 0..3, which add
  // and publish the four sums.
  if constexpr (!HALVES) {
#pragma unroll
    for (int f = 0; f < FT; ++f)
#pragma unroll
      for (int t = 0; t < TT; ++t) s_part[(wv * SUB + f * TT + t) * 64 + lane] = acc[f][t];
  } else if (wv >= LIN_WAVES / 2) {
#pragma unroll
    for (int f = 0; f < FT; ++f)
#pragma unroll
      for (int t = 0; t < TT; ++t)
        s_part[((wv - LIN_WAVES / 2) * SUB + f * TT + t) * 64 + lane] = acc[f][t];
  }
  if constexpr (HALVES) {
    __syncthreads();
    if (wv < LIN_WAVES / 2) {
#pragma unroll
      for (int f = 0; f < FT; ++f)
#pragma unroll
        for (int t = 0; t < TT; ++t) acc[f][t] += s_part[(wv * SUB + f * TT + t) * 64 + lane];
    }
    __syncthreads();
    if (wv < LIN_WAVES / 2) {
#pragma unroll
      for (int f = 0; f < FT; ++f)
#pragma unroll
        for (int t = 0; t < TT; ++t) s_part[(wv * SUB + f * TT + t) * 64 + lane] = acc[f][t];
    }
  }
  if (MODE != LIN_PLAIN && row_st)
    rsl.finish(row_st, row_t, m0, M, MODE == LIN_NORM_IN ? nrm.eps : nrm.res_eps, s_ms);
  __syncthreads();

  if constexpr (MODE == LIN_RESIDUAL) {
    if (res_finisher)
      residual_epilogue<DT, FT, TT, HALVES>(s_part, wv, lane, m0, res_n, M, N, rin, s_ms, y, ldy,
                                            nrm);
    return;
  }
  if (!finisher || qn >= N) return;
#pragma unroll
  for (int i = 0; i < QPW; ++i) {
    const int m = m0 + 16 * (qt + i) + (lane & 15);
    if (m >= M) return;
    const floatx4_t v = sum_partials<SUB, HALVES>(s_part, QPW * wv + i, lane);
    float mean = 0.f, rstd = 1.f;
    if constexpr (MODE == LIN_NORM_IN) {
      const float2 ms = s_ms[16 * (qt + i) + (lane & 15)];
      mean = ms.x;
      rstd = ms.y;
    }
    uint32_t h[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float o = MODE == LIN_NORM_IN ? fmaf(fmaf(-mean, fa[j], v[j]), rstd, fb[j])
                                          : v[j] + bv[j];
      h[j] = Mfma<DT>::narrow(GELU ? gelu_of_stored<DT>(o) : o);
    }
    if constexpr (YP) {  // 4 consecutive columns of one row: 8 bytes of one lane's chunk
      *reinterpret_cast<uint2 *>(y + packed_offset(m, qn, N)) =
          make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
      continue;
    }
    uint16_t *dst = y + (int64_t)m * ldy + qn;
    if (vec_store && qn + 3 < N) {
      *reinterpret_cast<uint2 *>(dst) = make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (qn + j < N) dst[j] = (uint16_t)h[j];
    }
  }
}

static int check_features(int out_features, int in_features, int dtype, const char *who) {
  if (dtype != VFL_BFLOAT16 && dtype != VFL_FLOAT16) {
    set_error("%s: dtype %d has no kernel (bf16 and fp16 only)", who, dtype);
    return VFL_E_UNSUPPORTED;
  }
  if (out_features <= 0 || in_features <= 0) {
    set_error("%s: bad sizes (out %d in %d)", who, out_features, in_features);
    return VFL_E_INVALID;
  }
  if (in_features % LIN_K_MULTIPLE != 0) {
    set_error("%s: in_features must be a multiple of %d (got %d)", who, LIN_K_MULTIPLE,
              in_features);
    return VFL_E_UNSUPPORTED;
  }
  return VFL_OK;
}

}  // namespace vfl

using namespace vfl;

extern "C" int64_t vfl_linear_packed_elems(int rows, int cols) {
  if (rows <= 0 || cols <= 0) return 0;
  return packed_rows(rows) * cols;
}

extern "C" int vfl_pack_linear_weight(const void *weight, int64_t weight_stride,
                                      int out_features, int in_features, void *packed,
                                      int dtype, void *stream) {
  clear_error();
  int st = check_features(out_features, in_features, dtype, "pack_linear_weight");
  if (st != VFL_OK) return st;
  if (weight_stride < in_features) {
    set_error("pack_linear_weight: weight_stride %lld < in_features %d",
              (long long)weight_stride, in_features);
    return VFL_E_INVALID;
  }
  if (!weight || !packed) {
    set_error("pack_linear_weight: null pointer argument");
    return VFL_E_INVALID;
  }
  if (((uintptr_t)weight | (uintptr_t)packed) % 16 != 0 || weight_stride % 8 != 0) {
    set_error("pack_linear_weight: weight and packed must be 16-byte aligned, the weight "
              "row stride a multiple of 8 elements");
    return VFL_E_INVALID;
  }
  const int64_t chunks = packed_rows(out_features) * in_features / 8;
  pack_linear_weight_kernel<<<dim3((unsigned)((chunks + 255) / 256)), dim3(256), 0,
                              (hipStream_t)stream>>>(
      (const uint16_t *)weight, weight_stride, out_features, in_features, (uint16_t *)packed,
      chunks);
  return launch_status("pack_linear_weight");
}

template <bool XP, bool GELU, bool YP, bool PIPE, int MODE, int FT, int TT, int B,
          bool WR = false>
static void launch_linear_dt(hipStream_t s, int dtype, const void *x, int64_t x_stride,
                             const void *wp, const void *bias, void *y, int64_t y_stride,
                             int64_t rows, int out_features, int in_features, bool vec_store,
                             const LinNorm &nrm) {
  const dim3 grid((unsigned)(packed_rows(out_features) / (16 * FT)),
                  (unsigned)((rows + 16 * TT - 1) / (16 * TT)));
  if (dtype == VFL_BFLOAT16)
    decode_linear_kernel<VFL_BFLOAT16, XP, GELU, YP, PIPE, MODE, FT, TT, B, WR>
        <<<grid, dim3(64 * LIN_WAVES), 0, s>>>(
        (const uint16_t *)x, x_stride, (const uint16_t *)wp, (const uint16_t *)bias,
        (uint16_t *)y, y_stride, (int)rows, out_features, in_features, vec_store, nrm);
  else
    decode_linear_kernel<VFL_FLOAT16, XP, GELU, YP, PIPE, MODE, FT, TT, B, WR>
        <<<grid, dim3(64 * LIN_WAVES), 0, s>>>(
        (const uint16_t *)x, x_stride, (const uint16_t *)wp, (const uint16_t *)bias,
        (uint16_t *)y, y_stride, (int)rows, out_features, in_features, vec_store, nrm);
}

enum LinTile { TILE_32x16, TILE_32x32, TILE_64x32, TILE_64x64 };

// The output tile (features x tokens).  A CU takes two workgroups of 32 x 32 tiles or one of
// the larger ones, and moves operands at about 30 bytes a cycle whatever their source (the
// same with the weight in its L2), so what counts is how often the operands are read again
// -- half as often at 64 x 64 -- and whether the last round of workgroups is full.  Sums
// run in the same order for every tile: the results are the same bits.
// - 32 x 16 up to 16 rows: half the activation loads.  4 rows against 32 x 32, us: 1024 to
//   1024 3.7 / 4.2, to 4096 5.7 / 6.0, 4096 to 1024 9.7 / 11.5.
// - 64 x 64 where 32 x 32 tiles need a second round and it does not, or its second round is
//   nearly full.  Fused q|k|v and feed-forward of 256 rows, 32 x 32 / 64 x 64, us: 1024 to
//   3072 8.7 / 7.5, to 4096 12.2 / 10.0, 768 to 3072 8.7 / 7.8; 512 rows to 4096 19.0 / 17.2.
//   Elsewhere it is the slower one (1024 to 4096: 128 rows 8.1 / 10.4, 384 15.3 / 16.3).
// - 64 x 32 where 32 x 32 tiles put a second workgroup on some CUs: 512 rows, 4096 to 1024
//   15.8 / 13.4, 1024 to 1024 7.4 / 6.1; 128 rows, 768 to 3072 6.1 / 5.5, 1024 to 4096
//   8.1 / 7.2.  With one on each it loses (256 rows, 1024 to 1024: 5.4 / 5.9), and without
//   row statistics (LIN_PLAIN) so it does up to 768 inputs, three K steps a wave: 512 rows, 768
//   to 768 4.7 / 4.9 (352 rows 4.5 / 4.9); 128 rows, 768 to 2304 4.8 / 5.2; 320 rows, 512 to 1536
//   4.2 / 4.4; yet 512 rows, 1024 to 1024 5.8 / 5.4.
static LinTile pick_tile(int64_t rows, int out_features, int in_features, bool packed_x,
                         int mode) {
  if (rows <= 16) return TILE_32x16;
  if (out_features % 64 != 0) return TILE_32x32;
  const int64_t t32 = out_features / 32 * ((rows + 31) / 32);
  const int64_t t64 = out_features / 64 * ((rows + 63) / 64);
  if (!packed_x && mode != LIN_RESIDUAL &&
      ((t32 > 512 && t64 <= 256) || (t64 > 448 && t64 <= 512)))
    return TILE_64x64;
  if (mode == LIN_PLAIN && in_features < LIN_BATCH * LIN_K_MULTIPLE) return TILE_32x32;
  return t32 > 256 && t32 <= 512 ? TILE_64x32 : TILE_32x32;
}

// K steps per batch of loads: all of a wave's steps where the registers hold them (4 steps
// of the larger tiles, 16 of 32 x 16), double-buffered batches beyond.
template <bool XP, bool GELU, bool YP, int MODE = LIN_PLAIN>
static void launch_linear(hipStream_t s, int dtype, const void *x, int64_t x_stride,
                          const void *wp, const void *bias, void *y, int64_t y_stride,
                          int64_t rows, int out_features, int in_features, bool vec_store,
                          const LinNorm &nrm = LinNorm{}) {
  const LinTile tile = pick_tile(rows, out_features, in_features, XP, MODE);
  const int steps = in_features / LIN_K_MULTIPLE;
#define VFL_TILE(P, FT, TT, B)                                                               \
  launch_linear_dt<XP, GELU, YP, P, MODE, FT, TT, B>(s, dtype, x, x_stride, wp, bias, y,     \
                                                     y_stride, rows, out_features,           \
                                                     in_features, vec_store, nrm)
  if (tile == TILE_32x16) {
    if (steps <= LIN_BATCH) VFL_TILE(false, 2, 1, LIN_BATCH);
    else if (steps <= 16) VFL_TILE(false, 2, 1, 16);
    else VFL_TILE(true, 2, 1, LIN_BATCH);
    return;
  }
  if constexpr (!XP && MODE != LIN_RESIDUAL) {
    if (tile == TILE_64x64) {
      if (steps > LIN_BATCH) VFL_TILE(true, 4, 4, LIN_PIPE_BATCH);
      else VFL_TILE(false, 4, 4, LIN_BATCH);
      return;
    }
  }
  if (tile == TILE_64x32) {
    if (steps > LIN_BATCH) VFL_TILE(true, 4, 2, LIN_PIPE_BATCH);
    else VFL_TILE(false, 4, 2, LIN_BATCH);
  } else if (steps <= LIN_BATCH) {
    VFL_TILE(false, 2, 2, LIN_BATCH);
  } else {
    VFL_TILE(true, 2, 2, LIN_PIPE_BATCH);
  }
#undef VFL_TILE
}

extern "C" int vfl_linear(const void *x, int64_t x_stride, const void *packed_weight,
                          const void *bias, void *y, int64_t y_stride, int64_t rows,
                          int out_features, int in_features, int flags, int dtype,
                          void *stream) {
  clear_error();
  int st = check_features(out_features, in_features, dtype, "linear");
  if (st != VFL_OK) return st;
  if (rows < 0 || rows > 65535LL * LIN_TILE) {
    set_error("linear: rows must be in [0, %lld] (got %lld)", 65535LL * LIN_TILE,
              (long long)rows);
    return rows < 0 ? VFL_E_INVALID : VFL_E_UNSUPPORTED;
  }
  if (flags & ~(VFL_LINEAR_GELU | VFL_LINEAR_X_PACKED | VFL_LINEAR_Y_PACKED)) {
    set_error("linear: unknown flags 0x%x", flags);
    return VFL_E_INVALID;
  }
  const bool xp = flags & VFL_LINEAR_X_PACKED, yp = flags & VFL_LINEAR_Y_PACKED;
  if ((!xp && x_stride < in_features) || (!yp && y_stride < out_features)) {
    set_error("linear: row strides must cover the rows (x %lld y %lld)", (long long)x_stride,
              (long long)y_stride);
    return VFL_E_INVALID;
  }
  if (yp && out_features % LIN_TILE != 0) {
    set_error("linear: a packed output needs out_features a multiple of %d (got %d)", LIN_TILE,
              out_features);
    return VFL_E_UNSUPPORTED;
  }
  if (rows == 0) return VFL_OK;
  if (!x || !packed_weight || !y) {
    set_error("linear: null pointer argument");
    return VFL_E_INVALID;
  }
  if (((uintptr_t)x | (uintptr_t)packed_weight) % 16 != 0 || (!xp && x_stride % 8 != 0) ||
      (uintptr_t)y % (yp ? 8 : 2) != 0 || (uintptr_t)bias % 2 != 0) {
    set_error("linear: x and the packed weight must be 16-byte aligned, the x row stride a "
              "multiple of 8 elements");
    return VFL_E_INVALID;
  }
  const bool vec_store = (uintptr_t)y % 8 == 0 && y_stride % 4 == 0;
  hipStream_t s = (hipStream_t)stream;
  const bool gelu = flags & VFL_LINEAR_GELU;
#define VFL_LIN(XP, G, YP)                                                                   \
  launch_linear<XP, G, YP>(s, dtype, x, x_stride, packed_weight, bias, y, y_stride, rows, \
                           out_features, in_features, vec_store)
  if (!xp && !gelu && !yp)
    VFL_LIN(false, false, false);
  else if (!xp && gelu && yp)
    VFL_LIN(false, true, true);
  else if (xp && !gelu && !yp)
    VFL_LIN(true, false, false);
  else if (!xp && gelu && !yp)
    VFL_LIN(false, true, false);
  else if (!xp && !gelu && yp)
    VFL_LIN(false, false, true);
  else if (xp && gelu && !yp)
    VFL_LIN(true, true, false);
  else if (xp && !gelu && yp)
    VFL_LIN(true, false, true);
  else
    VFL_LIN(true, true, true);
#undef VFL_LIN
  return launch_status("linear");
}

extern "C" int vfl_linear_rows(const void *x, int64_t x_stride, const void *weight,
                               const void *bias, void *y, int64_t y_stride, int64_t rows,
                               int out_features, int in_features, int dtype, void *stream) {
  clear_error();
  int st = check_features(out_features, in_features, dtype, "linear_rows");
  if (st != VFL_OK) return st;
  if (rows < 0 || x_stride < in_features || y_stride < out_features) {
    set_error("linear_rows: bad sizes (rows %lld, row strides x %lld y %lld)", (long long)rows,
              (long long)x_stride, (long long)y_stride);
    return VFL_E_INVALID;
  }
  if (out_features % LIN_TILE != 0 || in_features > LIN_BATCH * LIN_K_MULTIPLE ||
      rows > 65535LL * 16) {
    set_error("linear_rows: out_features must be a multiple of %d, in_features and rows at most "
              "%d and %lld (got %d, %d, %lld)", LIN_TILE, LIN_BATCH * LIN_K_MULTIPLE,
              65535LL * 16, out_features, in_features, (long long)rows);
    return VFL_E_UNSUPPORTED;
  }
  if (rows == 0) return VFL_OK;
  if (!x || !weight || !y) {
    set_error("linear_rows: null pointer argument");
    return VFL_E_INVALID;
  }
  if (((uintptr_t)x | (uintptr_t)weight) % 16 != 0 || x_stride % 8 != 0 ||
      ((uintptr_t)y | (uintptr_t)bias) % 2 != 0) {
    set_error("linear_rows: x and the weight must be 16-byte aligned, the x row stride a "
              "multiple of 8 elements");
    return VFL_E_INVALID;
  }
  const bool vec_store = (uintptr_t)y % 8 == 0 && y_stride % 4 == 0;
#define VFL_TILE(FT, TT)                                                                     \
  launch_linear_dt<false, false, false, false, LIN_PLAIN, FT, TT, LIN_BATCH, true>(          \
      (hipStream_t)stream, dtype, x, x_stride, weight, bias, y, y_stride, rows, out_features, \
      in_features, vec_store, LinNorm{})
  switch (pick_tile(rows, out_features, in_features, false, LIN_PLAIN)) {
    case TILE_32x16: VFL_TILE(2, 1); break;
    case TILE_32x32: VFL_TILE(2, 2); break;
    case TILE_64x32: VFL_TILE(4, 2); break;
    case TILE_64x64: VFL_TILE(4, 4); break;
  }
#undef VFL_TILE
  return launch_status("linear_rows");
}

namespace vfl {

// h = LN(v) from v's tile statistics (the last sublayer's output before the LM head):
// one wave per row, the row's tiles combined in a fixed order, then the LayerNorm
// kernel's expression per element.
template <int DT>
__global__ __launch_bounds__(128) void layer_norm_apply_kernel(
    const uint16_t *__restrict__ v, int64_t v_stride, const float2 *__restrict__ st,
    const uint16_t *__restrict__ gamma, const uint16_t *__restrict__ beta, float eps,
    uint16_t *__restrict__ out, int64_t out_stride, int64_t rows, int dim) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 2 + (threadIdx.x >> 6);
  if (row >= rows) return;  // wave-uniform
  const int T = dim / LIN_STAT_TILE;
  const float2 *rs = st + row * T;
  float s = 0.f;
  for (int t = lane; t < T; t += 64) s += rs[t].x;
  const float mean = group_sum<64>(s) / (float)T;
  float m2 = 0.f;
  for (int t = lane; t < T; t += 64) {
    const float2 p = rs[t];
    const float d = p.x - mean;
    m2 += p.y + (float)LIN_STAT_TILE * d * d;
  }
  const float rstd = rsqrtf(group_sum<64>(m2) / (float)dim + eps);
  for (int i = 4 * lane; i < dim; i += 256) {
    const uint2 a = *reinterpret_cast<const uint2 *>(v + row * v_stride + i);
    const uint2 g = *reinterpret_cast<const uint2 *>(gamma + i);
    const uint2 b = *reinterpret_cast<const uint2 *>(beta + i);
    const uint32_t aw[2] = {a.x, a.y}, gw[2] = {g.x, g.y}, bw[2] = {b.x, b.y};
    uint32_t o[2];
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      const float lo = (Mfma<DT>::widen_lo(aw[w]) - mean) * rstd * Mfma<DT>::widen_lo(gw[w]) +
                       Mfma<DT>::widen_lo(bw[w]);
      const float hi = (Mfma<DT>::widen_hi(aw[w]) - mean) * rstd * Mfma<DT>::widen_hi(gw[w]) +
                       Mfma<DT>::widen_hi(bw[w]);
      o[w] = Mfma<DT>::narrow2(lo, hi);
    }
    *reinterpret_cast<uint2 *>(out + row * out_stride + i) = make_uint2(o[0], o[1]);
  }
}

}  // namespace vfl

static int check_norm_rows(int64_t rows, const char *who) {
  if (rows < 0 || rows > 65535LL * LIN_TILE) {
    set_error("%s: rows must be in [0, %lld] (got %lld)", who, 65535LL * LIN_TILE,
              (long long)rows);
    return rows < 0 ? VFL_E_INVALID : VFL_E_UNSUPPORTED;
  }
  return VFL_OK;
}

extern "C" int vfl_linear_norm(const void *x, int64_t x_stride, const float *x_stats, float eps,
                               const void *packed_weight, const float *u,
                               const float *folded_bias, void *y, int64_t y_stride,
                               int64_t rows, int out_features, int in_features, int flags,
                               int dtype, void *stream) {
  clear_error();
  int st = check_features(out_features, in_features, dtype, "linear_norm");
  if (st == VFL_OK) st = check_norm_rows(rows, "linear_norm");
  if (st != VFL_OK) return st;
  if (flags & ~(VFL_LINEAR_GELU | VFL_LINEAR_Y_PACKED)) {
    set_error("linear_norm: flags 0x%x (GELU and Y_PACKED only: x is a pre-norm sum)", flags);
    return VFL_E_INVALID;
  }
  const bool yp = flags & VFL_LINEAR_Y_PACKED, gelu = flags & VFL_LINEAR_GELU;
  if (x_stride < in_features || (!yp && y_stride < out_features) || !(eps >= 0.f)) {
    set_error("linear_norm: row strides must cover the rows (x %lld y %lld), eps >= 0",
              (long long)x_stride, (long long)y_stride);
    return VFL_E_INVALID;
  }
  if (yp && out_features % LIN_TILE != 0) {
    set_error("linear_norm: a packed output needs out_features a multiple of %d (got %d)",
              LIN_TILE, out_features);
    return VFL_E_UNSUPPORTED;
  }
  if (rows == 0) return VFL_OK;
  if (!x || !x_stats || !packed_weight || !u || !folded_bias || !y) {
    set_error("linear_norm: null pointer argument");
    return VFL_E_INVALID;
  }
  if (((uintptr_t)x | (uintptr_t)packed_weight) % 16 != 0 || x_stride % 8 != 0 ||
      (uintptr_t)x_stats % 8 != 0 || ((uintptr_t)u | (uintptr_t)folded_bias) % 4 != 0 ||
      (uintptr_t)y % (yp ? 8 : 2) != 0) {
    set_error("linear_norm: x and the packed weight must be 16-byte aligned, the x row stride "
              "a multiple of 8 elements, x_stats 8-byte and u / folded_bias 4-byte aligned");
    return VFL_E_INVALID;
  }
  LinNorm nrm{};
  nrm.x_stats = reinterpret_cast<const float2 *>(x_stats);
  nrm.u = u;
  nrm.fbias = folded_bias;
  nrm.eps = eps;
  nrm.vec4 = ((uintptr_t)u | (uintptr_t)folded_bias) % 16 == 0;
  const bool vec_store = (uintptr_t)y % 8 == 0 && y_stride % 4 == 0;
  hipStream_t s = (hipStream_t)stream;
#define VFL_LINN(G, YP)                                                                   \
  launch_linear<false, G, YP, LIN_NORM_IN>(s, dtype, x, x_stride, packed_weight, nullptr, \
                                           y, y_stride, rows, out_features, in_features,     \
                                           vec_store, nrm)
  if (!gelu && !yp)
    VFL_LINN(false, false);
  else if (gelu && yp)
    VFL_LINN(true, true);
  else if (gelu)
    VFL_LINN(true, false);
  else
    VFL_LINN(false, true);
#undef VFL_LINN
  return launch_status("linear_norm");
}

extern "C" int vfl_linear_residual(const void *x, int64_t x_stride, const void *packed_weight,
                                   const void *bias, const void *residual, int64_t r_stride,
                                   const float *r_stats, const void *r_gamma,
                                   const void *r_beta, float r_eps, void *y, int64_t y_stride,
                                   float *y_stats, int64_t rows, int out_features,
                                   int in_features, int flags, int dtype, void *stream) {
  clear_error();
  int st = check_features(out_features, in_features, dtype, "linear_residual");
  if (st == VFL_OK) st = check_norm_rows(rows, "linear_residual");
  if (st != VFL_OK) return st;
  if (flags & ~VFL_LINEAR_X_PACKED) {
    set_error("linear_residual: flags 0x%x (X_PACKED only: y is the pre-norm sum)", flags);
    return VFL_E_INVALID;
  }
  const bool xp = flags & VFL_LINEAR_X_PACKED;
  if (out_features % LIN_STAT_TILE != 0) {
    set_error("linear_residual: out_features must be a multiple of %d (got %d)", LIN_STAT_TILE,
              out_features);
    return VFL_E_UNSUPPORTED;
  }
  if ((!xp && x_stride < in_features) || y_stride < out_features || r_stride < out_features ||
      (r_stats && !(r_eps >= 0.f))) {
    set_error("linear_residual: row strides must cover the rows (x %lld y %lld residual %lld)",
              (long long)x_stride, (long long)y_stride, (long long)r_stride);
    return VFL_E_INVALID;
  }
  if (rows == 0) return VFL_OK;
  if (!x || !packed_weight || !residual || !y || !y_stats ||
      (r_stats && (!r_gamma || !r_beta))) {
    set_error("linear_residual: null pointer argument");
    return VFL_E_INVALID;
  }
  if ((const void *)y_stats == (const void *)r_stats) {
    set_error("linear_residual: y_stats must not alias r_stats (every workgroup of a row "
              "reads the residual's statistics)");
    return VFL_E_INVALID;
  }
  if (((uintptr_t)x | (uintptr_t)packed_weight) % 16 != 0 || (!xp && x_stride % 8 != 0) ||
      (uintptr_t)y % 8 != 0 || y_stride % 4 != 0 || (uintptr_t)bias % 2 != 0 ||
      (uintptr_t)residual % 8 != 0 || r_stride % 4 != 0 ||
      ((uintptr_t)y_stats | (uintptr_t)r_stats) % 8 != 0 ||
      ((uintptr_t)r_gamma | (uintptr_t)r_beta) % 8 != 0) {
    set_error("linear_residual: x and the packed weight must be 16-byte aligned (x row "
              "stride a multiple of 8 elements), y and the residual 8-byte aligned with row "
              "strides multiples of 4, gamma / beta and the statistics 8-byte aligned");
    return VFL_E_INVALID;
  }
  LinNorm nrm{};
  nrm.res = (const uint16_t *)residual;
  nrm.res_stride = r_stride;
  nrm.res_stats = reinterpret_cast<const float2 *>(r_stats);
  nrm.res_gamma = (const uint16_t *)r_gamma;
  nrm.res_beta = (const uint16_t *)r_beta;
  nrm.res_eps = r_eps;
  nrm.y_stats = reinterpret_cast<float2 *>(y_stats);
  hipStream_t s = (hipStream_t)stream;
  if (xp)
    launch_linear<true, false, false, LIN_RESIDUAL>(s, dtype, x, 0, packed_weight, bias, y,
                                                    y_stride, rows, out_features, in_features,
                                                    true, nrm);
  else
    launch_linear<false, false, false, LIN_RESIDUAL>(s, dtype, x, x_stride, packed_weight,
                                                     bias, y, y_stride, rows, out_features,
                                                     in_features, true, nrm);
  return launch_status("linear_residual");
}

extern "C" int vfl_layer_norm_apply(const void *v, int64_t v_stride, const float *v_stats,
                                    const void *gamma, const void *beta, float eps, void *out,
                                    int64_t out_stride, int64_t rows, int dim, int dtype,
                                    void *stream) {
  clear_error();
  if (dtype != VFL_BFLOAT16 && dtype != VFL_FLOAT16) {
    set_error("layer_norm_apply: dtype %d has no kernel (bf16 and fp16 only)", dtype);
    return VFL_E_UNSUPPORTED;
  }
  if (rows < 0 || dim <= 0 || dim % LIN_STAT_TILE != 0 || v_stride < dim ||
      out_stride < dim || !(eps >= 0.f)) {
    set_error("layer_norm_apply: bad sizes (rows %lld dim %d, a multiple of %d; strides "
              "covering dim; eps >= 0)", (long long)rows, dim, LIN_STAT_TILE);
    return VFL_E_INVALID;
  }
  if (rows == 0) return VFL_OK;
  if (rows > 2LL * 2147483647LL) {
    set_error("layer_norm_apply: too many rows");
    return VFL_E_UNSUPPORTED;
  }
  if (!v || !v_stats || !gamma || !beta || !out) {
    set_error("layer_norm_apply: null pointer argument");
    return VFL_E_INVALID;
  }
  if (((uintptr_t)v | (uintptr_t)out | (uintptr_t)gamma | (uintptr_t)beta |
       (uintptr_t)v_stats) % 8 != 0 || v_stride % 4 != 0 || out_stride % 4 != 0) {
    set_error("layer_norm_apply: v, out, gamma, beta and v_stats must be 8-byte aligned and "
              "the row strides multiples of 4 elements");
    return VFL_E_INVALID;
  }
  const dim3 grid((unsigned)((rows + 1) / 2));
  hipStream_t s = (hipStream_t)stream;
  const float2 *st = reinterpret_cast<const float2 *>(v_stats);
  if (dtype == VFL_BFLOAT16)
    layer_norm_apply_kernel<VFL_BFLOAT16><<<grid, dim3(128), 0, s>>>(
        (const uint16_t *)v, v_stride, st, (const uint16_t *)gamma, (const uint16_t *)beta, eps,
        (uint16_t *)out, out_stride, rows, dim);
  else
    layer_norm_apply_kernel<VFL_FLOAT16><<<grid, dim3(128), 0, s>>>(
        (const uint16_t *)v, v_stride, st, (const uint16_t *)gamma, (const uint16_t *)beta, eps,
        (uint16_t *)out, out_stride, rows, dim);
  return launch_status("layer_norm_apply");
}
