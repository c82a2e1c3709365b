// Encoder self-attention over packed prompts (bf16 / fp16, head size 64), gfx950: every
// prompt of an admitted batch attends over its own tokens, all prompts and heads in one
// launch, read from the fused q|k|v projection's rows and written to rows of the output
// (vflorence/models/bart.py's encoder attention, SDPA there).
//
// What bounds it: the vector work.  Per 32 queries x 64 keys a wave issues 20 matrix
// products (8 for the scores, 8 with V, 4 that sum the weights: 640 cycles) and about 1000
// cycles of vector work, half of it v_exp_f32; two or more waves per SIMD overlap the two.
//
// Tile.  Scores are computed transposed, S^T[key][query] = K Q^T (32x32x16 products), so a
// lane holds one query's column: the softmax reduces inside the lane plus one half-wave
// swap, the output O^T[dim][query] is rescaled by a lane scalar, and the probabilities are
// already in the second product's operand order: its k index runs over the keys in the
// order the first product left them (half-wave hf of step s holds keys 16 s + 4 hf + 0..3
// and 16 s + 8 + 4 hf + 0..3), which V's side follows by reading two 4-key groups.
// Precision: the weights are rounded to the element type for the second product, which
// costs least where the running maximum is exact (the largest weight is 1, unrounded)
// and the normalizer sums the rounded weights -- a third product, with a row of ones, which
// also takes 32 additions per tile off the vector units.  Error against fp64 (2-norm) over
// that of SDPA, which sums the weights unrounded, 12 heads, 2 to 1024 keys, scores of standard
// deviation 0.003 to 16: bf16 0.97-1.00 (flat 2.02e-3 both, 0.25 2.36e-3 / 2.36e-3, 1
// 2.19e-3 / 2.22e-3, 4 1.70e-3 / 1.73e-3), fp16 0.96-1.00 (2.74e-4 / 2.78e-4 at 1); prompts of
// two keys alone reach 1.003.  (A reference that moves only past a slack, as in the decode
// kernels: 2.09e-3 against 1.83e-3 for 4% less time; weights split in two 16-bit terms:
// 1.66e-3 for 25% more.)
// K tiles sit in LDS row by row, 16-byte chunks xor-swizzled by the row against bank
// conflicts; V tiles 4-key interleaved ([group][dim][4], transposed in registers on the
// way in).  Tiles are double-buffered, the next one's loads in flight during the products.
//
// KS key groups: the 4 waves of a workgroup take 128 / KS queries and split the key tiles
// KS ways, merging through LDS at the end; more groups fill the chip for few or short
// prompts (the dispatch rule is at the launch).  A (prompt, head)'s query tiles run on one
// XCD, which then reads its K/V once: workgroup ids go to XCDs round robin, so ids are laid
// out as 8 pairs x tiles.
//
// Measured in graphs against one SDPA launch (without its copies; MI355X, bf16, us):
// 1 x 590 tokens x 12 heads 11.5 against 21.4, 1 x 1024 x 16 heads 16.4 / 41.7, 8 x 300
// 13.8 / 18.5, 16 x 1024 117 / 156 (590 TFLOP/s), 64 x 128 18.7 / 36.3.  48 prompts of 19 to
// 1021 tokens, the whole layer with its projections: 1573 -> 327 us (GEMMs 211 of it).
#include "common.h"
#include "mfma_ops.h"

namespace vfl {

typedef float floatx16_t __attribute__((ext_vector_type(16)));

template <int DT> __device__ __forceinline__ floatx16_t mfma32(uint4 a, uint4 b, floatx16_t c);
template <>
__device__ __forceinline__ floatx16_t mfma32<VFL_BFLOAT16>(uint4 a, uint4 b, floatx16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                 __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
template <>
__device__ __forceinline__ floatx16_t mfma32<VFL_FLOAT16>(uint4 a, uint4 b, floatx16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, a),
                                                __builtin_bit_cast(half8_t, b), c, 0, 0, 0);
}

constexpr int ENC_D = 64;         // head size
constexpr int ENC_KEYS = 64;      // keys per tile
constexpr int ENC_WAVES = 4;
constexpr int ENC_TILE_BYTES = ENC_KEYS * ENC_D * 2;  // one K or V tile
// Runs of equal-length prompts per launch: they travel in the kernel's arguments (no
// device copy per call), 16 bytes each of the 4 KB an argument block may hold.
constexpr int ENC_SEGMENTS = 128;

struct EncSegments {
  int n;
  int first[ENC_SEGMENTS];   // first workgroup
  int start[ENC_SEGMENTS];   // first token
  int count[ENC_SEGMENTS];   // prompts
  int length[ENC_SEGMENTS];  // tokens per prompt
};

// The value of lane l ^ 32 and the lane's own, in some order.
__device__ __forceinline__ void half_pair(float x, float &a, float &b) {
  const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  a = __uint_as_float(s[0]);
  b = __uint_as_float(s[1]);
}

template <int DT, int KS>
__global__ __launch_bounds__(64 * ENC_WAVES) void encoder_attention_kernel(
    const uint16_t *__restrict__ q, const uint16_t *__restrict__ k,
    const uint16_t *__restrict__ v, int64_t stride, uint16_t *__restrict__ out,
    int64_t out_stride, int H, float scale_log2, EncSegments segs) {
  constexpr int GW = ENC_WAVES / KS;       // waves per key group
  constexpr int QT = 32 * GW;              // queries per workgroup
  constexpr int GT = 64 * GW;              // threads per key group
  constexpr int KC = ENC_KEYS * 8 / GT;    // 16-byte K chunks per thread and tile
  constexpr int VU = ENC_KEYS * 4 / GT;    // 4-key x 4-dim V units per thread and tile
  // [buffer][key group][K tile, V tile]; the merge reuses it
  __shared__ __align__(16) uint8_t s_tile[2 * KS * 2 * ENC_TILE_BYTES];
  static_assert(KS == 1 || (ENC_WAVES - GW) * (64 * 34 * 4) <= (int)sizeof(s_tile),
                "the partial outputs fit the tile buffers");

  int seg = 0;
  for (int hi = segs.n; hi - seg > 1;) {  // the last run whose first workgroup is <= ours
    const int mid = (seg + hi) / 2;
    if (segs.first[mid] <= (int)blockIdx.x) seg = mid;
    else hi = mid;
  }
  const int L = segs.length[seg];
  const int tiles = (L + QT - 1) / QT;
  const int u = (int)blockIdx.x - segs.first[seg];
  const int pair = 8 * (u / 8 / tiles) + u % 8;
  if (pair >= segs.count[seg] * H) return;  // workgroup-uniform
  const int q0 = (u / 8 % tiles) * QT;
  const int h = pair % H;
  const int64_t row0 = segs.start[seg] + (int64_t)(pair / H) * L;
  q += row0 * stride + h * ENC_D;
  k += row0 * stride + h * ENC_D;
  v += row0 * stride + h * ENC_D;

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int grp = wave / GW, gw = wave % GW;  // key group, wave within it
  const int gt = threadIdx.x % GT;
  const int col = lane & 31, hf = lane >> 5;
  uint8_t *tile0 = s_tile + grp * 2 * ENC_TILE_BYTES;
  constexpr int BUF = KS * 2 * ENC_TILE_BYTES;

  const int query = q0 + 32 * gw + col;
  uint4 qop[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk)
    qop[kk] = *reinterpret_cast<const uint4 *>(q + (int64_t)min(query, L - 1) * stride +
                                               16 * kk + 8 * hf);

  uint4 kr[KC];
  uint2 vr[VU][4];
  auto load = [&](int t) {  // keys past the prompt are zeros
#pragma unroll
    for (int i = 0; i < KC; ++i) {
      const int idx = gt + GT * i, key = t * ENC_KEYS + idx / 8;
      kr[i] = make_uint4(0, 0, 0, 0);
      if (key < L)
        kr[i] = *reinterpret_cast<const uint4 *>(k + (int64_t)key * stride + 8 * (idx % 8));
    }
#pragma unroll
    for (int i = 0; i < VU; ++i) {
      const int idx = gt + GT * i, key = t * ENC_KEYS + 4 * (idx / 16);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        vr[i][j] = make_uint2(0, 0);
        if (key + j < L)
          vr[i][j] = *reinterpret_cast<const uint2 *>(v + (int64_t)(key + j) * stride +
                                                      4 * (idx % 16));
      }
    }
  };
  auto store = [&](int buf) {
    uint8_t *kt = tile0 + buf * BUF, *vt = kt + ENC_TILE_BYTES;
#pragma unroll
    for (int i = 0; i < KC; ++i) {
      const int idx = gt + GT * i, r = idx / 8, c = idx % 8;
      *reinterpret_cast<uint4 *>(kt + r * 128 + ((c ^ (r & 7)) << 4)) = kr[i];
    }
#pragma unroll
    for (int i = 0; i < VU; ++i) {
      const int idx = gt + GT * i;
      const uint2 a = vr[i][0], b = vr[i][1], c = vr[i][2], d = vr[i][3];
      constexpr uint32_t LO = 0x05040100u, HI = 0x07060302u;
      uint4 *dst = reinterpret_cast<uint4 *>(vt + idx * 32);
      dst[0] = make_uint4(__builtin_amdgcn_perm(b.x, a.x, LO), __builtin_amdgcn_perm(d.x, c.x, LO),
                          __builtin_amdgcn_perm(b.x, a.x, HI), __builtin_amdgcn_perm(d.x, c.x, HI));
      dst[1] = make_uint4(__builtin_amdgcn_perm(b.y, a.y, LO), __builtin_amdgcn_perm(d.y, c.y, LO),
                          __builtin_amdgcn_perm(b.y, a.y, HI), __builtin_amdgcn_perm(d.y, c.y, HI));
    }
  };

  floatx16_t o[2];
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[b][i] = 0.f;
  float m = NEG_INF_F, l = 0.f;
  const uint32_t one2 = DT == VFL_BFLOAT16 ? 0x3f803f80u : 0x3c003c00u;
  const uint4 ones = make_uint4(one2, one2, one2, one2);

  auto attend = [&](int t, int buf) {
    const uint8_t *kt = tile0 + buf * BUF, *vt = kt + ENC_TILE_BYTES;
    floatx16_t s[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
#pragma unroll
      for (int i = 0; i < 16; ++i) s[b][i] = 0.f;
      const int r = 32 * b + col;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        const uint4 kop = *reinterpret_cast<const uint4 *>(
            kt + r * 128 + (((2 * kk + hf) ^ (r & 7)) << 4));
        s[b] = mfma32<DT>(kop, qop[kk], s[b]);
      }
    }
    if ((t + 1) * ENC_KEYS > L) {
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (t * ENC_KEYS + 32 * b + 8 * (i / 4) + 4 * hf + i % 4 >= L) s[b][i] = NEG_INF_F;
    }
    float mx = NEG_INF_F;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[b][i]);
    float ma, mb;
    half_pair(mx, ma, mb);
    mx = fmaxf(ma, mb) * scale_log2;
    const bool need = mx > m;
    if (__builtin_amdgcn_ballot_w64(need) != 0) {
      const float corr = need ? fast_exp2(m - mx) : 1.f;
      l *= corr;
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[b][i] *= corr;
      m = need ? mx : m;
    }
    const float ms = m == NEG_INF_F ? 0.f : m;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[b][i] = fast_exp2(fmaf(s[b][i], scale_log2, -ms));
    floatx16_t sum;  // every row: the tile's weights summed over its keys
#pragma unroll
    for (int i = 0; i < 16; ++i) sum[i] = 0.f;
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      const int e = 8 * (st & 1);
      const floatx16_t &p = s[st >> 1];
      const uint4 pop = make_uint4(Mfma<DT>::narrow2(p[e], p[e + 1]),
                                   Mfma<DT>::narrow2(p[e + 2], p[e + 3]),
                                   Mfma<DT>::narrow2(p[e + 4], p[e + 5]),
                                   Mfma<DT>::narrow2(p[e + 6], p[e + 7]));
      sum = mfma32<DT>(ones, pop, sum);
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const uint8_t *vp = vt + ((4 * st + hf) * ENC_D + 32 * b + col) * 8;
        const uint2 v0 = *reinterpret_cast<const uint2 *>(vp);
        const uint2 v1 = *reinterpret_cast<const uint2 *>(vp + 2 * ENC_D * 8);
        o[b] = mfma32<DT>(make_uint4(v0.x, v0.y, v1.x, v1.y), pop, o[b]);
      }
    }
    l += sum[0];
  };

  // Step t: the group's tile of step t is in buffer t & 1, the next one's rows in flight.
  const int ntiles = (L + ENC_KEYS - 1) / ENC_KEYS;
  const int steps = (ntiles + KS - 1) / KS;
  load(grp);
  store(0);
  if (steps > 1) load(KS + grp);
  __syncthreads();
  for (int t = 0; t < steps; ++t) {
    if (t + 1 < steps) {
      store((t + 1) & 1);
      if (t + 2 < steps) load((t + 2) * KS + grp);
    }
    if (t * KS + grp < ntiles) attend(t * KS + grp, t & 1);
    __syncthreads();
  }

  if constexpr (KS > 1) {
    float *part = reinterpret_cast<float *>(s_tile);  // [wave - GW][34][64]
    if (grp > 0) {
      float *dst = part + (wave - GW) * 34 * 64 + lane;
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) dst[(16 * b + i) * 64] = o[b][i];
      dst[32 * 64] = m;
      dst[33 * 64] = l;
    }
    __syncthreads();
    if (grp > 0) return;
    float M = m;
#pragma unroll
    for (int g = 1; g < KS; ++g) M = fmaxf(M, part[((g - 1) * GW + gw) * 34 * 64 + 32 * 64 + lane]);
    const float Ms = M == NEG_INF_F ? 0.f : M;
    const float f0 = fast_exp2(m - Ms);
    l *= f0;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[b][i] *= f0;
#pragma unroll
    for (int g = 1; g < KS; ++g) {
      const float *src = part + ((g - 1) * GW + gw) * 34 * 64 + lane;
      const float f = fast_exp2(src[32 * 64] - Ms);
      l = fmaf(src[33 * 64], f, l);
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[b][i] = fmaf(src[(16 * b + i) * 64], f, o[b][i]);
    }
  }
  if (query >= L) return;
  // l is 0 only where every score was -inf: NaN, as softmax gives
  const float inv = 1.f / l;
  uint16_t *dst = out + (row0 + query) * out_stride + h * ENC_D + 4 * hf;
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<uint2 *>(dst + 32 * b + 8 * i) =
          make_uint2(Mfma<DT>::narrow2(o[b][4 * i] * inv, o[b][4 * i + 1] * inv),
                     Mfma<DT>::narrow2(o[b][4 * i + 2] * inv, o[b][4 * i + 3] * inv));
}

}  // namespace vfl

using namespace vfl;

template <int DT, int KS>
static void launch_encoder(const void *q, const void *k, const void *v, int64_t stride, void *out,
                           int64_t out_stride, int H, float scale_log2, const EncSegments &segs,
                           int64_t groups, hipStream_t s) {
  encoder_attention_kernel<DT, KS><<<dim3((unsigned)groups), dim3(64 * ENC_WAVES), 0, s>>>(
      (const uint16_t *)q, (const uint16_t *)k, (const uint16_t *)v, stride, (uint16_t *)out,
      out_stride, H, scale_log2, segs);
}

extern "C" int vfl_encoder_attention(const void *q, const void *k, const void *v, int64_t stride,
                                     void *out, int64_t out_stride, int64_t num_tokens,
                                     const int64_t *segments, int64_t num_segments,
                                     int num_heads, int head_dim, float scale, int dtype,
                                     void *stream) {
  clear_error();
  if ((dtype != VFL_BFLOAT16 && dtype != VFL_FLOAT16) || head_dim != ENC_D) {
    set_error("encoder_attention: no kernel for dtype %d head_dim %d", dtype, head_dim);
    return VFL_E_UNSUPPORTED;
  }
  if (num_tokens < 0 || num_segments < 0 || num_heads <= 0 || num_heads > 65535 ||
      stride < (int64_t)num_heads * head_dim || out_stride < (int64_t)num_heads * head_dim ||
      !(scale > 0.f)) {
    set_error("encoder_attention: bad sizes (tokens %lld segments %lld heads %d strides %lld "
              "%lld scale %g)",
              (long long)num_tokens, (long long)num_segments, num_heads, (long long)stride,
              (long long)out_stride, (double)scale);
    return VFL_E_INVALID;
  }
  if (num_tokens > 2147483647LL) {
    set_error("encoder_attention: too many tokens");
    return VFL_E_UNSUPPORTED;
  }
  if (num_segments == 0) return VFL_OK;
  if (!segments || !q || !k || !v || !out) {
    set_error("encoder_attention: null pointer argument");
    return VFL_E_INVALID;
  }
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v) % 16 != 0 || stride % 8 != 0 ||
      (uintptr_t)out % 8 != 0 || out_stride % 4 != 0) {
    set_error("encoder_attention: q, k and v must be 16-byte aligned with a row stride that is "
              "a multiple of 8 elements, out 8-byte aligned with one that is a multiple of 4");
    return VFL_E_INVALID;
  }
  int64_t wide = 0, longest = 0;  // workgroups of 128 queries; tokens of the longest prompt
  for (int64_t i = 0; i < num_segments; ++i) {
    const int64_t *sg = segments + 3 * i;
    if (sg[0] < 0 || sg[1] < 0 || sg[2] < 0 || sg[0] > num_tokens || sg[2] > num_tokens ||
        (sg[2] > 0 && sg[1] > (num_tokens - sg[0]) / sg[2])) {
      set_error("encoder_attention: segment %lld (start %lld, %lld prompts of %lld tokens) lies "
                "outside the %lld tokens",
                (long long)i, (long long)sg[0], (long long)sg[1], (long long)sg[2],
                (long long)num_tokens);
      return VFL_E_INVALID;
    }
    wide += sg[1] * num_heads * ((sg[2] + 127) / 128);
    if (sg[1] > 0 && sg[2] > longest) longest = sg[2];
  }
  // Key groups by how far 128-query workgroups would leave the 256 CUs idle, up to one per
  // key tile.  One / two / four groups, us: 12 workgroups of one key tile 4.2 / 4.7 / 5.5, 24
  // workgroups 8.1 / 6.4 / 5.6, 60 15.4 / 11.5 / 18.9, 128 22.3 / 16.4 / 23.9, 160 15.9 /
  // 15.7 / 27.7, 384 13.8 / 17.0 / 34.2 (the groups' tile buffers leave one workgroup of four
  // groups, two of two on a CU).
  int ks = wide <= 32 ? 4 : (wide <= 192 ? 2 : 1);
  while (ks > 1 && ENC_KEYS * (ks / 2) >= longest) ks /= 2;
  const int qt = 128 / ks;
  const float scale_log2 = (float)((double)scale * 1.4426950408889634);
  hipStream_t s = (hipStream_t)stream;
  // Longest prompts first, so that the short ones fill the end of the launch.
  int64_t done = 0;
  while (done < num_segments) {
    EncSegments args;
    args.n = 0;
    int64_t groups = 0;
    const int64_t stop = num_segments - done < ENC_SEGMENTS ? num_segments - done : ENC_SEGMENTS;
    int order[ENC_SEGMENTS];
    for (int i = 0; i < (int)stop; ++i) {
      int at = i;
      for (; at > 0 && segments[3 * (done + order[at - 1]) + 2] < segments[3 * (done + i) + 2]; --at)
        order[at] = order[at - 1];
      order[at] = i;
    }
    for (int i = 0; i < (int)stop; ++i) {
      const int64_t *sg = segments + 3 * (done + order[i]);
      if (sg[1] == 0 || sg[2] == 0) continue;
      args.first[args.n] = (int)groups;
      args.start[args.n] = (int)sg[0];
      args.count[args.n] = (int)sg[1];
      args.length[args.n] = (int)sg[2];
      ++args.n;
      groups += (sg[1] * num_heads + 7) / 8 * 8 * ((sg[2] + qt - 1) / qt);
      if (groups > 2147483647LL) {
        set_error("encoder_attention: too many prompts x heads for one grid");
        return VFL_E_UNSUPPORTED;
      }
    }
    done += stop;
    if (args.n == 0) continue;
#define VFL_ENC(DT)                                                                             \
  (ks == 1 ? launch_encoder<DT, 1>(q, k, v, stride, out, out_stride, num_heads, scale_log2, args, \
                                   groups, s)                                                   \
   : ks == 2                                                                                    \
       ? launch_encoder<DT, 2>(q, k, v, stride, out, out_stride, num_heads, scale_log2, args,   \
                               groups, s)                                                       \
       : launch_encoder<DT, 4>(q, k, v, stride, out, out_stride, num_heads, scale_log2, args,   \
                               groups, s))
    if (dtype == VFL_BFLOAT16) VFL_ENC(VFL_BFLOAT16);
    else VFL_ENC(VFL_FLOAT16);
#undef VFL_ENC
    const int st = launch_status("encoder_attention");
    if (st != VFL_OK) return st;
  }
  return VFL_OK;
}
