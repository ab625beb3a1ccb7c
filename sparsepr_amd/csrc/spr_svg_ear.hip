// SVG-EAR routing scores: per (query head, query centroid, key cluster) the log
// value-error score of N8's default selector and the log attention mass.
//
// Replaces:
//   _svg_ear_value_error_kernel + svg_ear_value_error_scores_triton
//       (src/sparsepr/kernels/triton/svg_ear.py:95-192, :453-531)
//   _svg_ear_grouped_value_error_kernel + svg_ear_grouped_value_error_scores_triton
//       (svg_ear.py:195-286, :534-600): the same scores, one K/V walk per GQA group
//   _attention_mass_score_kernel + attention_mass_scores_triton (svg_ear.py:7-92, :372-450)
//
// Scores, for query centroid q and the tokens t of key cluster c (k, v bf16):
//   l_t = (q~ . k_t) / sqrt(D), q~ = q rounded to TF32 (the reference's tl.dot
//         input_precision="tf32"), l_c = (q . kc) / sqrt(D) (+ Jensen term)
//   value error: m = max(l_c, max_t l_t), w_c = e^(l_c - m), w_t = e^(l_t - m),
//       E = sum_t max(w_c^2 |vc|^2 + w_t^2 |v_t|^2 - 2 w_t w_c (v_t . vc), 0)
//       score = log(max(E / n_c, 1e-30)) + 2 m;  -inf for an empty cluster
//   attention mass: score = log(max(sum_t e^(l_t - m), 1e-30)) + m, m = max_t l_t
// The weights are taken against a reference that starts at l_c (the mass: at the first
// chunk's maximum) and moves only when a logit passes it by SE_SLACK (less where |v|^2 is large),
// with the sums rescaled; the scores do not depend on it but for rounding.
//
// Layout.  A first kernel writes the centroid logits l_c [query head, centroid, cluster]
// (fp32 dot products over d, sequential, 128 rows x 32 clusters per workgroup) into the score
// buffer; the score kernel overwrites each entry with its score.  The score kernel runs one
// workgroup per CU for (query head, 8 consecutive key clusters, up to 320 query rows): a wave
// per 32-row query block (two for up to five blocks, each folding every other chunk), two
// waves for the statistics of V, at most twelve, three per SIMD.  K and V are walked once for
// all rows.  Calls of up to 128 rows with many short clusters take four waves, one chunk per
// barrier and half the LDS, two workgroups per CU (the host's rule).  The clusters' tokens are one
// contiguous run, walked in 32-token chunks (a chunk never spans two clusters), whose K and V rows
// are DMA'd into swizzled LDS tiles (16-byte piece p of token row t at slot p ^ (t % 16): the MFMA
// fragment reads hit 16 distinct slots per 16 lanes) two steps ahead.  A query wave forms
// S^T = K Q~^T by 16 bf16 MFMAs per chunk: q~ is split into bf16 hi + lo with hi + lo == q~ exactly (q~ has 11
// significant bits, hi the top 8, lo the next 3), so every product is the reference's TF32
// product exactly and only the fp32 summation order differs.  |v_t|^2 and v_t . vc are products
// of the V tile with itself and with the three bf16 pieces of vc, a chunk ahead of their use.
//
// What bounds it: the folding, 5 VALU operations, an exponential (16 cycles) and half a max
// per (centroid, token) pair beside the MFMAs, which a wave does not overlap with its own
// (computing S a chunk ahead needs more registers than three waves per SIMD have, and with two to
// a CU it changed nothing).  Both kernels, against four waves per 128 rows that walked K and V again
// for every 128 rows and took the statistics of V on all their lanes: 24 heads x 118,800 tokens,
// 300 x 1000 1.37 -> 1.02 ms; 180 x 512 at 70,000 tokens 0.61 -> 0.46 ms; 128 x 512 at 118,800 0.51
// -> 0.51 ms; 6 heads x 9,000 tokens, 23 x 64 99 -> 61 us.  One wave for the statistics instead of
// two holds the others up (128 x 512: 0.64 ms); one chunk per barrier costs 5 %.
// The token runs come from a block prefix sum of the sizes and are clamped to the stored
// tokens, so no size vector can make the kernel read outside K or V.
#include <type_traits>

#include "spr_common.h"

namespace {

using spr::f32x16;
using spr::f32x4;
using spr::u32x4;

constexpr int SE_D = 128;
constexpr int SE_THREADS = 256;
constexpr int SE_CHUNK = 32;  // tokens per chunk: one 32-row MFMA block
constexpr int SE_KSTEPS = SE_D / 16;
constexpr float SE_LOG2E = 1.4426950408889634f;

// Round to TF32 (10 stored mantissa bits), to nearest with ties away from zero.
__device__ __forceinline__ float tf32_rna(float x) {
  return __uint_as_float((__float_as_uint(x) + 0x1000u) & 0xffffe000u);
}

__device__ __forceinline__ float exp_fast(float x) { return __builtin_amdgcn_exp2f(x * SE_LOG2E); }

// log(x) + y for x >= 0, rounded once: with the reference at the centroid logit the two can be large
// and of opposite signs, and a log rounded by itself would show in a small score.
__device__ __forceinline__ float log_plus(float x, double y) {
  int e = 0;
  const float m = frexpf(x, &e);
  return static_cast<float>(y + (0.6931471805599453 * e + static_cast<double>(logf(m))));
}

__device__ __forceinline__ float wave_sum(float v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

template <int CTRL>
__device__ __forceinline__ float dpp_mov(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}

// max / sum over lanes l and l ^ 32: v_permlane32_swap of x with itself gives the
// lower half-wave's value in the first result and the upper half's in the second on
// every lane, so both lanes of a pair combine the same two operands in the same order.
__device__ __forceinline__ float max_xor32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sum_xor32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// max over the wave: quad_perm [1, 0, 3, 2] and [2, 3, 0, 1], row_half_mirror and row_mirror give
// each lane its row of 16, the swaps the four rows
__device__ __forceinline__ float wave_max(float x) {
  x = fmaxf(x, dpp_mov<0xB1>(x));
  x = fmaxf(x, dpp_mov<0x4E>(x));
  x = fmaxf(x, dpp_mov<0x141>(x));
  x = fmaxf(x, dpp_mov<0x140>(x));
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return max_xor32(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
}

constexpr int SE_ROW = SE_D * 2;  // bytes per bf16 token row
constexpr int CL_CLUSTERS = 32;   // clusters per centroid-logit workgroup
constexpr int CL_PITCH = SE_D + 4;  // floats per centroid row in LDS
constexpr int CL_ROWS = 2 * (SE_THREADS / 4);  // query rows per centroid-logit workgroup

// l_c = (q . kc) / sqrt(D) (+ 0.5 min(sum_d q_d^2 var_d / D, cap)) for CL_ROWS query rows x
// CL_CLUSTERS clusters per workgroup: thread -> query rows tid / 4 and tid / 4 + CL_ROWS / 2,
// clusters tid % 4 + 4 j, j < 8 (each centroid read from LDS serves two rows, and the four
// neighbours' rows of CL_PITCH floats lie in distinct banks: 90 -> 68 us for 24 heads of
// 300 x 1000 against clusters 8 (tid % 4) + j of unpadded rows, four to a bank); fp32 fma
// chains over d in order.  Written to out [qh, qn, kn].
__global__ __launch_bounds__(SE_THREADS) void svg_ear_centroid_logit_kernel(
    const float* __restrict__ qc, const float* __restrict__ kcent, const float* __restrict__ var_k, float cap,
    int32_t qn, int32_t kn, int32_t group, float* __restrict__ out) {
  __shared__ __attribute__((aligned(16))) float kc_l[CL_CLUSTERS][CL_PITCH];
  __shared__ __attribute__((aligned(16))) float var_l[CL_CLUSTERS][CL_PITCH];
  const int64_t qh = blockIdx.z;
  const int64_t kh = qh / group;
  const int cb = blockIdx.x * CL_CLUSTERS;
  const int ncl = min(CL_CLUSTERS, kn - cb);
  const int tid = threadIdx.x;
  const float scale = 1.0f / 11.313708498984761f;
  for (int i = tid; i < CL_CLUSTERS * SE_D / 4; i += SE_THREADS) {
    const int c = i / (SE_D / 4), d = 4 * (i % (SE_D / 4));
    const bool live = c < ncl;
    const int64_t o = (kh * kn + cb + c) * SE_D + d;
    *reinterpret_cast<float4*>(&kc_l[c][d]) =
        live ? *reinterpret_cast<const float4*>(kcent + o) : float4{0.0f, 0.0f, 0.0f, 0.0f};
    *reinterpret_cast<float4*>(&var_l[c][d]) =
        (live && var_k != nullptr) ? *reinterpret_cast<const float4*>(var_k + o) : float4{0.0f, 0.0f, 0.0f, 0.0f};
  }
  __syncthreads();
  const int r0 = blockIdx.y * CL_ROWS + tid / 4;
  const int r1 = r0 + CL_ROWS / 2;
  const int c0 = tid % 4;
  if (r0 >= qn) return;
  const float* qrow0 = qc + (qh * qn + r0) * SE_D;
  const float* qrow1 = qc + (qh * qn + min(r1, qn - 1)) * SE_D;  // a row past qn computes, stores nothing
  float dot0[8], s20[8], dot1[8], s21[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) dot0[j] = s20[j] = dot1[j] = s21[j] = 0.0f;
  for (int d0 = 0; d0 < SE_D; d0 += 4) {
    const float4 qa = *reinterpret_cast<const float4*>(qrow0 + d0);
    const float4 qb = *reinterpret_cast<const float4*>(qrow1 + d0);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float4 kv = *reinterpret_cast<const float4*>(&kc_l[c0 + 4 * j][d0]);
      dot0[j] = __builtin_fmaf(qa.x, kv.x, dot0[j]);
      dot0[j] = __builtin_fmaf(qa.y, kv.y, dot0[j]);
      dot0[j] = __builtin_fmaf(qa.z, kv.z, dot0[j]);
      dot0[j] = __builtin_fmaf(qa.w, kv.w, dot0[j]);
      dot1[j] = __builtin_fmaf(qb.x, kv.x, dot1[j]);
      dot1[j] = __builtin_fmaf(qb.y, kv.y, dot1[j]);
      dot1[j] = __builtin_fmaf(qb.z, kv.z, dot1[j]);
      dot1[j] = __builtin_fmaf(qb.w, kv.w, dot1[j]);
      if (var_k != nullptr) {
        const float4 vv = *reinterpret_cast<const float4*>(&var_l[c0 + 4 * j][d0]);
        s20[j] = __builtin_fmaf(qa.x * qa.x, vv.x, s20[j]);
        s20[j] = __builtin_fmaf(qa.y * qa.y, vv.y, s20[j]);
        s20[j] = __builtin_fmaf(qa.z * qa.z, vv.z, s20[j]);
        s20[j] = __builtin_fmaf(qa.w * qa.w, vv.w, s20[j]);
        s21[j] = __builtin_fmaf(qb.x * qb.x, vv.x, s21[j]);
        s21[j] = __builtin_fmaf(qb.y * qb.y, vv.y, s21[j]);
        s21[j] = __builtin_fmaf(qb.z * qb.z, vv.z, s21[j]);
        s21[j] = __builtin_fmaf(qb.w * qb.w, vv.w, s21[j]);
      }
    }
  }
  auto store = [&](int r, const float (&dot)[8], const float (&s2)[8]) {
    float* orow = out + (qh * qn + r) * kn + cb + c0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (c0 + 4 * j < ncl) {
        float l = dot[j] * scale;
        if (var_k != nullptr) l += 0.5f * fminf(s2[j] / static_cast<float>(SE_D), cap);
        orow[4 * j] = l;
      }
    }
  };
  store(r0, dot0, s20);
  if (r1 < qn) store(r1, dot1, s21);
}

constexpr int SE_CPW = 8;     // key clusters per workgroup
constexpr int SE_SWAVES = 2;  // waves that take the V statistics
// A workgroup of the score kernel walks STEP chunks per barrier.
template <int STEP>
struct Step {
  static constexpr int QWAVES = STEP == 2 ? 10 : 4;  // the most query waves
  static constexpr int TILES = 4 * STEP;             // chunks of K in LDS
  static constexpr int VTILES = 3 * STEP;            // chunks of V, whose statistics are taken a step ahead
  static constexpr int STATS = 2 * STEP;             // chunks whose statistics are kept
};
constexpr int SE_TILE = SE_CHUNK * SE_ROW;  // bytes of a K or V tile
// A running reference is moved once a chunk's largest logit passes it by this much, or by less
// where the squared weights times the chunk's largest |v|^2, over all the cluster's tokens, would
// pass 2^123: whatever the values, the sums are finite where they are against the largest logit.
constexpr float SE_SLACK = 30.0f;

template <int MODE, int STEP>  // 0: value error (scores holds l_c on entry), 1: attention mass
__global__ __launch_bounds__(64 * (STEP == 2 ? Step<2>::QWAVES + SE_SWAVES : 4), STEP == 2 ? 3 : 2) void svg_ear_score_kernel(
    const float* __restrict__ qc, const uint16_t* __restrict__ ks, const uint16_t* __restrict__ vs,
    const float* __restrict__ vcent, const int32_t* __restrict__ k_sizes, int32_t qn, int32_t kn, int64_t t_stored,
    int32_t group, int32_t qgroups, int32_t qwaves, int32_t sets, float* __restrict__ scores) {
  using S = Step<STEP>;
  __shared__ __attribute__((aligned(1024))) uint8_t k_tiles[S::TILES * SE_TILE];
  __shared__ __attribute__((aligned(1024))) uint8_t v_tiles[MODE == 0 ? S::VTILES * SE_TILE : 16];
  // the value centroids as three bf16 pieces whose sum they are, and a row of zeros
  __shared__ __attribute__((aligned(16))) uint16_t vc_l[MODE == 0 ? 3 * SE_CPW + 1 : 1][SE_D];
  __shared__ __attribute__((aligned(16))) float vn_l[S::STATS][SE_CHUNK];  // |v_t|^2
  __shared__ __attribute__((aligned(16))) float cd_l[S::STATS][SE_CHUNK];  // -2 v_t . vc
  __shared__ float slack_l[S::STATS][2];  // the chunk's, the less of the two: at most SE_SLACK
  __shared__ float vc2_l[SE_CPW];
  // per cluster and row of a q wave: the sum, the reference it is taken against, the largest logit
  __shared__ float es_l[SE_CPW][32 * S::QWAVES];
  __shared__ float rf_l[SE_CPW][32 * S::QWAVES];
  __shared__ float tp_l[SE_CPW][32 * S::QWAVES];
  __shared__ int32_t len_l[SE_CPW];  // tokens in each run (clamped)
  __shared__ int64_t red_l[S::QWAVES + SE_SWAVES];

  // Workgroup b runs on XCD b % 8: the query groups of the same clusters follow one another
  // there and find K and V in its L2.
  const int turn = blockIdx.x / 8;
  const int c_begin = (turn / qgroups * 8 + static_cast<int>(blockIdx.x % 8)) * SE_CPW;
  if (c_begin >= kn) return;
  const int q0 = turn % qgroups * (32 * qwaves);
  const int ncl = min(SE_CPW, kn - c_begin);
  const int64_t qh = blockIdx.y;
  const int64_t kh = qh / group;
  const int tid = threadIdx.x;
  const int nthr = blockDim.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31;
  const int half = lane >> 5;
  const float scale = 1.0f / 11.313708498984761f;  // 1 / sqrt(128), as the fp32 quotient
  // wave w < qwaves * sets folds query block w % qwaves; with two sets each folds every other
  // chunk and the sums meet at the end
  const int set = wave / qwaves;
  const int q = q0 + 32 * (wave % qwaves) + col;
  const bool q_wave = set < sets && q0 + 32 * (wave % qwaves) < qn;
  // Who takes the statistics of V: at STEP 2 two waves of their own (stat 0 and 1), a chunk of a
  // step each; at STEP 1 waves 2 and 3, a half of every chunk's, or with three or four query waves
  // all four, a quarter each.
  const int stat = wave - qwaves * sets;
  const bool quarters = STEP == 1 && qwaves > 2;
  const int rows = 32 * qwaves;

  // the query rows on their way while the rest is set up (rows past the end read the last one,
  // waves without a block store nothing of theirs)
  const float* qrow = qc + (qh * qn + min(q, qn - 1)) * SE_D + 8 * half;
  float4 qraw[2 * SE_KSTEPS];
#pragma unroll
  for (int s = 0; s < SE_KSTEPS; ++s) {
    qraw[2 * s] = *reinterpret_cast<const float4*>(qrow + 16 * s);
    qraw[2 * s + 1] = *reinterpret_cast<const float4*>(qrow + 16 * s + 4);
  }
  // every sum starts empty, against l_c (written by svg_ear_centroid_logit_kernel)
  for (int i = tid; i < SE_CPW * rows; i += nthr) {
    const int j = i % SE_CPW, r = i / SE_CPW;
    float l = -__builtin_huge_valf();
    if (MODE == 0 && j < ncl && q0 + r < qn) l = scores[(qh * qn + q0 + r) * kn + c_begin + j];
    for (int t = 0; t < sets; ++t) {
      es_l[j][t * rows + r] = 0.0f;
      rf_l[j][t * rows + r] = l;
      tp_l[j][t * rows + r] = l;
    }
  }
  // ---- token runs of clusters c_begin .. c_begin + ncl - 1 (negative sizes count as 0)
  const int32_t* sz = k_sizes + kh * kn;
  const int32_t own = lane < ncl ? max(sz[c_begin + lane], 0) : 0;
  int64_t part = 0;
  for (int j = tid; j < c_begin; j += nthr) part += max(sz[j], 0);
  for (int o = 32; o > 0; o >>= 1) part += __shfl_xor(part, o, 64);
  if (lane == 0) red_l[wave] = part;
  if (MODE == 0) {
    for (int i = tid; i < SE_CPW * SE_D; i += nthr) {
      const int j = i / SE_D, d = i % SE_D;
      const float v = j < ncl ? vcent[(kh * kn + c_begin + j) * SE_D + d] : 0.0f;
      const uint32_t hi = __float_as_uint(v) & 0xffff0000u;
      const float r1 = v - __uint_as_float(hi);
      const uint32_t mid = __float_as_uint(r1) & 0xffff0000u;
      vc_l[3 * j][d] = static_cast<uint16_t>(hi >> 16);
      vc_l[3 * j + 1][d] = static_cast<uint16_t>(mid >> 16);
      vc_l[3 * j + 2][d] = spr::f32_to_bf16(r1 - __uint_as_float(mid));
    }
    for (int i = tid; i < SE_D; i += nthr) vc_l[3 * SE_CPW][i] = 0;
    for (int j = wave; j < ncl; j += nthr / 64) {
      const float* vr = vcent + (kh * kn + c_begin + j) * SE_D;
      const float x = vr[2 * lane], y = vr[2 * lane + 1];
      const float s2 = wave_sum(__builtin_fmaf(x, x, y * y));
      if (lane == 0) vc2_l[j] = s2;
    }
  }
  __syncthreads();
  // lane j holds cluster j's run (first stored token and length, clamped); the walks are scalar
  int64_t before = 0;
  for (int w = 0; w < nthr / 64; ++w) before += red_l[w];
  int64_t upto = own;
  for (int o = 1; o < SE_CPW; o <<= 1) {
    const int64_t up = __shfl_up(upto, o, 64);
    if (lane >= o) upto += up;
  }
  const int32_t run_start = static_cast<int32_t>(min(before + upto - own, t_stored));
  const int32_t run_len = static_cast<int32_t>(min(before + upto, t_stored)) - run_start;
  if (wave == 0 && lane < SE_CPW) len_l[lane] = run_len;  // read behind the last barrier
  const uint32_t filled = static_cast<uint32_t>(__ballot(lane < ncl && run_len > 0));
  struct Walk {
    int j, c0, len, start;  // cluster, first token of the chunk in it, its run
  };
  auto enter = [&](Walk& w, int from) {  // the first cluster with tokens at or after `from`; j = SE_CPW if none
    const uint32_t rest = filled & ~((1u << from) - 1u);
    w.j = rest != 0 ? __builtin_ctz(rest) : SE_CPW;
    w.c0 = 0;
    w.len = __builtin_amdgcn_readlane(run_len, w.j % SE_CPW);
    w.start = __builtin_amdgcn_readlane(run_start, w.j % SE_CPW);
  };
  auto advance = [&](Walk& w) {
    w.c0 += SE_CHUNK;
    if (w.c0 >= w.len) enter(w, w.j + 1);
  };
  auto inside = [](const Walk& w) { return w.j < SE_CPW; };

  // ---- K/V chunks land in LDS by DMA: 32 token rows of 256 bytes per tile; waves 0 .. 3 move
  // rows 4 w .. 4 w + 3 and 16 + 4 w .. + 3 (1 KB per instruction).  The lane that fills slot p
  // of row t fetches piece p ^ (t % 16) (the swizzle of the MFMA reads).  Rows past the
  // cluster's run hold the next cluster's tokens (masked in the scores); rows past the stored
  // tokens read as zero (buffer bounds).
  const spr::i32x4_s k_desc = spr::buffer_desc(ks + kh * t_stored * SE_D, static_cast<int32_t>(t_stored * SE_ROW));
  const spr::i32x4_s v_desc =
      spr::buffer_desc(MODE == 0 ? vs + kh * t_stored * SE_D : ks, static_cast<int32_t>(t_stored * SE_ROW));
  auto dma = [&](const Walk& w, int kt, int vt) {
    if (wave < 4) {
      const int r0 = 4 * wave, row = r0 + (lane >> 4);  // and 16 rows on, where the swizzle is the same
      const int32_t off = (w.start + w.c0 + row) * SE_ROW + (((lane ^ row) & 15) << 4);
      auto rows = [&](spr::i32x4_s desc, const uint8_t* tile) {
        spr::lds_dma16x2(desc, tile + r0 * SE_ROW, off, desc, tile + (r0 + 16) * SE_ROW, off + 16 * SE_ROW);
      };
      rows(k_desc, k_tiles + kt);
      if (MODE == 0) rows(v_desc, v_tiles + vt);
    }
  };
  constexpr int DMA_PER_CHUNK = MODE == 0 ? 4 : 2;  // per wave that moves any

  const int f_x = col & 15;
  auto tile_frag = [&](const uint8_t* t, int s) {  // token row col, dims 16 s + 8 half + 0 .. 7
    return *reinterpret_cast<const u32x4*>(t + col * SE_ROW + (((2 * s + half) ^ f_x) << 4));
  };
  // |v_t|^2 (the diagonal of V V^T) and -2 v_t . vc (V against the three pieces of vc in
  // columns 0 .. 2) of a chunk: exact products, fp32 sums
  // A chunk's slack from its |v|^2 (those of the next cluster's rows may be among them: it is then
  // shorter than it has to be): half of ln(2^123 / (len max |v|^2)), less than SE_SLACK only where
  // len |v|^2 passes 2^123 / e^60.  An overflowing product leaves none.
  auto chunk_slack = [&](int len, float vn) {
    const float sum = static_cast<float>(len) * vn;
    if (__ballot(sum > 6.0e10f) == 0ull) return SE_SLACK;
    return fminf(fmaxf(0.5f / SE_LOG2E * (123.0f - __builtin_amdgcn_logf(wave_max(sum))), 0.0f), SE_SLACK);
  };
  auto quad_sum3 = [&](float x) {  // columns 0 .. 3 (the last is zero) lie in one quad
    x += dpp_mov<0xB1>(x);
    return x + dpp_mov<0x4E>(x);
  };
  auto vstats = [&](auto norms, auto dots, int j, int len, const uint8_t* vt, int buf) {
    constexpr bool NORMS = decltype(norms)::value, DOTS = decltype(dots)::value;
    f32x16 vv = f32x16{}, vc = f32x16{};
    const uint16_t* brow = vc_l[col < 3 ? 3 * j + col : 3 * SE_CPW] + 8 * half;
#pragma unroll
    for (int s = 0; s < SE_KSTEPS; ++s) {
      const u32x4 a = tile_frag(vt, s);
      if (NORMS) vv = __builtin_amdgcn_mfma_f32_32x32x16_bf16(spr::as_bf16x8(a), spr::as_bf16x8(a), vv, 0, 0, 0);
      if (DOTS) {
        const u32x4 b = *reinterpret_cast<const u32x4*>(brow + 16 * s);
        vc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(spr::as_bf16x8(a), spr::as_bf16x8(b), vc, 0, 0, 0);
      }
    }
    if (NORMS) {
      float diag = 0.0f;  // row col is element 4 (col / 8) + col % 4 of the half with bit 2 of col
#pragma unroll
      for (int e = 0; e < 16; ++e) diag = e == 4 * (col >> 3) + (col & 3) ? vv[e] : diag;
      const bool mine = half == ((col >> 2) & 1);
      if (mine) vn_l[buf][col] = diag;
      const float slack = chunk_slack(len, mine ? diag : 0.0f);
      if (lane < 2) slack_l[buf][lane] = slack;
    }
    if (DOTS) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f32x4 c;
#pragma unroll
        for (int r = 0; r < 4; ++r) c[r] = -2.0f * quad_sum3(vc[4 * i + r]);
        if (col == 0) *reinterpret_cast<f32x4*>(&cd_l[buf][8 * i + 4 * half]) = c;
      }
    }
  };
  // A quarter of that by 16 x 16 blocks: |v_t|^2, or -2 v_t . vc, of the chunk's lower or upper 16
  // tokens.
  auto vstats_quarter = [&](int part, bool dots, int j, int len, const uint8_t* vt, int buf) {
    const int c16 = lane & 15, g = lane >> 4, row = 16 * part + c16;
    const uint16_t* brow = vc_l[c16 < 3 ? 3 * j + c16 : 3 * SE_CPW] + 8 * g;
    f32x4 acc = f32x4{};
#pragma unroll
    for (int s = 0; s < SE_D / 32; ++s) {  // token row, dims 32 s + 8 g + 0 .. 7
      const u32x4 a = *reinterpret_cast<const u32x4*>(vt + row * SE_ROW + (((4 * s + g) ^ c16) << 4));
      const u32x4 b = dots ? *reinterpret_cast<const u32x4*>(brow + 32 * s) : a;
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(spr::as_bf16x8(a), spr::as_bf16x8(b), acc, 0, 0, 0);
    }
    // lane (column c16, g) holds rows 4 g + 0 .. 3
    if (dots) {
      f32x4 c;
#pragma unroll
      for (int r = 0; r < 4; ++r) c[r] = -2.0f * quad_sum3(acc[r]);
      if (c16 == 0) *reinterpret_cast<f32x4*>(&cd_l[buf][16 * part + 4 * g]) = c;
    } else {
      float diag = 0.0f;
#pragma unroll
      for (int r = 0; r < 4; ++r) diag = r == (c16 & 3) ? acc[r] : diag;
      const bool mine = g == c16 >> 2;
      if (mine) vn_l[buf][row] = diag;
      const float slack = chunk_slack(len, mine ? diag : 0.0f);
      if (lane == 0) slack_l[buf][part] = slack;
    }
  };

  Walk wc, wn, wd;  // the next chunk to fold, to take statistics of, to DMA
  enter(wc, 0);
  wn = wd = wc;
  int folded = 0, taken = 0, issued = 0;  // how many of each so far
  // Step p folds chunks STEP p .. + STEP - 1 and takes the statistics of the STEP after them; as
  // many more are in flight and another STEP go to the tiles of the step before.  Every wave takes
  // the same steps.
  auto issue = [&] {
#pragma unroll
    for (int i = 0; i < STEP; ++i) {
      if (inside(wd)) {
        dma(wd, issued % S::TILES * SE_TILE, issued % S::VTILES * SE_TILE);
        ++issued;
        advance(wd);
      }
    }
  };
  auto landed = [&](int upto) {  // chunks below `upto`, for every wave; STEP more may be in flight
    if (issued >= upto + STEP) spr::wait_vm<STEP * DMA_PER_CHUNK>();
    else if (STEP == 2 && issued == upto + 1) spr::wait_vm<DMA_PER_CHUNK>();
    else spr::wait_vm<0>();
    spr::lds_barrier();
  };
  auto first = [&] {
    issue();
    issue();
    landed(STEP);
    issue();
  };
  auto begin_step = [&] {
    landed(folded + 2 * STEP);
    issue();
  };
  auto stats = [&] {
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
#pragma unroll
    for (int i = 0; i < STEP; ++i) {
      if (inside(wn)) {
        const uint8_t* vt = v_tiles + taken % S::VTILES * SE_TILE;
        const int buf = taken % S::STATS;
        if constexpr (STEP == 2) {
          if (i == stat) vstats(yes, yes, wn.j, wn.len, vt, buf);
        } else if (quarters) {
          vstats_quarter(wave & 1, wave >= 2, wn.j, wn.len, vt, buf);
        } else if (wave == 2) {
          vstats(yes, no, wn.j, wn.len, vt, buf);
        } else if (wave == 3) {
          vstats(no, yes, wn.j, wn.len, vt, buf);
        }
        ++taken;
        advance(wn);
      }
    }
  };
  if (q_wave) {
    // B fragments: q~ dims 16 s + 8 half + 0..7 as bf16 hi and lo, in registers before the
    // first DMA (a later wait for them would drain it)
    u32x4 qhi[SE_KSTEPS], qlo[SE_KSTEPS];
#pragma unroll
    for (int s = 0; s < SE_KSTEPS; ++s) {
      const float4 a = qraw[2 * s], b = qraw[2 * s + 1];
      const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
      uint32_t h[4], l[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float t0 = tf32_rna(v[2 * i]), t1 = tf32_rna(v[2 * i + 1]);
        const float h0 = __uint_as_float(__float_as_uint(t0) & 0xffff0000u);
        const float h1 = __uint_as_float(__float_as_uint(t1) & 0xffff0000u);
        h[i] = (__float_as_uint(h0) >> 16) | (__float_as_uint(h1) & 0xffff0000u);
        // t - h has at most 3 significant bits: exact in fp32 and in bf16
        l[i] = (__float_as_uint(t0 - h0) >> 16) | (__float_as_uint(t1 - h1) & 0xffff0000u);
      }
      qhi[s] = u32x4{h[0], h[1], h[2], h[3]};
      qlo[s] = u32x4{l[0], l[1], l[2], l[3]};
      asm volatile("" : "+v"(qhi[s].x), "+v"(qhi[s].y), "+v"(qhi[s].z), "+v"(qhi[s].w));
      asm volatile("" : "+v"(qlo[s].x), "+v"(qlo[s].y), "+v"(qlo[s].z), "+v"(qlo[s].w));
    }
    auto smma = [&](f32x16& acc, const uint8_t* kt) {
      acc = f32x16{};
#pragma unroll
      for (int s = 0; s < SE_KSTEPS; ++s) {
        const u32x4 a = tile_frag(kt, s);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(spr::as_bf16x8(a), spr::as_bf16x8(qhi[s]), acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(spr::as_bf16x8(a), spr::as_bf16x8(qlo[s]), acc, 0, 0, 0);
      }
    };
    float ref = 0.0f, lc = 0.0f, top = 0.0f, esum = 0.0f, cw = 1.0f;
    // S^T of a chunk (16 MFMAs), folded into the state:
    // E = sum_t max(c_w^2 |vc|^2 + r (r |v|^2 - 2 c_w v.vc), 0) with r = e^(l_t - ref),
    // c_w = e^(l_c - ref).  ref starts at l_c (c_w = 1: no product per element) and moves only
    // when a logit passes it by the chunk's slack; the result does not depend on it but for rounding.
    auto fold = [&](auto masked, const uint8_t* kt, int buf, int cn, int jc) {
      constexpr bool MASKED = decltype(masked)::value;
      f32x16 cur;
      smma(cur, kt);
      // element e is token 8 (e / 4) + 4 half + e % 4 of the chunk; a token past the run (the next
      // cluster's, or zeros) gets the logit -inf, and its error term is cleared
      const int lim = cn - 4 * half;
      if (MASKED) {
#pragma unroll
        for (int e = 0; e < 16; ++e) cur[e] = 8 * (e / 4) + (e % 4) < lim ? cur[e] : -__builtin_huge_valf();
      }
      float cmax = -__builtin_huge_valf();
#pragma unroll
      for (int e = 0; e < 16; ++e) cmax = fmaxf(cmax, cur[e]);
      // max over the raw dot products, scaled once: fl(a s) is monotone in a for s > 0
      cmax = max_xor32(cmax) * scale;
      top = fmaxf(top, cmax);
      const bool up = cmax > ref + (MODE == 0 ? fminf(slack_l[buf][0], slack_l[buf][1]) : SE_SLACK);
      if (__ballot(up) != 0ull) {
        const float to = up ? cmax : ref;
        const float alpha = up ? exp_fast(ref - to) : 1.0f;
        esum *= MODE == 0 ? alpha * alpha : alpha;
        ref = to;
        cw = up ? exp_fast(lc - ref) : cw;
      }
      const float c1 = scale * SE_LOG2E;
      const float negm = -ref * SE_LOG2E;
      float add0 = 0.0f, add1 = 0.0f;
      auto terms = [&](auto scaled) {
        constexpr bool SCALED = decltype(scaled)::value;
        const float base = SCALED ? cw * cw * vc2_l[jc] : vc2_l[jc];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const f32x4 vn = *reinterpret_cast<const f32x4*>(&vn_l[buf][8 * i + 4 * half]);
          const f32x4 cd = *reinterpret_cast<const f32x4*>(&cd_l[buf][8 * i + 4 * half]);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float w = __builtin_amdgcn_exp2f(__builtin_fmaf(cur[4 * i + r], c1, negm));
            float err = fmaxf(__builtin_fmaf(w, __builtin_fmaf(w, vn[r], SCALED ? cw * cd[r] : cd[r]), base), 0.0f);
            if (MASKED) err = 8 * i + r < lim ? err : 0.0f;
            if (r % 2 == 0) add0 += err; else add1 += err;
          }
        }
      };
      if (MODE == 0) {
        if (__ballot(cw != 1.0f) == 0ull) terms(std::false_type{}); else terms(std::true_type{});
      } else {
#pragma unroll
        for (int e = 0; e < 16; e += 2) {
          add0 += __builtin_amdgcn_exp2f(__builtin_fmaf(cur[e], c1, negm));
          add1 += __builtin_amdgcn_exp2f(__builtin_fmaf(cur[e + 1], c1, negm));
        }
      }
      esum += add0 + add1;
    };
    if (inside(wc)) {
      first();
      if (MODE == 0 && quarters) stats();
    }
    while (inside(wc)) {
      begin_step();
      if (MODE == 0 && quarters) stats();
      for (int i = 0; i < STEP && inside(wc); ++i) {
        if (sets == 1 || i == set) {
          const int slot = set * rows + 32 * (wave % qwaves) + col;
          if (wc.c0 < sets * SE_CHUNK) {  // this wave's first chunk of the cluster
            lc = rf_l[wc.j][slot];
            ref = lc;
            top = lc;
            cw = 1.0f;
            esum = 0.0f;
          }
          const int cn = min(SE_CHUNK, wc.len - wc.c0);
          const uint8_t* kt = k_tiles + folded % S::TILES * SE_TILE;
          if (cn == SE_CHUNK) fold(std::false_type{}, kt, folded % S::STATS, cn, wc.j);
          else fold(std::true_type{}, kt, folded % S::STATS, cn, wc.j);
          if (wc.c0 + sets * SE_CHUNK >= wc.len) {  // its last
            const float total = sum_xor32(esum);
            if (half == 0) {
              es_l[wc.j][slot] = total;
              rf_l[wc.j][slot] = ref;
              tp_l[wc.j][slot] = top;
            }
          }
        }
        ++folded;
        advance(wc);
      }
    }
  } else {
    if (inside(wc)) {
      first();
      if constexpr (MODE == 0) stats();
    }
    while (inside(wc)) {
      begin_step();
      if constexpr (MODE == 0) stats();
      for (int i = 0; i < STEP && inside(wc); ++i) {
        ++folded;
        advance(wc);
      }
    }
  }
  __syncthreads();
  // scores out, SE_CPW consecutive clusters of a query row at a time; empty clusters -inf
  for (int i = tid; i < SE_CPW * rows; i += nthr) {
    const int j = i % SE_CPW, r = i / SE_CPW;
    if (j >= ncl || q0 + r >= qn) continue;
    float total = es_l[j][r], ref = rf_l[j][r], top = tp_l[j][r];
    if (sets == 2) {
      const float r1 = rf_l[j][rows + r], to = fmaxf(ref, r1);
      const float a0 = ref == to ? 1.0f : exp_fast(ref - to), a1 = r1 == to ? 1.0f : exp_fast(r1 - to);
      total = MODE == 0 ? total * (a0 * a0) + es_l[j][rows + r] * (a1 * a1) : total * a0 + es_l[j][rows + r] * a1;
      ref = to;
      top = fmaxf(top, tp_l[j][rows + r]);
    }
    float score = -__builtin_huge_valf();
    if ((filled >> j) & 1u) {
      // value error: log(max(E / n, 1e-30)) of the weights taken from the largest logit
      score = MODE == 0 ? fmaxf(log_plus(total / static_cast<float>(len_l[j]), 2.0 * ref),
                                -69.07755278982137f + 2.0f * top)
                        : log_plus(fmaxf(total, 1.0e-30f), ref);
    }
    scores[(qh * qn + q0 + r) * kn + c_begin + j] = score;
  }
}

// ---------------------------------------------------------------- compensation
// svg_ear_compensation_triton (svg_ear.py:289-369 kernel, :603-678 wrapper): the sparse
// output (numerator, denominator 1, running max = its LSE) extended by the centroid
// approximation of the key clusters the map did not select.  One workgroup per (64 query
// rows, head); thread t owns row t / 4 and dims 32 (t % 4) .. + 31.  Key clusters go in
// blocks of BK (the reference's BLOCK_K), their TF32-rounded K and V centroids staged in
// LDS: the logit of a cluster is the quad's partial TF32 dot products summed over the four
// lanes (DPP) / sqrt(D) + log(max(count, 1)); per block the running max moves and the state
// is rescaled, the weights (TF32-rounded, as the reference's tl.dot sees them) times the V
// centroids are summed apart and then added (N3: all valid clusters added, the selected
// ones subtracted, as the reference orders it).  fp32 throughout.
__device__ __forceinline__ float quad_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, false));  // [1,0,3,2]
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, false));  // [2,3,0,1]
  return v;
}
constexpr int SC_BQ = 64;
constexpr int SC_PART = SE_D / 4;
__device__ __forceinline__ float ldf(const uint16_t* p) { return spr::bf16_to_f32(*p); }  // bf16
__device__ __forceinline__ float ldf(const float* p) { return *p; }
template <typename T>
struct TypeTag {
  using type = T;
};
template <int BK, bool N3, typename TQ, typename TS>
__global__ __launch_bounds__(256) void svg_ear_compensation_kernel(
    const TQ* __restrict__ q, const TS* __restrict__ sparse, const float* __restrict__ lse,
    const int32_t* __restrict__ qlabels, const uint8_t* __restrict__ dmap, int32_t qc1,
    const float* __restrict__ kc, const float* __restrict__ counts, const float* __restrict__ vc, int64_t tokens,
    int32_t kn, float scale, float* __restrict__ out) {
  constexpr int D = SE_D;
  __shared__ __attribute__((aligned(16))) float kcs[BK][D];
  __shared__ __attribute__((aligned(16))) float vcs[BK][D];
  __shared__ float lcnt[BK];
  __shared__ int32_t cvalid[BK];
  const int t = threadIdx.x, qi = t >> 2, d0 = SC_PART * (t & 3);
  const int64_t h = blockIdx.y;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * SC_BQ + qi;
  const bool live = row < tokens;
  const int64_t r = live ? row : tokens - 1;  // rows past the end read the last row, store nothing
  float qv[SC_PART], acc[SC_PART];
#pragma unroll
  for (int j = 0; j < SC_PART; ++j) {
    qv[j] = tf32_rna(ldf(q + (h * tokens + r) * D + d0 + j));
    acc[j] = ldf(sparse + (h * tokens + r) * D + d0 + j);
  }
  float denom = 1.0f;
  float row_max = lse[h * tokens + r];
  const int32_t drow = min(max(qlabels[h * tokens + r] + 1, 0), qc1 - 1);
  const uint8_t* dm = dmap + (h * qc1 + drow) * static_cast<int64_t>(kn + 1) + 1;
  for (int k0 = 0; k0 < kn; k0 += BK) {
    __syncthreads();  // the previous block's centroids are read
    for (int e = t; e < BK * D; e += 256) {
      const int k = e / D, dd = e - k * D, kk = k0 + k;
      kcs[k][dd] = kk < kn ? tf32_rna(kc[(h * kn + kk) * D + dd]) : 0.0f;
      vcs[k][dd] = kk < kn ? tf32_rna(vc[(h * kn + kk) * D + dd]) : 0.0f;
    }
    if (t < BK) {
      const int kk = k0 + t;
      const float c = kk < kn ? counts[h * kn + kk] : 0.0f;
      lcnt[t] = logf(fmaxf(c, 1.0f));
      cvalid[t] = (kk < kn && c > 0.0f) ? 1 : 0;
    }
    __syncthreads();
    float lg[BK];
    uint32_t take = 0, selm = 0;  // bit k: cluster k0 + k added / (N3) selected and added
    float bmax = -__builtin_huge_valf();
#pragma unroll
    for (int k = 0; k < BK; ++k) {
      float pdot = 0.0f;
#pragma unroll
      for (int j = 0; j < SC_PART; j += 4) {
        const spr::f32x4 kv = *reinterpret_cast<const spr::f32x4*>(&kcs[k][d0 + j]);
#pragma unroll
        for (int u = 0; u < 4; ++u) pdot = __builtin_fmaf(qv[j + u], kv[u], pdot);
      }
      lg[k] = quad_sum(pdot) * scale + lcnt[k];
      const bool act = live && cvalid[k] != 0;
      const bool sel = k0 + k < kn ? dm[k0 + k] != 0 : true;
      const bool tk = N3 ? act : (act && !sel);
      take |= static_cast<uint32_t>(tk) << k;
      selm |= static_cast<uint32_t>(N3 && act && sel) << k;
      if (tk) bmax = fmaxf(bmax, lg[k]);
    }
    const float new_max = fmaxf(row_max, bmax);
    const float old = exp_fast(row_max - new_max);  // NaN when both are -inf, as the reference's
    float wsum = 0.0f, ssum = 0.0f;
    float dota[SC_PART], dots[SC_PART];
#pragma unroll
    for (int j = 0; j < SC_PART; ++j) dota[j] = dots[j] = 0.0f;
#pragma unroll
    for (int k = 0; k < BK; ++k) {
      const float w = (take >> k) & 1u ? exp_fast(lg[k] - new_max) : 0.0f;
      const float ws = (selm >> k) & 1u ? w : 0.0f;
      wsum += w;
      ssum += ws;
      const float wt = tf32_rna(w), wst = tf32_rna(ws);
#pragma unroll
      for (int j = 0; j < SC_PART; j += 4) {
        const spr::f32x4 vv = *reinterpret_cast<const spr::f32x4*>(&vcs[k][d0 + j]);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          dota[j + u] = __builtin_fmaf(wt, vv[u], dota[j + u]);
          if constexpr (N3) dots[j + u] = __builtin_fmaf(wst, vv[u], dots[j + u]);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < SC_PART; ++j) {
      acc[j] = acc[j] * old + dota[j];
      if constexpr (N3) acc[j] -= dots[j];
    }
    denom = N3 ? (denom * old + wsum) - ssum : denom * old + wsum;
    row_max = new_max;
  }
  if (live) {
    const float inv_den = 1.0f / fmaxf(denom, 1e-30f);
    float* orow = out + (h * tokens + row) * D + d0;
#pragma unroll
    for (int j = 0; j < SC_PART; j += 4) {
      *reinterpret_cast<spr::f32x4*>(orow + j) =
          spr::f32x4{acc[j] * inv_den, acc[j + 1] * inv_den, acc[j + 2] * inv_den, acc[j + 3] * inv_den};
    }
  }
}

}  // namespace

// q [bh, tokens, 128] (q_dtype 0 bf16 / 2 fp32), sparse [bh, tokens, 128] (sparse_dtype 0 / 2),
// lse fp32 [bh, tokens], qlabels int32 [bh, tokens], dmap uint8 [bh, qc1, kn + 1] (row
// qlabel + 1, column cluster + 1), kcentroids / vcentroids fp32 [bh, kn, 128], kcounts fp32
// [bh, kn] -> out fp32 [bh, tokens, 128].  reformulation 0 "skipped", 1 "n3_residual";
// block_k 16 or 32.
extern "C" int spr_svg_ear_compensation(const void* q, int32_t q_dtype, const void* sparse, int32_t sparse_dtype,
                                        const float* lse, const int32_t* qlabels, const uint8_t* dmap, int32_t qc1,
                                        const float* kcentroids, const float* kcounts, const float* vcentroids,
                                        int64_t bh, int64_t tokens, int32_t d, int32_t kn, int32_t reformulation,
                                        int32_t block_k, float* out, hipStream_t stream) {
  SPR_REQUIRE(bh >= 0 && tokens >= 0 && kn >= 0 && qc1 >= 1, "spr_svg_ear_compensation: bad size");
  SPR_REQUIRE(d == SE_D, "spr_svg_ear_compensation: requires DIM=128, got %d", d);
  SPR_REQUIRE(reformulation == 0 || reformulation == 1, "spr_svg_ear_compensation: reformulation must be 0 or 1");
  SPR_REQUIRE(block_k == 16 || block_k == 32, "spr_svg_ear_compensation: block_k must be 16 or 32 (got %d)", block_k);
  SPR_REQUIRE((q_dtype == 0 || q_dtype == 2) && (sparse_dtype == 0 || sparse_dtype == 2),
              "spr_svg_ear_compensation: q and sparse must be bf16 (0) or fp32 (2)");
  SPR_REQUIRE(bh <= 65535, "spr_svg_ear_compensation: too many heads");
  if (bh == 0 || tokens == 0) return SPR_OK;
  SPR_REQUIRE(q && sparse && lse && qlabels && dmap && out && (kn == 0 || (kcentroids && kcounts && vcentroids)),
              "spr_svg_ear_compensation: null pointer");
  const dim3 grid(static_cast<uint32_t>(spr::ceil_div(tokens, SC_BQ)), static_cast<uint32_t>(bh));
  const float scale = 1.0f / sqrtf(static_cast<float>(d));
  auto go = [&](auto bk, auto n3, auto tq, auto ts) {
    using TQ = typename decltype(tq)::type;
    using TS = typename decltype(ts)::type;
    svg_ear_compensation_kernel<decltype(bk)::value, decltype(n3)::value, TQ, TS><<<grid, 256, 0, stream>>>(
        static_cast<const TQ*>(q), static_cast<const TS*>(sparse), lse, qlabels, dmap, qc1, kcentroids, kcounts,
        vcentroids, tokens, kn, scale, out);
  };
  auto by_types = [&](auto bk, auto n3) {
    using BF = TypeTag<uint16_t>;
    using F32 = TypeTag<float>;
    if (q_dtype == 0) {
      if (sparse_dtype == 0) go(bk, n3, BF{}, BF{}); else go(bk, n3, BF{}, F32{});
    } else {
      if (sparse_dtype == 0) go(bk, n3, F32{}, BF{}); else go(bk, n3, F32{}, F32{});
    }
  };
  auto by_mode = [&](auto bk) {
    if (reformulation == 1) by_types(bk, std::true_type{}); else by_types(bk, std::false_type{});
  };
  if (block_k == 16) by_mode(std::integral_constant<int, 16>{}); else by_mode(std::integral_constant<int, 32>{});
  SPR_LAUNCHED("svg_ear_compensation_kernel");
  return SPR_OK;
}

extern "C" size_t spr_svg_ear_scores_flops(int64_t q_heads, int32_t qn, int64_t tokens) {
  return static_cast<size_t>(2) * q_heads * qn * tokens * SE_D;
}

extern "C" int spr_svg_ear_scores(const float* q_centroids, const uint16_t* k_sorted, const uint16_t* v_sorted,
                                  const float* k_centroids, const float* v_centroids, const float* var_k_diag,
                                  float jensen_var_cap, const int32_t* k_sizes, int64_t q_heads, int32_t qn,
                                  int32_t kn, int64_t kv_heads, int64_t t_stored, int32_t d, int32_t group,
                                  int32_t mode, float* scores, hipStream_t stream) {
  SPR_REQUIRE(mode == 0 || mode == 1, "spr_svg_ear_scores: mode must be 0 (value error) or 1 (attention mass)");
  SPR_REQUIRE(d == SE_D, "spr_svg_ear_scores: head dim must be 128 (got %d)", d);
  SPR_REQUIRE(qn >= 1 && kn >= 1 && kv_heads >= 1 && group >= 1 && t_stored >= 1,
              "spr_svg_ear_scores: bad size");
  SPR_REQUIRE(q_heads == kv_heads * group, "spr_svg_ear_scores: q_heads %lld != kv_heads %lld * group %d",
              static_cast<long long>(q_heads), static_cast<long long>(kv_heads), group);
  SPR_REQUIRE(q_heads <= 65535 && kn <= (1 << 30) && qn <= (1 << 22), "spr_svg_ear_scores: grid too large");
  SPR_REQUIRE(t_stored < (int64_t(1) << 31) / (2 * SE_D) - SE_CHUNK,
              "spr_svg_ear_scores: at most %lld stored tokens per head",
              static_cast<long long>((int64_t(1) << 31) / (2 * SE_D) - SE_CHUNK - 1));
  SPR_REQUIRE(q_centroids && k_sorted && k_sizes && scores, "spr_svg_ear_scores: null pointer");
  if (mode == 0) {
    SPR_REQUIRE(v_sorted && k_centroids && v_centroids, "spr_svg_ear_scores: value error needs V and centroids");
    SPR_REQUIRE(!(jensen_var_cap > 0.0f) || var_k_diag != nullptr,
                "spr_svg_ear_scores: Jensen-aware routing requires var_k_diag");
  }
  // Query blocks of 32 rows, one wave each, in groups of equal size; four waves of all move the
  // tiles.  Up to four blocks leave most of a CU idle: its workgroups then take half the LDS, so
  // that two share it, where there are 1.5 or more for each CU and the clusters are short enough
  // (in long ones the second chunk per barrier and the two sets of query waves are worth more).
  // Up to two blocks, 24 heads x 40,000 tokens, 64 rows: 1,000 clusters 284 -> 216 us, 134 clusters
  // 184 -> 180; 118,800 tokens, 134 clusters (not short) 440 -> 461; 8 heads x 40,000 tokens (304
  // workgroups), 64 rows: 92 -> 98 us.  Three and four blocks of value error leave the statistics no
  // wave of their own, so only short clusters gain, and longer ones where three or more workgroups
  // per CU fill the turns.  Speed against whole workgroups, 97 to 128 rows: clusters of 24 tokens
  // 1.03 to 1.23, of 40 0.98 to 1.11 (from 768 workgroups on 1.12 to 1.18), of 90 0.94 to 0.97 (0.99
  // to 1.08), of 221 at 475 workgroups 0.82; 65 to 96 rows: of 24 0.98 to 1.13, of 40 0.91 to 0.94
  // (1.05), of 90 0.83 to 0.88 (0.93 to 1.02).
  const int32_t qblocks = (qn + 31) / 32;
  const int64_t groups = spr::ceil_div(kn, SE_CPW) * q_heads;
  const int64_t cluster_tokens =  // mean of the longest that are short
      mode != 0 || qblocks <= 2 ? 512 : (qblocks == 3 ? 24 : 48) * (groups >= 768 ? 2 : 1);
  const bool few = qblocks <= Step<1>::QWAVES && groups >= 384 && t_stored <= cluster_tokens * kn;
  const int32_t most = few ? Step<1>::QWAVES : Step<2>::QWAVES;
  const int32_t qgroups = (qblocks + most - 1) / most;
  const int32_t qwaves = (qblocks + qgroups - 1) / qgroups;
  const int32_t sets = !few && 2 * qwaves <= most ? 2 : 1;
  const int64_t turns = static_cast<int64_t>((kn + 8 * SE_CPW - 1) / (8 * SE_CPW)) * qgroups;
  SPR_REQUIRE(turns * 8 < (int64_t(1) << 31), "spr_svg_ear_scores: grid too large");
  const dim3 grid(static_cast<uint32_t>(turns * 8), static_cast<uint32_t>(q_heads));
  const int32_t waves = qwaves * sets + (mode == 0 && !few ? SE_SWAVES : 0);
  const uint32_t threads = 64 * (waves < 4 ? 4 : waves);
  if (mode == 0) {
    const bool jensen = jensen_var_cap > 0.0f;
    svg_ear_centroid_logit_kernel<<<dim3(static_cast<uint32_t>((kn + CL_CLUSTERS - 1) / CL_CLUSTERS),
                                         static_cast<uint32_t>((qn + CL_ROWS - 1) / CL_ROWS),
                                         static_cast<uint32_t>(q_heads)),
                                    SE_THREADS, 0, stream>>>(q_centroids, k_centroids, jensen ? var_k_diag : nullptr,
                                                             jensen ? jensen_var_cap : 0.0f, qn, kn, group, scores);
    SPR_LAUNCHED("svg_ear_centroid_logit_kernel");
    auto score = [&](auto step) {
      svg_ear_score_kernel<0, decltype(step)::value><<<grid, threads, 0, stream>>>(
          q_centroids, k_sorted, v_sorted, v_centroids, k_sizes, qn, kn, t_stored, group, qgroups, qwaves, sets, scores);
    };
    if (few) score(std::integral_constant<int, 1>{}); else score(std::integral_constant<int, 2>{});
    SPR_LAUNCHED("svg_ear_score_kernel<value>");
  } else {
    auto score = [&](auto step) {
      svg_ear_score_kernel<1, decltype(step)::value><<<grid, threads, 0, stream>>>(
          q_centroids, k_sorted, nullptr, nullptr, k_sizes, qn, kn, t_stored, group, qgroups, qwaves, sets, scores);
    };
    if (few) score(std::integral_constant<int, 1>{}); else score(std::integral_constant<int, 2>{});
    SPR_LAUNCHED("svg_ear_score_kernel<mass>");
  }
  return SPR_OK;
}
