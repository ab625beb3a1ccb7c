// Role-coordinate projection with row RMS normalisation (N8's Q role features), and the
// K (or V) role projection with one RMS scale per head.
//
// Replaces:
//   _role_projection_rms_kernel + role_projection_rms_triton
//       (src/sparsepr/kernels/triton/role_projection.py:16-55, :58-103)
//   _role_k_projection_normalize_fp32 / _role_kv_projection_normalize_fp32, torch.compile'd
//       under role_kv_matmul_precision (src/sparsepr/models/common/n8_v6.py:77-149), and
//       normalize_feature_scale(project_tokens(...)) (operator_kmeans.py:540-550)
//
//   p = x . F~, out = p / sqrt(max(sum_r p_r^2 / R, 1e-12))
// for x bf16 [bh, n, d] and the factor F fp32 [bh, d, R]; F~ is F as the fp32 matmul sees it:
//   PREC 0 ("high", and tl.dot(..., input_precision="tf32")): rounded to TF32 (nearest, ties
//          away; a bf16 x is exact in TF32), split into bf16 hi + lo with hi + lo == F~;
//   PREC 1 ("highest", plain fp32): F itself, split into bf16 hi + mid + lo (8 significant
//          bits each, 24 in all) with hi + mid + lo == F;
//   PREC 2 ("medium", bf16 operands): F rounded to bf16 (nearest even).
// Each product of a bf16 x with a bf16 piece is exact, so only the fp32 summation order
// differs from the reference's.
//
// Layout of role_projection_kernel (role_projection_rows_kernel's stands beside it): workgroups
// of four waves per head, as many as stay resident, each walking token blocks of its head
// (rp_tokens); F~^T hi / lo of the head sit in LDS (R rows padded to a multiple of 32, d
// columns, 16-byte pieces swizzled by row).  A wave computes P^T = F~^T X^T for 32 tokens per
// step: A = F~^T fragments from LDS, B = X^T fragments straight from HBM (lane = token, 16
// contiguous bytes per 16-dim step, the next block's prefetched), so each lane ends up with
// R / 2 values of one token and the row's sum of squares needs one exchange between the two
// half-waves.
#include <algorithm>
#include <type_traits>

#include "spr_common.h"

namespace {

using spr::f32x16;
using spr::u32x4;

constexpr int RP_THREADS = 256;
constexpr int RP_WAVES = RP_THREADS / 64;
// Tokens per block (a workgroup takes several blocks of its head): 256 for the row-normalised
// projection (MODE 0) and the K projection's scaling pass (MODE 2), 1024 for its sum pass
// (MODE 1: one fp64 partial per block, which MODE 2 sums in block order).  Measured in the N8
// step against 512 for all: Q projection 0.39 -> 0.36 ms, K projection 0.64 -> 0.61 ms.
constexpr int rp_tokens(int mode) { return mode == 1 ? 1024 : 256; }
constexpr int RP_MAX_R = 128;

__device__ __forceinline__ float tf32_rna(float x) {
  return __uint_as_float((__float_as_uint(x) + 0x1000u) & 0xffffe000u);
}

__device__ __forceinline__ float sum_xor32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// D = head dim (D / 8 sixteen-byte pieces per F~^T row); RB = rank padded to 32, in 32-row blocks.
// MODE 0: rows normalised by their RMS.  MODE 1: no output; the workgroup's sum of p^2 goes to
// partial[head][block] (fp64).  MODE 2: p divided by the head's scale sqrt(max(mean p^2, ...))
// formed from the partials in block order (the same on every workgroup); block 0 stores it.
// MODE 2 writes (weight p) / scale into columns out_col .. out_col + R of rows out_ld floats long.
// NP = bf16 pieces of F~ (PREC 0: 2, 1: 3, 2: 1).
template <int D, int RB, int MODE, int PREC>
__global__ __launch_bounds__(RP_THREADS) void role_projection_kernel(const uint16_t* __restrict__ x,
                                                                     const float* __restrict__ factor, int64_t n,
                                                                     int32_t rank, float* __restrict__ out,
                                                                     int32_t out_ld, int32_t out_col, float weight,
                                                                     double* __restrict__ partial,
                                                                     float* __restrict__ head_scale) {
  constexpr int64_t RP_TOKENS = rp_tokens(MODE);
  constexpr int KSTEPS = D / 16;
  constexpr int ROWB = D * 2;  // bytes per F~^T row (bf16)
  constexpr int RP = RB * 32;
  constexpr int NP = PREC == 0 ? 2 : (PREC == 1 ? 3 : 1);
  __shared__ __attribute__((aligned(16))) uint8_t fpc[NP][RP * ROWB];
  const int64_t b = blockIdx.y;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int col = lane & 31;
  const int half = lane >> 5;

  // F~^T pieces into LDS: element (r, k) of row r at piece (k / 8) ^ (r % (D / 8)), slot k % 8.
  // Each piece is the top 16 bits (a bf16) of what the earlier pieces leave, so the pieces
  // sum to F~ exactly (the remainders are exact in fp32).
  const float* fb = factor + b * D * rank;
  for (int i = tid; i < RP * D / 2; i += RP_THREADS) {
    const int r = i / (D / 2), k = 2 * (i % (D / 2));
    float v[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const float f = r < rank ? fb[static_cast<int64_t>(k + u) * rank + r] : 0.0f;
      v[u] = PREC == 0 ? tf32_rna(f) : (PREC == 2 ? spr::bf16_to_f32(spr::f32_to_bf16(f)) : f);
    }
    const int off = r * ROWB + ((((k >> 3) ^ (r % (D / 8))) << 4) | ((k & 7) << 1));
#pragma unroll
    for (int pc = 0; pc < NP; ++pc) {
      const uint32_t h0 = __float_as_uint(v[0]) & 0xffff0000u, h1 = __float_as_uint(v[1]) & 0xffff0000u;
      *reinterpret_cast<uint32_t*>(fpc[pc] + off) = (h0 >> 16) | h1;
      v[0] -= __uint_as_float(h0);
      v[1] -= __uint_as_float(h1);
    }
  }
  __syncthreads();

  const uint16_t* xb = x + b * n * D;
  float* ob = out + b * n * (MODE == 2 ? out_ld : rank);
  __shared__ double red_l[RP_WAVES];
  float div = 1.0f;
  if (MODE == 2) {
    // the head's scale: fp64 sum of the partials in block order, then as the reference
    // rounds it: fp32 mean, sqrt, clamp at 1e-8
    const int64_t nparts = (n + rp_tokens(1) - 1) / rp_tokens(1);  // the first pass's blocks
    double tot = 0.0;
    for (int64_t i = 0; i < nparts; ++i) tot += partial[b * nparts + i];
    div = fmaxf(sqrtf(static_cast<float>(tot / (static_cast<double>(n) * rank))), 1.0e-8f);
    if (blockIdx.x == 0 && tid == 0) head_scale[b] = div;
  }
  // Token blocks of RP_TOKENS: this workgroup takes blocks blockIdx.x, + gridDim.x, ... of its
  // head (the grid holds as many workgroups per head as stay resident at once, so no second
  // round of workgroups trails the first).  MODE 1 writes one partial per block.
  const int64_t nvb = (n + RP_TOKENS - 1) / RP_TOKENS;
  // X^T fragments of a 32-token block: lane = token, 16 bytes per 16-dim step (zero past the end)
  auto load_x = [&](u32x4 (&xf)[KSTEPS], int64_t t0, int64_t t_end) {
    const int64_t t = t0 + col;
    const bool live = t < t_end;
    const uint16_t* xr = xb + (live ? t : t0) * D + 8 * half;
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) {
      xf[s] = *reinterpret_cast<const u32x4*>(xr + 16 * s);
      if (!live) xf[s] = u32x4{0, 0, 0, 0};
    }
  };
  // this wave's next 32-token block after (vb, t0): the next one of the block, else the
  // first of the workgroup's next block; vb = nvb when there is none
  auto skip_empty = [&](int64_t& vb, int64_t& t0) {  // a short last block may hold none of this wave's rows
    while (vb < nvb && t0 >= min((vb + 1) * RP_TOKENS, n)) {
      vb += gridDim.x;
      t0 = vb * RP_TOKENS + 32 * wave;
    }
  };
  auto advance = [&](int64_t& vb, int64_t& t0) {
    t0 += 32 * RP_WAVES;
    skip_empty(vb, t0);
  };
  int64_t vb = blockIdx.x, t0 = vb * RP_TOKENS + 32 * wave;
  skip_empty(vb, t0);
  u32x4 xn[KSTEPS];
  if (vb < nvb) load_x(xn, t0, min((vb + 1) * RP_TOKENS, n));
  double wsum = 0.0;  // MODE 1: this lane's sum of p^2 over the current block
  for (int64_t cur = blockIdx.x; cur < nvb; cur += gridDim.x) {
    const int64_t t_end = min((cur + 1) * RP_TOKENS, n);
    while (vb == cur) {
      const int64_t t = t0 + col;
      const bool live = t < t_end;
      u32x4 xf[KSTEPS];
#pragma unroll
      for (int s = 0; s < KSTEPS; ++s) xf[s] = xn[s];
      const int64_t t_row = t0;
      // the next block's loads are in flight during this block's MFMAs and stores
      advance(vb, t0);
      if (vb < nvb) load_x(xn, t0, min((vb + 1) * RP_TOKENS, n));
      f32x16 acc[RB];
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        acc[rb] = f32x16{};
        const int r = 32 * rb + col;
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s) {
          const int off = r * ROWB + (((2 * s + half) ^ (r % (D / 8))) << 4);
#pragma unroll
          for (int pc = 0; pc < NP; ++pc) {
            const u32x4 a = *reinterpret_cast<const u32x4*>(fpc[pc] + off);
            acc[rb] =
                __builtin_amdgcn_mfma_f32_32x32x16_bf16(spr::as_bf16x8(a), spr::as_bf16x8(xf[s]), acc[rb], 0, 0, 0);
          }
        }
      }
      // lane (token col, half) holds p_r for r = 32 rb + 8 (e / 4) + 4 half + e % 4 (zero past rank)
      float ss = 0.0f;
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
#pragma unroll
        for (int e = 0; e < 16; ++e) ss = __builtin_fmaf(acc[rb][e], acc[rb][e], ss);
      }
      if (MODE == 1) {
        wsum += live ? static_cast<double>(ss) : 0.0;
        continue;
      }
      ss = sum_xor32(ss);
      const float inv = 1.0f / sqrtf(fmaxf(ss / static_cast<float>(rank), 1.0e-12f));
      auto nrm = [&](float v) { return MODE == 0 ? v * inv : (weight * v) / div; };
      if (live) {
        const int64_t tt = t_row + col;
        float* orow = MODE == 2 ? ob + tt * out_ld + out_col : ob + tt * rank;
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const int r0 = 32 * rb + 8 * g + 4 * half;
            if (r0 + 3 < rank && (rank & 3) == 0 && (MODE != 2 || ((out_ld | out_col) & 3) == 0)) {
              *reinterpret_cast<float4*>(orow + r0) = make_float4(nrm(acc[rb][4 * g]), nrm(acc[rb][4 * g + 1]),
                                                                  nrm(acc[rb][4 * g + 2]), nrm(acc[rb][4 * g + 3]));
            } else {
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                if (r0 + i < rank) orow[r0 + i] = nrm(acc[rb][4 * g + i]);
              }
            }
          }
        }
      }
    }
    if (MODE == 1) {
      // lanes in order, then waves in order: the same fp64 sum on every run
      for (int o = 1; o < 64; o <<= 1) wsum += __shfl_xor(wsum, o, 64);
      if (lane == 0) red_l[wave] = wsum;
      __syncthreads();
      if (tid == 0) {
        double tsum = 0.0;
        for (int w = 0; w < RP_WAVES; ++w) tsum += red_l[w];
        partial[b * nvb + cur] = tsum;
      }
      __syncthreads();
      wsum = 0.0;
    }
  }
}

// ---------------------------------------------------------------- ranks 16, 32, 48, 64
// The same projections for the ranks in use on long calls, bound by HBM: X rows are read 1 KB of
// consecutive bytes per instruction and turned into MFMA fragments through LDS, and the features
// leave it in row order, where the kernel above reads 16 bytes of 32 rows per load and writes 32
// bytes of 32 rows per store.  One workgroup of eight waves per CU takes a contiguous share of
// all (head, unit) pairs and stages the factor when its share enters a head; its waves take the
// units of a head in turn and walk them in 32-token tiles of their own, the next tile's rows in
// registers meanwhile, with no barrier.  Tiles: 16-byte piece j of row r at slot j ^ swz(r), so
// the fragment reads of 16 rows hit all 64 banks; output rows at a pitch of R + 4 floats,
// likewise.  Factor fragments are read four ahead of their MFMA: left to itself the compiler
// read each right before its use, some 130 cycles apart.
// 24 heads x 118,800 tokens, D = 128: rank 64 with row RMS 330 -> 304 us, rank 48 with the head's
// RMS 205 + 320 -> 186 + 262 us (the first 4.4 -> 4.8 TB/s); a call of both 793 -> 731 us.
// Twelve waves 808 us, four with a triple DMA buffer 766, eight with two tiles ahead 746, the
// factor in registers 963 (it spills).
constexpr int RS_WAVES = 8;
// tokens of a unit: one tile, or 256 in the sum pass, which leaves one fp64 partial for each
constexpr int rs_unit(int mode) { return mode == 1 ? 256 : 32; }
constexpr int RS_TILE = 32;

template <int D, int R>
struct RowStream {
  static constexpr int ROWB = 2 * D;
  static constexpr int PIECES = ROWB / 16;
  static constexpr int LOAD_ROWS = 64 / PIECES;              // rows per load instruction
  static constexpr int LOADS = RS_TILE / LOAD_ROWS;          // per tile
  static constexpr int PITCH = 4 * R + 16;               // bytes of an output row in LDS
  static constexpr int STORES = RS_TILE * R * 4 / 1024;      // 16 bytes a lane, per tile
  static constexpr int BUF_RAW = RS_TILE * (ROWB > PITCH ? ROWB : PITCH);
  static constexpr int BUF = (BUF_RAW + 255) / 256 * 256;
  static constexpr int RB = (R + 31) / 32;
  __device__ static __forceinline__ int swz(int r) { return D == 128 ? r & 15 : (r >> 1) & 7; }
};

// MODE and PREC as above.  MODE 1: partial[head][unit].
template <int D, int R, int MODE, int PREC>
__global__ __launch_bounds__(RS_WAVES * 64, RS_WAVES / 4) void role_projection_rows_kernel(
    const uint16_t* __restrict__ x, const float* __restrict__ factor, int64_t bh, int64_t n, float* __restrict__ out,
    int32_t out_ld, int32_t out_col, float weight, double* __restrict__ partial, float* __restrict__ head_scale) {
  using T = RowStream<D, R>;
  constexpr int KSTEPS = D / 16;
  constexpr int NP = PREC == 0 ? 2 : (PREC == 1 ? 3 : 1);
  __shared__ __attribute__((aligned(16))) uint8_t fpc[NP][T::RB * 32 * T::ROWB];
  __shared__ __attribute__((aligned(1024))) uint8_t tiles[RS_WAVES][T::BUF];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31;
  const int half = lane >> 5;
  constexpr int64_t RS_UNIT = rs_unit(MODE);
  const int64_t units = (n + RS_UNIT - 1) / RS_UNIT;  // of a head
  const int64_t all = bh * units;
  const int64_t u_begin = all * blockIdx.x / gridDim.x, u_end = all * (blockIdx.x + 1) / gridDim.x;
  uint8_t* const tile = tiles[wave];

  for (int64_t u_at = u_begin; u_at < u_end;) {
    const int64_t b = u_at / units;
    const int64_t first = u_at - b * units, last = min(u_end - b * units, units);  // this head's share
    u_at = b * units + last;
    // F~^T pieces (as in the kernel above), once every wave is done with the last head's
    __syncthreads();
    const float* fb = factor + b * D * R;
    for (int i = tid; i < T::RB * 32 * D / 2; i += RS_WAVES * 64) {
      const int r = i % (T::RB * 32), k = 2 * (i / (T::RB * 32));
      float v[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const float f = r < R ? fb[(k + u) * R + r] : 0.0f;
        v[u] = PREC == 0 ? tf32_rna(f) : (PREC == 2 ? spr::bf16_to_f32(spr::f32_to_bf16(f)) : f);
      }
      const int off = r * T::ROWB + (((k >> 3) ^ T::swz(r)) << 4 | ((k & 7) << 1));
#pragma unroll
      for (int pc = 0; pc < NP; ++pc) {
        const uint32_t h0 = __float_as_uint(v[0]) & 0xffff0000u, h1 = __float_as_uint(v[1]) & 0xffff0000u;
        *reinterpret_cast<uint32_t*>(fpc[pc] + off) = (h0 >> 16) | h1;
        v[0] -= __uint_as_float(h0);
        v[1] -= __uint_as_float(h1);
      }
    }
    float div = 1.0f;
    if (MODE == 2) {
      // the head's scale: fp64 sum of the first pass's partials, lanes in turn and then by halves (the
      // same order everywhere), then as the reference rounds it: fp32 mean, sqrt, clamp at 1e-8
      double tot = 0.0;
      const int64_t parts = (n + rs_unit(1) - 1) / rs_unit(1);
      for (int64_t i = lane; i < parts; i += 64) tot += partial[b * parts + i];
      for (int o = 32; o > 0; o >>= 1) tot += __shfl_xor(tot, o, 64);
      div = fmaxf(sqrtf(static_cast<float>(tot / (static_cast<double>(n) * R))), 1.0e-8f);
      if (first == 0 && tid == 0) head_scale[b] = div;
    }
    __syncthreads();

    const uint16_t* xb = x + b * n * D;
    float* const ob = MODE == 1 ? nullptr : out + b * n * out_ld + out_col;
    // this wave's tiles: units first + wave, + RS_WAVES, ..., each in tiles of 32 tokens below n
    auto valid = [&](int64_t u, int64_t t) { return u < last && t < min((u + 1) * RS_UNIT, n); };
    auto advance = [&](int64_t& u, int64_t& t) {
      t += RS_TILE;
      if (t >= min((u + 1) * RS_UNIT, n)) {
        u += RS_WAVES;
        t = u * RS_UNIT;
      }
    };
    int64_t uc = first + wave, tc = uc * RS_UNIT;  // the tile computed
    // a tile's rows, 1 KB of consecutive bytes per load; rows past n read the last one
    // (native vectors: an array of structs carried round the loop went through scratch memory)
    typedef uint32_t v4 __attribute__((ext_vector_type(4)));
    v4 xn[T::LOADS];
    auto load = [&](int64_t t) {
#pragma unroll
      for (int i = 0; i < T::LOADS; ++i) {
        const int64_t row = min(t + T::LOAD_ROWS * i + lane / T::PIECES, n - 1);
        xn[i] = *reinterpret_cast<const v4*>(xb + row * D + lane % T::PIECES * 8);
      }
    };
    if (valid(uc, tc)) load(tc);
    double wsum = 0.0;  // MODE 1: this lane's sum of p^2 over the unit
    while (valid(uc, tc)) {
#pragma unroll
      for (int i = 0; i < T::LOADS; ++i) {
        const int row = T::LOAD_ROWS * i + lane / T::PIECES;
        *reinterpret_cast<v4*>(tile + row * T::ROWB + ((lane % T::PIECES ^ T::swz(row)) << 4)) = xn[i];
      }
      const int64_t t = tc, u = uc;
      advance(uc, tc);
      if (valid(uc, tc)) load(tc);  // in flight until the next turn
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // every lane's rows, before the reads across lanes
      u32x4 xf[KSTEPS];
#pragma unroll
      for (int s = 0; s < KSTEPS; ++s)
        xf[s] = *reinterpret_cast<const u32x4*>(tile + col * T::ROWB + (((2 * s + half) ^ T::swz(col)) << 4));
      // factor fragments read four ahead of their MFMA
      constexpr int FR = T::RB * KSTEPS * NP;
      auto frag = [&](int f) {
        const int rb = f / (KSTEPS * NP), st = f / NP % KSTEPS, r = 32 * rb + col;
        return *reinterpret_cast<const u32x4*>(fpc[f % NP] + r * T::ROWB + (((2 * st + half) ^ T::swz(r)) << 4));
      };
      f32x16 acc[T::RB];
      u32x4 fr[5];
#pragma unroll
      for (int f = 0; f < 4 && f < FR; ++f) fr[f] = frag(f);
#pragma unroll
      for (int f = 0; f < FR; ++f) {
        if (f + 4 < FR) fr[(f + 4) % 5] = frag(f + 4);
        const int rb = f / (KSTEPS * NP);
        if (f % (KSTEPS * NP) == 0) acc[rb] = f32x16{};
        acc[rb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(spr::as_bf16x8(fr[f % 5]),
                                                          spr::as_bf16x8(xf[f / NP % KSTEPS]), acc[rb], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      // lane (token col, half) holds p_r for r = 32 rb + 8 (e / 4) + 4 half + e % 4 (zero past R)
      float ss = 0.0f;
#pragma unroll
      for (int rb = 0; rb < T::RB; ++rb) {
#pragma unroll
        for (int e = 0; e < 16; ++e) ss = __builtin_fmaf(acc[rb][e], acc[rb][e], ss);
      }
      if (MODE == 1) {
        wsum += t + col < n ? static_cast<double>(ss) : 0.0;
        if (uc != u) {  // lanes by halves: the same fp64 sum on every run
          for (int o = 1; o < 64; o <<= 1) wsum += __shfl_xor(wsum, o, 64);
          if (lane == 0) partial[b * units + u] = wsum;
          wsum = 0.0;
        }
      } else {
        ss = sum_xor32(ss);
        const float inv = 1.0f / sqrtf(fmaxf(ss / static_cast<float>(R), 1.0e-12f));
        auto nrm = [&](float v) { return MODE == 0 ? v * inv : (weight * v) / div; };
        // the fragments are in registers: the tile's buffer takes the output rows
#pragma unroll
        for (int rb = 0; rb < T::RB; ++rb) {
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            if (32 * rb + 8 * g >= R) continue;
            *reinterpret_cast<float4*>(tile + col * T::PITCH + 4 * (32 * rb + 8 * g + 4 * half)) =
                make_float4(nrm(acc[rb][4 * g]), nrm(acc[rb][4 * g + 1]), nrm(acc[rb][4 * g + 2]),
                            nrm(acc[rb][4 * g + 3]));
          }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // every lane's rows, before the reads across lanes
#pragma unroll
        for (int i = 0; i < T::STORES; ++i) {
          const int piece = 64 * i + lane, row = piece / (R / 4), c = piece % (R / 4);
          const float4 v = *reinterpret_cast<const float4*>(tile + row * T::PITCH + 16 * c);
          if (t + row < n) *reinterpret_cast<float4*>(ob + (t + row) * out_ld + 4 * c) = v;
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the tile is read before the next one is written
    }
  }
}

}  // namespace

// Compute units of the calling thread's current device (queried once per device).
static int rp_cu_count() {
  static int cached[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cached[dev] == 0) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
    cached[dev] = cus;
  }
  return cached[dev];
}

// Workgroups per head: as many as stay resident together (per_cu per CU, from the
// occupancy calculator), shared evenly by the heads, at most one per token block.
static uint32_t rp_groups_per_head(int64_t bh, int64_t n, int per_cu, int tokens) {
  const int64_t resident = static_cast<int64_t>(std::max(per_cu, 1)) * rp_cu_count();
  const int64_t nvb = (n + tokens - 1) / tokens;
  return static_cast<uint32_t>(std::max<int64_t>(1, std::min<int64_t>(nvb, resident / std::max<int64_t>(bh, 1))));
}

// Resident workgroups per CU of role_projection_kernel<D, RB, MODE, PREC> (queried once per
// instantiation; 1 if the query fails).
template <int D, int RB, int MODE, int PREC>
static int rp_occupancy() {
  static int cached = 0;
  if (cached == 0) {
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, role_projection_kernel<D, RB, MODE, PREC>, RP_THREADS, 0) !=
            hipSuccess ||
        nb <= 0)
      nb = 1;
    cached = nb;
  }
  return cached;
}

// The streaming kernel's calls: the ranks it is built for, 16-byte rows on both sides, and work
// that fills it: four 32-token tiles per wave of the chip, in heads long enough (8,192 tokens)
// that a workgroup's factor staging, once per head that its share touches, is a small part.
// Measured with both kernels, rank 64 + 48, D = 128: 8 heads x 12,000 tokens (1.5 tiles a wave)
// 55 us above -> 60 here, 24 x 5,461 (2 a wave, 5,461-token heads) 61 -> 72, 24 x 10,923 (4) 92
// -> 88, 12 x 30,000 with ranks 32 + 16 and D = 64 (5.5) 56 -> 47, 24 x 118,800 (43) 793 -> 731;
// between two and four tiles it depends on how shares and heads meet (8 x 16,384 59 -> 55), so
// the line lies where every one gains.
static bool rp_streams(const void* x, const void* out, int64_t bh, int64_t n, int32_t rank, int32_t out_ld,
                       int32_t out_col) {
  return (rank == 16 || rank == 32 || rank == 48 || rank == 64) && out_ld % 4 == 0 && out_col % 4 == 0 &&
         reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0 && n >= 8192 &&
         bh * ((n + RS_TILE - 1) / RS_TILE) >= static_cast<int64_t>(4) * RS_WAVES * rp_cu_count();
}

template <int MODE, int PREC>
static void launch_role_projection_rows(int64_t bh, hipStream_t stream, const uint16_t* xp, const float* factor,
                                        int64_t n, int32_t d, int32_t rank, float* out, int32_t out_ld,
                                        int32_t out_col, float weight, double* partial, float* head_scale) {
  const int64_t all = bh * ((n + rs_unit(MODE) - 1) / rs_unit(MODE));
  const uint32_t groups =
      static_cast<uint32_t>(std::max<int64_t>(1, std::min<int64_t>(rp_cu_count(), (all + RS_WAVES - 1) / RS_WAVES)));
  auto run = [&](auto dd, auto rr) {
    role_projection_rows_kernel<decltype(dd)::value, decltype(rr)::value, MODE, PREC>
        <<<groups, RS_WAVES * 64, 0, stream>>>(xp, factor, bh, n, out, out_ld, out_col, weight, partial, head_scale);
  };
  auto by_rank = [&](auto dd) {
    if (rank == 16) run(dd, std::integral_constant<int, 16>{});
    else if (rank == 32) run(dd, std::integral_constant<int, 32>{});
    else if (rank == 48) run(dd, std::integral_constant<int, 48>{});
    else run(dd, std::integral_constant<int, 64>{});
  };
  if (d == 128) by_rank(std::integral_constant<int, 128>{});
  else by_rank(std::integral_constant<int, 64>{});
}

template <int MODE, int PREC>
static void launch_role_projection(int64_t bh, hipStream_t stream, const uint16_t* xp, const float* factor,
                                   int64_t n, int32_t d, int32_t rank, float* out, int32_t out_ld, int32_t out_col,
                                   float weight, double* partial, float* head_scale) {
  const int rb = (rank + 31) / 32;
#define SPR_RP(DD, RBB)                                                                                      \
  role_projection_kernel<DD, RBB, MODE, PREC>                                                                \
      <<<dim3(rp_groups_per_head(bh, n, (rp_occupancy<DD, RBB, MODE, PREC>()), rp_tokens(MODE)), \
              static_cast<uint32_t>(bh)),                                                                    \
         RP_THREADS, 0, stream>>>(xp, factor, n, rank, out, out_ld, out_col, weight, partial, head_scale)
  if (d == 128) {
    if (rb == 1) SPR_RP(128, 1); else if (rb == 2) SPR_RP(128, 2); else if (rb == 3) SPR_RP(128, 3); else SPR_RP(128, 4);
  } else {
    if (rb == 1) SPR_RP(64, 1); else if (rb == 2) SPR_RP(64, 2); else if (rb == 3) SPR_RP(64, 3); else SPR_RP(64, 4);
  }
#undef SPR_RP
}

extern "C" int spr_role_projection_rms(const void* x, const float* factor, int64_t bh, int64_t n, int32_t d,
                                       int32_t rank, float* out, hipStream_t stream) {
  SPR_REQUIRE(bh >= 0 && n >= 0, "spr_role_projection_rms: bad size");
  SPR_REQUIRE(d == 64 || d == 128, "spr_role_projection_rms: head dim must be 64 or 128 (got %d)", d);
  SPR_REQUIRE(rank >= 1 && rank <= RP_MAX_R, "spr_role_projection_rms: rank must be in [1, %d] (got %d)", RP_MAX_R,
              rank);
  if (bh == 0 || n == 0) return SPR_OK;
  SPR_REQUIRE(x && factor && out, "spr_role_projection_rms: null pointer");
  SPR_REQUIRE(bh <= 65535, "spr_role_projection_rms: too many heads");
  if (rp_streams(x, out, bh, n, rank, rank, 0)) {
    launch_role_projection_rows<0, 0>(bh, stream, static_cast<const uint16_t*>(x), factor, n, d, rank, out, rank, 0,
                                      1.0f, nullptr, nullptr);
  } else {
    launch_role_projection<0, 0>(bh, stream, static_cast<const uint16_t*>(x), factor, n, d, rank, out, rank, 0, 1.0f,
                                 nullptr, nullptr);
  }
  SPR_LAUNCHED("role_projection_kernel");
  return SPR_OK;
}

extern "C" size_t spr_role_k_projection_workspace(int64_t bh, int64_t n) {
  // one fp64 partial per 256-token unit of the streaming kernel (one per 1,024-token block suffices
  // for the other)
  return static_cast<size_t>(bh) * static_cast<size_t>((n + rs_unit(1) - 1) / rs_unit(1)) * sizeof(double);
}

extern "C" int spr_role_k_projection_ex(const void* x, const float* factor, int64_t bh, int64_t n, int32_t d,
                                        int32_t rank, int32_t precision, float weight, float* out, int32_t out_ld,
                                        int32_t out_col, float* key_scale, void* workspace, size_t workspace_bytes,
                                        hipStream_t stream) {
  SPR_REQUIRE(bh >= 0 && n >= 0, "spr_role_k_projection: bad size");
  SPR_REQUIRE(d == 64 || d == 128, "spr_role_k_projection: head dim must be 64 or 128 (got %d)", d);
  SPR_REQUIRE(rank >= 1 && rank <= RP_MAX_R, "spr_role_k_projection: rank must be in [1, %d] (got %d)", RP_MAX_R,
              rank);
  SPR_REQUIRE(precision >= 0 && precision <= 2, "spr_role_k_projection: precision must be 0, 1 or 2 (got %d)",
              precision);
  SPR_REQUIRE(out_col >= 0 && out_ld >= out_col + rank, "spr_role_k_projection: columns %d + %d exceed rows of %d",
              out_col, rank, out_ld);
  if (bh == 0) return SPR_OK;
  SPR_REQUIRE(n >= 1, "spr_role_k_projection: no tokens");
  SPR_REQUIRE(x && factor && out && key_scale, "spr_role_k_projection: null pointer");
  SPR_REQUIRE(bh <= 65535, "spr_role_k_projection: too many heads");
  // a partial per 1,024-token block is enough for the kernel above; the streaming one wants all
  const size_t least = static_cast<size_t>(bh) * ((n + rp_tokens(1) - 1) / rp_tokens(1)) * sizeof(double);
  if (workspace == nullptr || workspace_bytes < least) {
    spr_set_error("spr_role_k_projection: workspace of %zu bytes needed", least);
    return SPR_EWORKSPACE;
  }
  const uint16_t* xp = static_cast<const uint16_t*>(x);
  double* part = static_cast<double*>(workspace);
  const bool streams = rp_streams(x, out, bh, n, rank, out_ld, out_col) &&
                       workspace_bytes >= spr_role_k_projection_workspace(bh, n);
#define SPR_KP(PP)                                                                                             \
  do {                                                                                                         \
    if (streams) {                                                                                             \
      launch_role_projection_rows<1, PP>(bh, stream, xp, factor, n, d, rank, nullptr, 0, 0, 1.0f, part, nullptr); \
      SPR_LAUNCHED("role_projection_rows_kernel<sum of squares>");                                             \
      launch_role_projection_rows<2, PP>(bh, stream, xp, factor, n, d, rank, out, out_ld, out_col, weight, part,  \
                                         key_scale);                                                           \
      SPR_LAUNCHED("role_projection_rows_kernel<head scale>");                                                 \
      break;                                                                                                   \
    }                                                                                                          \
    launch_role_projection<1, PP>(bh, stream, xp, factor, n, d, rank, nullptr, 0, 0, 1.0f, part, nullptr);   \
    SPR_LAUNCHED("role_projection_kernel<sum of squares>");                                                    \
    launch_role_projection<2, PP>(bh, stream, xp, factor, n, d, rank, out, out_ld, out_col, weight, part,     \
                                  key_scale);                                                                  \
    SPR_LAUNCHED("role_projection_kernel<head scale>");                                                        \
  } while (0)
  if (precision == 0) SPR_KP(0); else if (precision == 1) SPR_KP(1); else SPR_KP(2);
#undef SPR_KP
  return SPR_OK;
}

extern "C" int spr_role_k_projection(const void* x, const float* factor, int64_t bh, int64_t n, int32_t d,
                                     int32_t rank, float* out, float* key_scale, void* workspace,
                                     size_t workspace_bytes, hipStream_t stream) {
  return spr_role_k_projection_ex(x, factor, bh, n, d, rank, 0, 1.0f, out, rank, 0, key_scale, workspace,
                                  workspace_bytes, stream);
}
