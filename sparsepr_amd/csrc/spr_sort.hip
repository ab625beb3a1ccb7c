// Stable argsort of small-range cluster labels (counting sort), per row.
//
// Produces the `sorted_indices = argsort(labels)` that every permute call site
// computes with torch.argsort (reference permute.py:154-157, n8_v6.py:905,
// hunyuanvideo.py:189, kmeans_utils.py:1676) and the per-cluster sizes and
// start offsets that the block-sparse attention schedule and the centroid
// update consume.  Within a cluster tokens keep ascending index order.
//
// Short rows of up to SMALL_BINS bins (sorts_small): one launch, one workgroup per row.
// Longer rows, three launches:
//   1. per (row, chunk of CHUNK tokens) label histogram in LDS;
//   2. per row: label totals, exclusive scan over labels, per-chunk bases;
//   3. per (row, chunk): every wave ranks a consecutive part of the chunk against counters of
//      its own, the counters become bases by a scan over the waves, and the token ids scatter.
// What bounds them is the serial chain of a wave's 64-token groups (each ranks against the
// counters the one before left, an LDS round trip), so a chunk is shared by as many waves as
// the counters leave room for: 24 rows of 118,800 labels, 256 bins: 57 us (one wave per 1024
// labels, 39 of them in the scatter) -> 44 us; 2 rows of 4096, 64 bins: 18 -> 6.4 us.
// Labels outside [0, k) go to a trailing overflow bucket (sorted last).
#include <type_traits>

#include "spr_common.h"

namespace {

constexpr int CHUNK = 4096;
constexpr int MAX_BINS = 8192;  // k + 1 <= MAX_BINS (32 KB of LDS counters)
constexpr int COUNTERS = 16384;   // LDS counters of a ranking workgroup (64 KB), shared by its waves;
constexpr int FEW_COUNTERS = 32768;  // 128 KB where the workgroups are at most one per CU
constexpr int SMALL_N = 16384;    // longest row sorted by one workgroup of 16 waves ...
constexpr int SMALL_BINS = COUNTERS / 16;  // ... whose counters fit

__device__ __forceinline__ uint32_t bin_of(int32_t label, int32_t k) {
  return (label >= 0 && label < k) ? static_cast<uint32_t>(label) : static_cast<uint32_t>(k);
}

__global__ __launch_bounds__(512) void label_hist_kernel(const int32_t* __restrict__ labels, int64_t n,
                                                         int32_t k, int32_t nchunks,
                                                         int32_t* __restrict__ hist) {
  extern __shared__ int32_t h[];  // [k + 1]
  const int32_t bins = k + 1;
  const int64_t row = blockIdx.y;
  const int64_t c0 = static_cast<int64_t>(blockIdx.x) * CHUNK;
  for (int j = threadIdx.x; j < bins; j += blockDim.x) h[j] = 0;
  __syncthreads();
  const int64_t c1 = c0 + CHUNK < n ? c0 + CHUNK : n;
  for (int64_t t = c0 + threadIdx.x; t < c1; t += blockDim.x) {
    atomicAdd(&h[bin_of(labels[row * n + t], k)], 1);
  }
  __syncthreads();
  int32_t* out = hist + (row * nchunks + blockIdx.x) * bins;
  for (int j = threadIdx.x; j < bins; j += blockDim.x) out[j] = h[j];
}

// One block per row.  hist[row][chunk][bin] counts -> bases (in place).
__global__ __launch_bounds__(1024) void label_scan_kernel(int32_t* __restrict__ hist, int32_t k,
                                                          int32_t nchunks, int32_t* __restrict__ sizes,
                                                          int32_t* __restrict__ offsets) {
  __shared__ int32_t tot[MAX_BINS];
  __shared__ int32_t wsum[16];
  constexpr int U = 8;  // chunk rows in flight per thread
  const int32_t bins = k + 1;
  const int64_t row = blockIdx.x;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  int32_t* hrow = hist + row * static_cast<int64_t>(nchunks) * bins;
  for (int j = tid; j < bins; j += blockDim.x) {
    int32_t s = 0;
    int c = 0;
    for (; c + U <= nchunks; c += U) {
      int32_t v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = hrow[(c + u) * bins + j];
#pragma unroll
      for (int u = 0; u < U; ++u) s += v[u];
    }
    for (; c < nchunks; ++c) s += hrow[c * bins + j];
    tot[j] = s;
  }
  __syncthreads();
  // exclusive scan of tot[0..bins): a contiguous segment per thread, segment sums
  // scanned across the block with wave shuffles
  const int per = (bins + blockDim.x - 1) / blockDim.x;
  const int lo = tid * per;
  const int hi = lo + per < bins ? lo + per : bins;
  int32_t seg = 0;
  for (int j = lo; j < hi; ++j) seg += tot[j];
  int32_t incl = seg;
  for (int o = 1; o < 64; o <<= 1) {
    const int32_t up = __shfl_up(incl, o, 64);
    if (lane >= o) incl += up;
  }
  if (lane == 63) wsum[wave] = incl;
  __syncthreads();
  int32_t before = 0;
  for (int w = 0; w < wave; ++w) before += wsum[w];
  {
    int32_t run = before + incl - seg;
    for (int j = lo; j < hi; ++j) {
      int32_t v = tot[j];
      if (sizes != nullptr && j < k) sizes[row * k + j] = v;
      tot[j] = run;
      run += v;
    }
  }
  __syncthreads();
  for (int j = tid; j < bins; j += blockDim.x) {
    if (offsets != nullptr) offsets[row * (k + 1) + j] = tot[j];
    int32_t run = tot[j];
    int c = 0;
    for (; c + U <= nchunks; c += U) {
      int32_t v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = hrow[(c + u) * bins + j];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        hrow[(c + u) * bins + j] = run;
        run += v[u];
      }
    }
    for (; c < nchunks; ++c) {
      int32_t a = hrow[c * bins + j];
      hrow[c * bins + j] = run;
      run += a;
    }
  }
}

// Ranks of a wave's labels among its earlier equal ones: group g of 64 consecutive labels sits
// in bin[g] (-1 past the end), cnt holds the wave's count per bin, which the ranks extend.
template <int G>
__device__ __forceinline__ void rank_groups(const int32_t (&bin)[G], int32_t (&rank)[G], int nbits, int lane,
                                            int32_t* __restrict__ cnt) {
#pragma unroll
  for (int g = 0; g < G; ++g) {
    // lanes holding the same bin, one ballot per bin bit (nbits bits hold every bin and
    // keep the pattern of -1, past the end, apart from all of them); the rank is the
    // number of such lanes below this one, which keeps the sort stable
    uint64_t same = ~0ull;
    for (int bit = 0; bit < nbits; ++bit) {
      const bool set = (bin[g] >> bit) & 1;
      const uint64_t m = __ballot(set);
      same &= set ? m : ~m;
    }
    const int below = __popcll(same & ((1ull << lane) - 1ull));
    const int count = __popcll(same);
    const bool live = bin[g] >= 0;
    rank[g] = live ? cnt[bin[g]] + below : 0;
    __builtin_amdgcn_wave_barrier();
    if (live && below == count - 1) cnt[bin[g]] = rank[g] + 1;
    __builtin_amdgcn_wave_barrier();
  }
}

// Workgroup per (row, chunk) of W waves; wave w ranks labels w * 64 G .. + 64 G of the chunk.
template <int W>
__global__ __launch_bounds__(W * 64) void label_scatter_kernel(const int32_t* __restrict__ labels, int64_t n,
                                                               int32_t k, int32_t nchunks,
                                                               const int32_t* __restrict__ bases,
                                                               int32_t* __restrict__ sorted_idx) {
  extern __shared__ int32_t cnt[];  // [W][k + 1]
  constexpr int G = CHUNK / 64 / W;
  const int32_t bins = k + 1;
  const int nbits = 32 - __builtin_clz(static_cast<uint32_t>(bins));  // 2^nbits > k + 1 > every bin
  const int64_t row = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t t0 = static_cast<int64_t>(blockIdx.x) * CHUNK + wave * (64 * G) + lane;
  int32_t bin[G], rank[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int64_t t = t0 + 64 * g;
    bin[g] = t < n ? static_cast<int32_t>(bin_of(labels[row * n + t], k)) : -1;
  }
  for (int j = tid; j < W * bins; j += W * 64) cnt[j] = 0;
  __syncthreads();
  rank_groups<G>(bin, rank, nbits, lane, cnt + wave * bins);
  __syncthreads();
  const int32_t* b = bases + (row * nchunks + blockIdx.x) * bins;
  for (int j = tid; j < bins; j += W * 64) {
    int32_t run = b[j];
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const int32_t c = cnt[w * bins + j];
      cnt[w * bins + j] = run;
      run += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int g = 0; g < G; ++g) {
    if (bin[g] < 0) continue;
    const int64_t pos = static_cast<int64_t>(cnt[wave * bins + bin[g]]) + rank[g];
    if (pos >= 0 && pos < n) sorted_idx[row * n + pos] = static_cast<int32_t>(t0 + 64 * g);
  }
}

// A whole row in one workgroup of 16 waves, 64 G labels each (n <= 1024 G): ranks, then the
// counters' scan over waves and bins gives sizes, offsets and the waves' bases.
template <int G>
__global__ __launch_bounds__(1024) void label_sort_small_kernel(const int32_t* __restrict__ labels, int32_t n,
                                                                int32_t k, int32_t* __restrict__ sorted_idx,
                                                                int32_t* __restrict__ sizes,
                                                                int32_t* __restrict__ offsets) {
  extern __shared__ int32_t cnt[];  // [16][k + 1]
  __shared__ int32_t wsum[16];
  constexpr int W = 16;
  const int32_t bins = k + 1;  // at most SMALL_BINS: one bin per thread below
  const int nbits = 32 - __builtin_clz(static_cast<uint32_t>(bins));
  const int64_t row = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int32_t* lab = labels + row * n;
  const int32_t t0 = wave * (64 * G) + lane;
  int32_t bin[G], rank[G];
#pragma unroll
  for (int g = 0; g < G; ++g) bin[g] = t0 + 64 * g < n ? static_cast<int32_t>(bin_of(lab[t0 + 64 * g], k)) : -1;
  for (int j = tid; j < W * bins; j += W * 64) cnt[j] = 0;
  __syncthreads();
  rank_groups<G>(bin, rank, nbits, lane, cnt + wave * bins);
  __syncthreads();
  int32_t total = 0;
  if (tid < bins) {
#pragma unroll
    for (int w = 0; w < W; ++w) total += cnt[w * bins + tid];
  }
  int32_t incl = total;
  for (int o = 1; o < 64; o <<= 1) {
    const int32_t up = __shfl_up(incl, o, 64);
    if (lane >= o) incl += up;
  }
  if (lane == 63) wsum[wave] = incl;
  __syncthreads();
  int32_t run = incl - total;
  for (int w = 0; w < wave; ++w) run += wsum[w];
  if (tid < bins) {
    if (sizes != nullptr && tid < k) sizes[row * k + tid] = total;
    if (offsets != nullptr) offsets[row * (k + 1) + tid] = run;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const int32_t c = cnt[w * bins + tid];
      cnt[w * bins + tid] = run;
      run += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int g = 0; g < G; ++g) {
    if (bin[g] < 0) continue;
    const int32_t pos = cnt[wave * bins + bin[g]] + rank[g];
    if (pos >= 0 && pos < n) sorted_idx[row * n + pos] = t0 + 64 * g;
  }
}

__global__ void fill_i32_kernel(int32_t* __restrict__ p, int64_t count, int32_t value) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < count;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x)
    p[i] = value;
}

// One launch instead of three, and with one workgroup per row the faster up to 8,192 labels (24
// rows, 256 bins, in a graph: 8,192 labels 12.3 us, 15 in three launches; 16,384 22.3 us, 16 in three),
// above that where the rows fill the chip (256 rows of 16,384: 43 us, 44 in three launches, with 8
// bins 18 and 28).
bool sorts_small(int64_t rows, int64_t n, int32_t k) {
  return n <= (rows >= 128 ? SMALL_N : SMALL_N / 2) && k + 1 <= SMALL_BINS;
}

}  // namespace

extern "C" size_t spr_argsort_labels_workspace(int64_t rows, int64_t n, int32_t k) {
  if (sorts_small(rows, n, k)) return 16;  // none is used
  const int64_t nchunks = spr::ceil_div(n, CHUNK);
  return static_cast<size_t>(rows * nchunks * (static_cast<int64_t>(k) + 1) * 4);
}

// labels int32 [rows, n] in [0, k) -> sorted_idx int32 [rows, n] (stable),
// sizes int32 [rows, k] (nullable), offsets int32 [rows, k + 1] (nullable).
extern "C" int spr_argsort_labels(const int32_t* labels, int64_t rows, int64_t n, int32_t k,
                                  int32_t* sorted_idx, int32_t* sizes, int32_t* offsets, void* workspace,
                                  size_t workspace_bytes, hipStream_t stream) {
  SPR_REQUIRE(rows >= 0 && n >= 0, "spr_argsort_labels: negative size");
  SPR_REQUIRE(k >= 1 && k + 1 <= MAX_BINS, "spr_argsort_labels: k=%d outside [1, %d]", k, MAX_BINS - 1);
  SPR_REQUIRE(n < (int64_t(1) << 31), "spr_argsort_labels: n too large");
  SPR_REQUIRE(rows <= 65535, "spr_argsort_labels: rows=%lld exceeds 65535", (long long)rows);
  if (rows == 0) return SPR_OK;
  if (n == 0) {
    // Empty rows: sizes and offsets are all zero.
    if (sizes) fill_i32_kernel<<<64, 256, 0, stream>>>(sizes, rows * k, 0);
    if (offsets) fill_i32_kernel<<<64, 256, 0, stream>>>(offsets, rows * (k + 1), 0);
    SPR_LAUNCHED("spr_argsort_labels");
    return SPR_OK;
  }
  SPR_REQUIRE(labels && sorted_idx && workspace, "spr_argsort_labels: null pointer");
  const size_t need = spr_argsort_labels_workspace(rows, n, k);
  if (workspace_bytes < need) {
    spr_set_error("spr_argsort_labels: workspace %zu < %zu bytes", workspace_bytes, need);
    return SPR_EWORKSPACE;
  }
  const size_t bin_bytes = static_cast<size_t>(k + 1) * sizeof(int32_t);
  if (sorts_small(rows, n, k)) {
    if (n <= 4096) {
      label_sort_small_kernel<4><<<dim3(rows), 1024, 16 * bin_bytes, stream>>>(labels, static_cast<int32_t>(n), k,
                                                                              sorted_idx, sizes, offsets);
    } else if (n <= 8192) {
      label_sort_small_kernel<8><<<dim3(rows), 1024, 16 * bin_bytes, stream>>>(labels, static_cast<int32_t>(n), k,
                                                                              sorted_idx, sizes, offsets);
    } else {
      label_sort_small_kernel<16><<<dim3(rows), 1024, 16 * bin_bytes, stream>>>(labels, static_cast<int32_t>(n), k,
                                                                               sorted_idx, sizes, offsets);
    }
    SPR_LAUNCHED("label_sort_small_kernel");
    return SPR_OK;
  }
  const int32_t nchunks = static_cast<int32_t>(spr::ceil_div(n, CHUNK));
  int32_t* hist = static_cast<int32_t*>(workspace);
  label_hist_kernel<<<dim3(nchunks, rows), 512, bin_bytes, stream>>>(labels, n, k, nchunks, hist);
  SPR_LAUNCHED("label_hist_kernel");
  label_scan_kernel<<<dim3(rows), 1024, 0, stream>>>(hist, k, nchunks, sizes, offsets);
  SPR_LAUNCHED("label_scan_kernel");
  // as many waves per chunk as counters fit: a whole CU's LDS where the chunks leave CUs idle (2
  // rows of 8,192 labels, 4,096 bins: the sort 45.8 us with two waves, 31.7 with four)
  const int32_t counters = static_cast<int64_t>(nchunks) * rows <= 256 ? FEW_COUNTERS : COUNTERS;
  auto scatter = [&](auto waves) -> int {
    constexpr int W = decltype(waves)::value;
    const size_t bytes = W * bin_bytes;
    if (bytes > 65536) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&label_scatter_kernel<W>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, FEW_COUNTERS * 4);
      if (e != hipSuccess) {
        spr_set_error("spr_argsort_labels: hipFuncSetAttribute failed: %s", hipGetErrorString(e));
        return SPR_ELAUNCH;
      }
    }
    label_scatter_kernel<W><<<dim3(nchunks, rows), W * 64, bytes, stream>>>(labels, n, k, nchunks, hist, sorted_idx);
    return SPR_OK;
  };
  int st;
  if (16 * (k + 1) <= counters) st = scatter(std::integral_constant<int, 16>{});
  else if (8 * (k + 1) <= counters) st = scatter(std::integral_constant<int, 8>{});
  else if (4 * (k + 1) <= counters) st = scatter(std::integral_constant<int, 4>{});
  else st = scatter(std::integral_constant<int, 2>{});
  if (st != SPR_OK) return st;
  SPR_LAUNCHED("label_scatter_kernel");
  return SPR_OK;
}
