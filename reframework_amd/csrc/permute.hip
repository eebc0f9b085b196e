// Stable counting sort of routed slots by expert.
//
// Replaces the grouping of fused_experts (reframework/moe/fused.py:70-80),
// which visits experts in ascending id and, inside an expert, slots in
// ascending flat (t,k) order. Two launches, no host round trip:
//   1. count:   each block histograms kPermuteChunk slots into LDS and writes
//               its per-expert counts (256 slots a block, one per thread: at
//               1024 a block ranked its slots in four dependent rounds, and
//               the scatter of 8192 slots ran on 8 CUs);
//   2. scatter: each block rebuilds the global expert starts and its own
//               prefix from the count table, ranks its slots stably with
//               wavefront ballots, and writes slot_to_row / row_src. Block 0
//               also writes expert_offsets and the tile map the expert-FFN
//               kernels are launched over.
// Up to kPermuteSingleMax slots one block of that many threads does both.
// Only indices move here (4*T*K bytes each way); token rows are gathered later
// by the gate_up kernel straight from x, so no permuted copy of x is written.
#include "common.h"

namespace moe355 {
namespace {

constexpr int kThreads = 256;
constexpr int kRounds = kPermuteChunk / kThreads;  // count + scatter launches
constexpr int kWaves = kThreads / kWave;
constexpr int kOneThreads = kPermuteSingleMax;      // the one-block permute: a thread per slot
constexpr int kOneWaves = kOneThreads / kWave;
static_assert(kMaxExperts <= 256, "the scatter ranks slots by the 8 bits of the expert id");

__global__ __launch_bounds__(kThreads) void count_kernel(const PermuteArgs a) {
  __shared__ int hist[kMaxExperts];
  const int b = blockIdx.x, tid = threadIdx.x;
  for (int e = tid; e < a.E; e += kThreads) hist[e] = 0;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    const int slot = b * kPermuteChunk + r * kThreads + tid;
    if (slot < a.R) {
      const int e = routed_expert(a, slot);
      if (e >= 0) atomicAdd(&hist[e], 1);
    }
  }
  __syncthreads();
  for (int e = tid; e < a.E; e += kThreads) a.block_counts[b * a.E + e] = hist[e];
}

// Rank of this lane's slot among the wave's slots of the same expert (e < 0: not
// routed): the routed lanes that agree with this lane on each of the 8 bits of
// the expert id (E <= 256), one ballot per bit instead of one per distinct
// expert. `same` gets those lanes.
__device__ __forceinline__ int rank_in_wave(int e, int lane, unsigned long long* same) {
  unsigned long long m = __ballot(e >= 0);
#pragma unroll
  for (int bit = 0; bit < 8; ++bit) {
    const bool set = (e >> bit) & 1;
    const unsigned long long b = __ballot(set);
    m &= set ? b : ~b;
  }
  *same = m;
  return __popcll(m & ((1ull << lane) - 1ull));
}

// Exclusive scan by one wave of E values, lane l owning l*per .. l*per+per-1
// (per <= 4 for E <= 256): out[i] for i <= E, out[E] the sum.
template <typename F>
__device__ __forceinline__ void wave_scan(int E, int lane, F value, int* out) {
  constexpr int kPer = kMaxExperts / kWave;
  const int per = (E + kWave - 1) / kWave;
  int v[kPer], sum = 0;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int x = lane * per + i;
    v[i] = i < per && x < E ? value(x) : 0;
    sum += v[i];
  }
  int inc = sum;  // inclusive across lanes
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const int up = __shfl_up(inc, o, kWave);
    if (lane >= o) inc += up;
  }
  int ex = inc - sum;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int x = lane * per + i;
    if (i < per && x < E) out[x] = ex;
    ex += v[i];
  }
  if (lane == kWave - 1) out[E] = inc;
}

// The tile map lists the experts' tiles in an interleaved order of their
// sizes (largest, smallest, second largest, second smallest, ..; ties by
// expert id), so the GEMMs' rounds mix weight-stream-bound items of small
// experts with MFMA-bound items of large ones: fine-grained 4096 tokens
// gate_up -2 %, Phi-3.5 2048 tokens -2 %, Mixtral 4096 tokens down -2 %
// against expert-id order. Rank r of the size order goes to place 2 r in
// the first half, 2 (E - 1 - r) + 1 in the second.
__device__ __forceinline__ int size_place(const int* total, int E, int e) {
  const int n = total[e];
  int r = 0;
  for (int f = 0; f < E; ++f) r += (total[f] > n || (total[f] == n && f < e)) ? 1 : 0;
  return 2 * r < E ? 2 * r : 2 * (E - 1 - r) + 1;
}

// Tile j of the map (place_start: first tile of each place of `order`).
__device__ __forceinline__ void write_tile(const PermuteArgs& a, const int* start, const int* order,
                                           const int* place_start, int j) {
  int lo = 0, hi = a.E - 1;  // last place with place_start[p] <= j
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (place_start[mid] <= j) lo = mid; else hi = mid - 1;
  }
  const int e = order[lo];
  a.tile_map[2 + 2 * j] = e;
  a.tile_map[3 + 2 * j] =
      start[e] + (j - place_start[lo]) * tile_height(start[e + 1] - start[e], a.tile_rows);
}

// All slots fit one block (up to kPermuteSingleMax), one thread each: a chain of
// dependent steps, so the fewest of them decide. Each wave ranks its 64 slots
// and counts them per expert; a thread per expert turns the waves' counts into
// bases; then one wave scans the experts while the others rank them by size, and
// rows and tile map are written. With 256 threads in four rounds, each with its
// own barriers, and a counting pass before them this took 10.9 us at 1024 slots
// of 8 experts and 12.5 at 999 of 12; now 5.7 and 5.6.
__global__ __launch_bounds__(kOneThreads) void permute_one_kernel(const PermuteArgs a) {
  __shared__ int wave_cnt[kOneWaves][kMaxExperts];  // slots of expert e in a wave, then before it
  __shared__ int total[kMaxExperts], start[kMaxExperts + 1];
  __shared__ int order[kMaxExperts], place_start[kMaxExperts + 1];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;

  const int e = tid < a.R ? routed_expert(a, tid) : -1;
  for (int x = lane; x < a.E; x += kWave) wave_cnt[wave][x] = 0;  // this wave's own row
  unsigned long long same;
  const int rank = rank_in_wave(e, lane, &same);
  if (e >= 0 && rank == 0) wave_cnt[wave][e] = __popcll(same);
  __syncthreads();
  if (tid < a.E) {
    int c[kOneWaves], sum = 0;
#pragma unroll
    for (int w = 0; w < kOneWaves; ++w) c[w] = wave_cnt[w][tid];
#pragma unroll
    for (int w = 0; w < kOneWaves; ++w) {
      wave_cnt[w][tid] = sum;
      sum += c[w];
    }
    total[tid] = sum;
  }
  __syncthreads();
  if (wave == 0) wave_scan(a.E, lane, [&](int x) { return total[x]; }, start);
  for (int x = tid - kWave; x >= 0 && x < a.E; x += kOneThreads) order[size_place(total, a.E, x)] = x;
  __syncthreads();
  if (wave == 1)
    wave_scan(a.E, lane, [&](int x) { return (total[order[x]] + a.tile_rows - 1) / a.tile_rows; },
              place_start);
  if (tid < a.R) {
    const int row = e >= 0 ? start[e] + wave_cnt[wave][e] + rank : -1;
    a.slot_to_row[tid] = row;
    if (row >= 0) a.row_src[row] = tid / a.K;
  }
  for (int x = tid; x <= a.E; x += kOneThreads) a.offsets[x] = start[x];
  __syncthreads();
  const int ntiles = min(place_start[a.E], a.max_tiles);
  if (tid == 0) {
    a.tile_map[0] = ntiles;
    a.tile_map[1] = a.tile_rows;
  }
  for (int j = tid; j < ntiles; j += kOneThreads) write_tile(a, start, order, place_start, j);
}

__global__ __launch_bounds__(kThreads) void scatter_kernel(const PermuteArgs a) {
  __shared__ int base[kMaxExperts];       // first row of this block's slots of expert e
  __shared__ int start[kMaxExperts + 1];  // expert_offsets
  __shared__ int total[kMaxExperts];
  __shared__ int wave_cnt[kWaves][kMaxExperts];

  const int b = blockIdx.x, tid = threadIdx.x;
  const int lane = tid & (kWave - 1), wave = tid / kWave;

  {
    // Slots of expert e in all blocks (total) and in the blocks before this
    // one (base), from the count table. Thread tid sums expert tid % E over
    // part tid / E of the blocks (P = min(256 / E, 8) parts; one part when
    // E > 128) with its loads unrolled, so they are in flight together; the
    // parts are added in LDS, at most 8 per expert. One thread per expert
    // walking every block paid one L2 round trip per block (32 for 64 experts
    // at 4096 tokens).
    __shared__ int ptot[kThreads], ppre[kThreads];
    const int P = min(kThreads / a.E, 8);
    const int e = tid % a.E, p = tid / a.E;
    int tot = 0, pre = 0;
    if (p < P) {
      const int per = (a.n_blocks + P - 1) / P;
      const int b1 = min(a.n_blocks, (p + 1) * per);
#pragma unroll 8
      for (int bb = p * per; bb < b1; ++bb) {
        const int c = a.block_counts[bb * a.E + e];
        tot += c;
        pre += bb < b ? c : 0;
      }
    }
    ptot[tid] = tot;
    ppre[tid] = pre;
    __syncthreads();
    for (int x = tid; x < a.E; x += kThreads) {
      int t2 = 0, p2 = 0;
      for (int q = 0; q < P; ++q) {
        t2 += ptot[q * a.E + x];
        p2 += ppre[q * a.E + x];
      }
      total[x] = t2;
      base[x] = p2;
    }
  }
  __syncthreads();
  if (wave == 0) wave_scan(a.E, lane, [&](int x) { return total[x]; }, start);
  __syncthreads();
  for (int e = tid; e < a.E; e += kThreads) base[e] += start[e];

  if (b == 0) {
    __shared__ int order[kMaxExperts];            // expert at place p
    __shared__ int place_start[kMaxExperts + 1];  // first tile of place p
    for (int e = tid; e <= a.E; e += kThreads) a.offsets[e] = start[e];
    for (int e = tid; e < a.E; e += kThreads) order[size_place(total, a.E, e)] = e;
    __syncthreads();
    if (wave == 0)
      wave_scan(a.E, lane, [&](int x) { return (total[order[x]] + a.tile_rows - 1) / a.tile_rows; },
                place_start);
    __syncthreads();
    const int ntiles = min(place_start[a.E], a.max_tiles);
    if (tid == 0) {
      a.tile_map[0] = ntiles;
      a.tile_map[1] = a.tile_rows;
    }
    for (int j = tid; j < ntiles; j += kThreads) write_tile(a, start, order, place_start, j);
  }

  for (int r = 0; r < kRounds; ++r) {
    for (int i = tid; i < kWaves * a.E; i += kThreads) wave_cnt[i / a.E][i % a.E] = 0;
    __syncthreads();
    const int slot = b * kPermuteChunk + r * kThreads + tid;
    const int e = slot < a.R ? routed_expert(a, slot) : -1;
    unsigned long long same;
    const int rank = rank_in_wave(e, lane, &same);
    if (e >= 0 && rank == 0) wave_cnt[wave][e] = __popcll(same);
    __syncthreads();
    if (slot < a.R) {
      if (e >= 0) {
        int row = base[e] + rank;
        for (int w = 0; w < wave; ++w) row += wave_cnt[w][e];
        a.slot_to_row[slot] = row;
        a.row_src[row] = slot / a.K;
      } else {
        a.slot_to_row[slot] = -1;
      }
    }
    __syncthreads();
    for (int ee = tid; ee < a.E; ee += kThreads) {
      int add = 0;
      for (int w = 0; w < kWaves; ++w) add += wave_cnt[w][ee];
      base[ee] += add;
    }
    __syncthreads();
  }
}

}  // namespace

hipError_t launch_permute(const PermuteArgs& a, hipStream_t s) {
  if (a.R == 0) return hipSuccess;
  if (a.n_blocks == 1) {
    permute_one_kernel<<<dim3(1), dim3(kOneThreads), 0, s>>>(a);
    return hipGetLastError();
  }
  count_kernel<<<dim3(a.n_blocks), dim3(kThreads), 0, s>>>(a);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
  scatter_kernel<<<dim3(a.n_blocks), dim3(kThreads), 0, s>>>(a);
  return hipGetLastError();
}

}  // namespace moe355
