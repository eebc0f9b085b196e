// Grouped expert FFN on one workgroup per (K-split, weight tile, token tile)
// item: fp32 layers, sizes the bf16/f16 tiled kernels do not take (H no multiple
// of 256, I no multiple of 128, token rows past 2 GB), and bf16/f16 groups of
// about 10 to 64 rows on 128-row token tiles. Any H and I of whole 16-byte
// vectors run here. Groups of up to ten rows run ffn_skinny_kernel instead.
//
// Replaces the per-expert GEMMs of fused_experts (reframework/moe/fused.py:76-83)
// with the same contract as the tiled kernels: items over the permute's tile
// map, token rows gathered from x through row_src, the gated activation fused
// into gate_up, fp32 partials per K-split (or, y16, the rounded sum) from down.
//
// Tile: kW weight rows (gate_up: half gate rows, half the matching up rows) x
// up to kT token rows, 4 waves in a 2x2 arrangement, steps of 128 bytes of K
// (64 k of 16-bit types, 32 of fp32). Both types read the same 16-byte operand
// chunks: lane l takes row l % 16, chunk 4 h + l / 16 of the step; a 16-bit
// chunk pair is one v_mfma_f32_16x16x32, an fp32 pair four
// v_mfma_f32_16x16x4_f32 (pipe::Mfma16). The K loop exists in one copy per
// number of 32-row token groups, which are all it loads and multiplies.
//
// Global -> registers -> LDS: kDepth steps are in flight in registers while
// one is multiplied from the LDS, and two to five workgroups share a CU, so
// that one's loads fly while another's MFMAs run. Register staging rather than
// direct-to-LDS loads, because chunks past the K range are replaced by zeros on
// the way (in both operands: past a weight row lies the next one, whose values
// may be infinite) and operands need not be 16-byte aligned.
//
// fp32 is bound by its MFMA rate (157 TFLOP/s, a sixteenth of bf16's; a large
// library product reaches 153, an all-register probe 150; the MFMAs are busy 73 to 80 % of the cycles in
// which a CU holds work) and by the last round of items, which is why its tile
// is small. 16-bit sizes on this path are bound by the weight stream
// and the LDS. Before, one kernel did both with fp32 FMAs on the VALU, one
// element per LDS read (gate_up + down, 64 x 64 tiles, 16 k a step). Layers,
// before -> now: fp32 H 1024, I 2816, 8 experts top-2, 512 tokens 1.04 -> 0.21 ms
// (86 TFLOP/s), 128 tokens 0.88 -> 0.10 ms; bf16 H 1240, I 3304, 12 experts
// top-3, 333 tokens 1.44 -> 0.123 ms, 60 tokens 1.24 -> 0.084 ms (the activation's
// expf and division are 1 % of it).
//
// Groups of 10 to 64 rows of the tiled sizes are bound by the weight stream.
// Against the persistent 128-row kernel (one workgroup per CU, which overlaps
// nothing with its barriers and epilogues and shares L2 between weights and
// tokens), layers: Mixtral shape, 44 / 197 / 256 tokens 559 / 567 / 577 ->
// 450 / 479 / 513 us; 16 experts of I 6400, 300 tokens 486 -> 444; 66 experts
// top-8 of H 2048, I 1408, 128 / 300 tokens 249 / 256 -> 219 / 237. Above some 40 to
// 75 rows per expert, by the size of the layer, the persistent kernel wins
// (mid_sized in capi.hip has the line and both sides of it).
#include <algorithm>
#include <climits>

#include "common.h"
#include "dma_pipe.h"

namespace moe355 {
namespace {

constexpr int kThreads = 256;
constexpr int kGridX = 1 << 22;  // workgroups per grid row: HIP takes fewer than 2^32 threads in x
constexpr int kRowBytes = 128;  // bytes of one operand row per step
constexpr int kChunks = kRowBytes / 16;
constexpr int kRowsPerPass = kThreads / kChunks;  // 32 rows per load of the workgroup

// kFastAct: gate_act_fast, on the plans that the tiled kernels share (128-row
// maps); MOE355_PATH_SIMT applies gate_act in every type.
template <int W, int T, int Depth, bool FastAct = false>
struct Config {
  static constexpr int kW = W, kT = T, kDepth = Depth;
  static constexpr bool kFastAct = FastAct;
};

// LDS place of chunk c of row r: 16 rows read at one chunk hit 16 distinct
// 16-byte bank groups, and the 8 whole rows a wave writes cover 1 KB.
__device__ __forceinline__ uint32_t lds_at(int r, int c) {
  return static_cast<uint32_t>(r * kRowBytes + ((c ^ ((r >> 1) & 7)) << 4));
}

template <typename T, bool kGateUp, typename C>
__global__ __launch_bounds__(kThreads, 2) void ffn_general_kernel(const FfnArgs a) {
  constexpr int N = Vec16<T>::N;                    // elements per chunk
  constexpr int NI = C::kW / 32, NX = C::kT / 32;   // weight blocks, token groups
  constexpr int kWLoads = C::kW / kRowsPerPass, D = C::kDepth;
  constexpr int kBufBytes = (C::kW + C::kT) * kRowBytes;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[D][kBufBytes];

  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wave_w = wave >> 1, wave_t = wave & 1;

  // Item of this workgroup. Workgroups go to the XCDs round-robin, so with a
  // multiple of 8 of (weight tile, split) pairs q every XCD takes the pairs
  // q % 8 of every token tile, and a slab that several tiles read is fetched into
  // one L2. 16-bit gate_up walks the token tiles of a pair first, down and fp32
  // the pairs of a tile (us, token tile first / pair first / consecutive items
  // per XCD, as other sizes keep: Mixtral shape f16, 197 tokens, gate_up 306 / 329
  // / 316, down 169 / 162 / 166; fp32 H 1024, I 2816, 8 experts, 100 tokens,
  // gate_up 61 / 50 / 60: its few unequal items spread over the CUs).
  const int n_t = a.tile_map[0];
  const int n_q = a.n_wtiles * a.splits, n_items = n_t * n_q;
  const int pid = blockIdx.y * gridDim.x + blockIdx.x;  // rows of kGridX keep the XCD of pid % 8
  if (pid >= n_items) return;
  int tt, q0;
  if (n_q % 8) {
    const int L = xcd_remap(pid, n_items);
    tt = L % n_t;
    q0 = L / n_t;
  } else if (kGateUp && !std::is_same<T, float>::value) {
    const int slot = pid >> 3;
    tt = slot % n_t;
    q0 = slot / n_t * 8 + (pid & 7);
  } else {
    tt = pid / n_q;
    q0 = pid % n_q;
  }
  const int wtile = q0 % a.n_wtiles, split = q0 / a.n_wtiles;
  const int e = a.tile_map[2 + 2 * tt], row0 = a.tile_map[3 + 2 * tt];
  const int first = a.offsets[e], last = a.offsets[e + 1];  // the expert's rows
  const int row_end = min(row0 + C::kT, last);

  const int ld = kGateUp ? a.H : a.I, nout = kGateUp ? a.I : a.H;
  const int kbeg = split * a.k_per_split, kend = min(ld, kbeg + a.k_per_split);
  const int nchunks = kend > kbeg ? (kend - kbeg) / N : 0;  // ld and k_per_split are whole chunks
  const int nsteps = (nchunks + kChunks - 1) / kChunks;

  // Load q of a step: rows q * 32 + tid / 8 of the operand, chunk tid % 8.
  // Weight rows past the last feature and token rows past the group's end read
  // the last one: their results are not stored.
  const int lrow = tid / kChunks, lc = tid % kChunks;
  const T* wp[kWLoads];
  const T* xp[NX];
  const T* w = static_cast<const T*>(a.w[e]);
#pragma unroll
  for (int q = 0; q < kWLoads; ++q) {
    const int r = q * kRowsPerPass + lrow;
    const int f = kGateUp ? wtile * (C::kW / 2) + (r & (C::kW / 2 - 1)) : wtile * C::kW + r;
    const int wr = min(f, nout - 1) + (kGateUp && r >= C::kW / 2 ? a.I : 0);
    wp[q] = w + static_cast<size_t>(wr) * ld + kbeg;
  }
#pragma unroll
  for (int q = 0; q < NX; ++q) {
    const int prow = min(row0 + q * kRowsPerPass + lrow, row_end - 1);
    const int src = kGateUp ? a.row_src[prow] : prow;
    xp[q] = static_cast<const T*>(a.x) + static_cast<size_t>(src) * ld + kbeg;
  }
  const uint32_t at = lds_at(lrow, lc);  // row 32 q + lrow lies 32 q rows on

  // Operand rows of this wave: weight blocks i (gate_up: the first half gate,
  // the second the matching up rows), token blocks 2 j + wave_t.
  const int lr = lane & 15, kq = lane >> 4;
  auto w_row = [&](int i) {
    return kGateUp ? wave_w * (C::kW / 4) + (i % (NI / 2)) * 16 + (i >= NI / 2 ? C::kW / 2 : 0)
                   : wave_w * (C::kW / 2) + i * 16;
  };
  const uint32_t coff[2] = {lds_at(lr, kq), lds_at(lr, 4 + kq)};  // block rows are multiples of 16

  f32x4 acc[NI][NX];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NX; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto barrier = [&]() {  // waits for LDS accesses only: the loads stay in flight
    pipe::wait_lgkm0();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
  };

  // The K loop for J token groups; kOnce: the weights are read by this item
  // alone and loaded non-temporally, so that they do not evict the token rows
  // every item of the expert reads from L2.
  auto k_loop = [&](auto jc, auto once) {
    constexpr int J = decltype(jc)::value;
    constexpr bool kOnce = decltype(once)::value;
    u32x4 wr[D][kWLoads], xr[D][J];
    const bool last_block = row_end - row0 > 32 * (J - 1) + 16 * wave_t;  // this wave's J-th in use
    // Steps past the last load it again (never stored), and chunks past the K
    // range the last one (zeros by store_step): every load is unconditional, so
    // the compiler counts the loads in flight exactly and waits for the oldest
    // step only (under a branch it drained the newer step's loads as well).
    auto load_step = [&](int slot, int st) {
      const int off = min(min(st, nsteps - 1) * kChunks + lc, nchunks - 1) * N;
#pragma unroll
      for (int q = 0; q < kWLoads; ++q)
        wr[slot][q] = kOnce ? load16_any_once(wp[q] + off) : load16_any(wp[q] + off);
#pragma unroll
      for (int q = 0; q < J; ++q) xr[slot][q] = load16_any(xp[q] + off);
    };
    auto store_step = [&](int slot, int st, uint8_t* buf) {
      const u32x4 zero = {0, 0, 0, 0};
      const bool in = st * kChunks + lc < nchunks;
#pragma unroll
      for (int q = 0; q < kWLoads; ++q)
        *reinterpret_cast<u32x4*>(buf + at + q * kRowsPerPass * kRowBytes) = in ? wr[slot][q] : zero;
#pragma unroll
      for (int q = 0; q < J; ++q)
        *reinterpret_cast<u32x4*>(buf + at + (C::kW + q * kRowsPerPass) * kRowBytes) =
            in ? xr[slot][q] : zero;
    };
    auto multiply = [&](const uint8_t* buf) {
      const uint8_t* xb = buf + (C::kW + wave_t * 16) * kRowBytes;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        u32x4 fa[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i)
          fa[i] = *reinterpret_cast<const u32x4*>(buf + w_row(i) * kRowBytes + coff[h]);
#pragma unroll
        for (int j = 0; j < J; ++j) {
          if (j == J - 1 && !last_block) continue;
          const u32x4 b = *reinterpret_cast<const u32x4*>(xb + j * 32 * kRowBytes + coff[h]);
#pragma unroll
          for (int i = 0; i < NI; ++i) acc[i][j] = pipe::Mfma16<T>::mma(fa[i], b, acc[i][j]);
        }
      }
    };
    // One LDS buffer (D = 1): written between two barriers, after every wave's
    // reads of the step before. Two (D = 2): a buffer is written again two steps
    // after its use, and the one barrier between comes after those reads.
    auto step = [&](auto dc, int st) {
      constexpr int d = decltype(dc)::value;
      if (D == 1 && st > 0) barrier();
      store_step(d, st, lds[d]);
      load_step(d, st + D);
      barrier();
      multiply(lds[d]);
    };
#pragma unroll
    for (int d = 0; d < D; ++d) load_step(d, d);
    int st = 0;
    for (; st + D <= nsteps; st += D) {
      step(std::integral_constant<int, 0>{}, st);
      if constexpr (D == 2) step(std::integral_constant<int, 1>{}, st + 1);
    }
    if (st < nsteps) step(std::integral_constant<int, 0>{}, st);
  };
  auto dispatch = [&](auto once) {
    const int groups = (row_end - row0 + 31) / 32;
    if (groups <= 1)
      k_loop(std::integral_constant<int, 1>{}, once);
    else if (NX <= 2 || groups == 2)
      k_loop(std::integral_constant<int, 2>{}, once);
    else if constexpr (NX > 2) {
      if (groups == 3)
        k_loop(std::integral_constant<int, 3>{}, once);
      else
        k_loop(std::integral_constant<int, 4>{}, once);
    }
  };
  if (nsteps > 0) {
    if (a.stream_once && last - first <= C::kT)
      dispatch(std::true_type{});
    else
      dispatch(std::false_type{});
  }

  // Lane (lr, kq) holds features 4 kq .. 4 kq + 3 of each weight block for
  // token lr of each token block.
#pragma unroll
  for (int j = 0; j < NX; ++j) {
    const int prow = row0 + (2 * j + wave_t) * 16 + lr;
    if (prow >= row_end) continue;
    if constexpr (kGateUp) {
#pragma unroll
      for (int i = 0; i < NI / 2; ++i) {
        const int f = wtile * (C::kW / 2) + w_row(i) + 4 * kq;
        if (f >= a.I) continue;
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float g = acc[i][j][r], u = acc[i + NI / 2][j][r];
          v[r] = (C::kFastAct ? gate_act_fast(a.act, g) : gate_act(a.act, g)) * u;
        }
        store4<T>(static_cast<T*>(a.out) + static_cast<size_t>(prow) * a.I + f, v[0], v[1], v[2],
                  v[3]);
      }
    } else {
      const size_t row = (static_cast<size_t>(split) * a.R + prow) * a.H;
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int f = wtile * C::kW + w_row(i) + 4 * kq;
        if (f >= a.H) continue;
        const f32x4 v = acc[i][j];
        if (a.y16)
          store4<T>(static_cast<T*>(a.out) + row + f, v[0], v[1], v[2], v[3]);
        else
          store4<float>(static_cast<float*>(a.out) + row + f, v[0], v[1], v[2], v[3]);
      }
    }
  }
}

// Tiles measured at the layers above (us): fp32 64 x 64 one step deep 205 at 512
// tokens, two steps deep 211, 128 x 64 two deep 263; bf16 128 x 64 two steps deep
// 129-131, 64 x 64 145-148, and with weights loaded past L2 206 (rows there
// do not start on 128-byte lines, so every line serves two steps). Mixtral shape
// on 128-row maps, 100 and 197 tokens: 128 x 128 two deep 467 and 488, one deep
// 484 and 525, 64 x 128 one deep 476 and 544, 256 x 64 (64-row maps) 500 and 507.
typedef Config<64, 64, 1> ConfigF32;
typedef Config<128, 64, 2> Config16;
typedef Config<128, 128, 2, true> ConfigMid;

template <typename T, bool kGateUp, typename C>
hipError_t launch_items(FfnArgs a, hipStream_t s) {
  a.n_wtiles = kGateUp ? (a.I + C::kW / 2 - 1) / (C::kW / 2) : (a.H + C::kW - 1) / C::kW;
  const long long items = static_cast<long long>(a.n_wtiles) * a.max_tiles * a.splits;
  if (items == 0) return hipSuccess;
  if (items > INT_MAX - kGridX || a.tile_rows > C::kT) return hipErrorInvalidValue;
  const dim3 grid(static_cast<unsigned>(std::min<long long>(items, kGridX)),
                  static_cast<unsigned>((items + kGridX - 1) / kGridX));
  ffn_general_kernel<T, kGateUp, C><<<grid, dim3(kThreads), 0, s>>>(a);
  return hipGetLastError();
}

template <bool kGateUp>
hipError_t launch_general(const FfnArgs& a, int dtype, hipStream_t s) {
  if (a.tile_rows == 128 && dtype != MOE355_F32)
    return dtype == MOE355_BF16 ? launch_items<bf16, kGateUp, ConfigMid>(a, s)
                                : launch_items<f16, kGateUp, ConfigMid>(a, s);
  if (dtype == MOE355_BF16) return launch_items<bf16, kGateUp, Config16>(a, s);
  if (dtype == MOE355_F16) return launch_items<f16, kGateUp, Config16>(a, s);
  return launch_items<float, kGateUp, ConfigF32>(a, s);
}

}  // namespace

hipError_t launch_gate_up_general(const FfnArgs& a, int dtype, hipStream_t s) {
  return launch_general<true>(a, dtype, s);
}

hipError_t launch_down_general(const FfnArgs& a, int dtype, hipStream_t s) {
  return launch_general<false>(a, dtype, s);
}

}  // namespace moe355
