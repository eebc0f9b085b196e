// Wave-level softmax + top-k and a transposed wave reduction, shared by the
// router kernels (router.hip) and the fused residual add + RMSNorm + router
// kernel (norm.hip). Included inside their anonymous namespaces.
#pragma once

constexpr int kMaxPerLane = kMaxExperts / kWave;

// v of the lane that the DPP control names (lanes without a source keep their
// own), a few cycles against a shuffle's round trip through the LDS unit.
template <int kCtrl, int kRowMask = 0xf>
__device__ __forceinline__ float dpp(float v) {
  const int x = __float_as_int(v);
  return __int_as_float(__builtin_amdgcn_update_dpp(x, x, kCtrl, kRowMask, 0xf, false));
}

// Maximum over the wave (NaN ignored), the same in every lane.
__device__ __forceinline__ float wave_max_dpp(float v) {
  v = fmaxf(v, dpp<0x111>(v));       // row_shr 1, 2, 4, 8: lane 15 of each row of
  v = fmaxf(v, dpp<0x112>(v));       // 16 lanes holds the row's maximum
  v = fmaxf(v, dpp<0x114>(v));
  v = fmaxf(v, dpp<0x118>(v));
  v = fmaxf(v, dpp<0x142, 0xa>(v));  // row_bcast 15 into rows 1 and 3
  v = fmaxf(v, dpp<0x143, 0xc>(v));  // row_bcast 31 into rows 2 and 3
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), kWave - 1));
}

// Maximum over each row of 16 lanes (NaN ignored), in every lane of it.
__device__ __forceinline__ float row_max_dpp(float v) {
  v = fmaxf(v, dpp<0x121>(v));  // row_ror 1, 2, 4, 8
  v = fmaxf(v, dpp<0x122>(v));
  v = fmaxf(v, dpp<0x124>(v));
  return fmaxf(v, dpp<0x128>(v));
}

// Softmax + top-k + renormalisation of one token's logits by one wave.
// lg: E fp32 logits (LDS or global). Mirrors torch_fused_topk (fused.py:42-45)
// and, when kmin > 0, the entropy-adaptive branch of FusedMoE.route
// (moe_layer.py:326-342).
// One wave runs this as a serial chain, so its latency counts: each of the K
// selections is a DPP maximum and one ballot per 64 experts (the lowest lane
// that holds it is the lowest id), selection k stays in lane k, and the lanes
// finish and store their own. Against shuffle butterflies over (value, id) pairs
// with lane 0 finishing through LDS, whole kernels: top-6 of 64 for 8 tokens
// 7.2 -> 4.7 us, router of 8 experts top-2 for one token 6.3 -> 5.1 us, MFMA
// router of 64 experts top-6 for 4096 tokens (group16_topk) 18.6 -> 16.1 us.
__device__ void wave_topk(const float* lg, int E, int K, int renorm, int kmin, float* w_out,
                          int32_t* id_out, int lane) {
  float v[kMaxPerLane];
  bool live[kMaxPerLane];
#pragma unroll
  for (int j = 0; j < kMaxPerLane; ++j) {
    const int e = lane + kWave * j;
    live[j] = e < E;
    v[j] = live[j] ? lg[e] : -INFINITY;
  }
  float m = -INFINITY;
#pragma unroll
  for (int j = 0; j < kMaxPerLane; ++j)
    if (live[j]) m = fmaxf(m, v[j]);
  m = wave_max_dpp(m);
  float s = 0.f;
#pragma unroll
  for (int j = 0; j < kMaxPerLane; ++j)
    if (live[j]) s += expf(v[j] - m);
  s = wave_sum(s);

  // Shannon entropy of the softmax, only for the entropy-adaptive branch.
  float hs = 0.f;
  if (kmin > 0) {
#pragma unroll
    for (int j = 0; j < kMaxPerLane; ++j) {
      if (live[j]) {
        const float p = expf(v[j] - m) / s;
        hs += p * logf(fmaxf(p, 1e-9f));
      }
    }
    hs = -wave_sum(hs);
  }

  // Selection k: lane k % 64, register k / 64.
  float sel[kMaxPerLane];
  int id[kMaxPerLane];
#pragma unroll
  for (int j = 0; j < kMaxPerLane; ++j) {
    sel[j] = -INFINITY;
    id[j] = INT_MAX;
  }
  for (int k = 0; k < K; ++k) {
    float bv = -INFINITY;
#pragma unroll
    for (int j = 0; j < kMaxPerLane; ++j)
      if (live[j]) bv = fmaxf(bv, v[j]);
    bv = wave_max_dpp(bv);
    int bi = INT_MAX;  // stays so when only NaN logits are left
#pragma unroll
    for (int j = kMaxPerLane - 1; j >= 0; --j) {
      if (kWave * j >= E) continue;
      const unsigned long long at = __ballot(live[j] && v[j] == bv);
      if (at) bi = kWave * j + __builtin_ctzll(at);
    }
#pragma unroll
    for (int j = 0; j < kMaxPerLane; ++j) {
      if (lane + kWave * j == bi) live[j] = false;
      if (lane + kWave * j == k) {
        sel[j] = bv;
        id[j] = bi;
      }
    }
  }

  int kd = K;
  if (kmin > 0) {
    const float hn = E > 1 ? hs / logf(static_cast<float>(E)) : 0.f;
    const float kf = rintf(static_cast<float>(kmin) + static_cast<float>(K - kmin) * hn);
    kd = static_cast<int>(fminf(fmaxf(kf, static_cast<float>(kmin)), static_cast<float>(K)));
  }
  float w[kMaxPerLane];
#pragma unroll
  for (int j = 0; j < kMaxPerLane; ++j)
    w[j] = lane + kWave * j < kd ? expf(sel[j] - m) / s : 0.f;
  float sum = 0.f;  // in ascending k
#pragma unroll
  for (int j = 0; j < kMaxPerLane; ++j)
    for (int k = kWave * j; k < min(K, kWave * (j + 1)); ++k)
      sum += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w[j]), k - kWave * j));
  const bool norm = kmin > 0 || renorm;
  const float denom = kmin > 0 ? fmaxf(sum, 1e-9f) : sum;
#pragma unroll
  for (int j = 0; j < kMaxPerLane; ++j) {
    const int k = lane + kWave * j;
    if (k < K) {
      w_out[k] = norm ? w[j] / denom : w[j];
      id_out[k] = id[j];
    }
  }
}

// Wave-wide sum of V values per lane in log2(64) shuffle rounds, returning
// one total per lane: while more than one value is left, each round sends
// half of the lane's values to its partner and keeps the other half, so the V
// sums finish after 63 shuffles in total instead of 6*V. Lane l ends up with
// the sum of value index l >> (6 - log2 V).
template <int V>
__device__ __forceinline__ float transpose_reduce(float (&v)[V], int lane) {
#pragma unroll
  for (int r = 0; r < 6; ++r) {
    const int d = 32 >> r;
    const int n = (V >> r) > 1 ? (V >> r) : 1;
    if (n > 1) {
      // Bitwise select on the values: a lane-dependent `up ? v[i] : v[j]`
      // can be folded into a per-lane array index, which sends the whole
      // array to scratch memory.
      const uint32_t m = (lane & d) != 0 ? 0xffffffffu : 0u;
#pragma unroll
      for (int i = 0; i < n / 2; ++i) {
        const uint32_t lo = __float_as_uint(v[i]), hi = __float_as_uint(v[i + n / 2]);
        const float send = __uint_as_float((lo & m) | (hi & ~m));
        const float keep = __uint_as_float((hi & m) | (lo & ~m));
        v[i] = keep + __shfl_xor(send, d, kWave);
      }
    } else {
      v[0] += __shfl_xor(v[0], d, kWave);
    }
  }
  return v[0];
}

constexpr int log2i(int v) { return v <= 1 ? 0 : 1 + log2i(v / 2); }

// Softmax + top-k + renormalisation of one token by a 16-lane group (the
// lanes l .. l + 15 of one wave, sub = l % 16): lane sub holds experts
// sub + 16 j, j < NV. Selection as wave_topk (value, then lower id on exact
// ties), each maximum a DPP rotation inside the group. Lane sub == 0 writes the
// results. K <= 8. The groups of a wave may differ in activity, not the lanes of
// one group.
template <int NV>
__device__ void group16_topk(const float* lg, int E, int K, int renorm, int kmin, float* w_out,
                             int32_t* id_out, int sub) {
  const int row0 = threadIdx.x & (kWave - 16);  // first lane of the group
  float v[NV];
  bool live[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int e = sub + 16 * j;
    live[j] = e < E;
    v[j] = live[j] ? lg[e] : -INFINITY;
  }
  float m = -INFINITY;
#pragma unroll
  for (int j = 0; j < NV; ++j)
    if (live[j]) m = fmaxf(m, v[j]);
  m = row_max_dpp(m);
  float s = 0.f;
#pragma unroll
  for (int j = 0; j < NV; ++j)
    if (live[j]) s += expf(v[j] - m);
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) s += __shfl_xor(s, o, 16);
  float hs = 0.f;
  if (kmin > 0) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      if (live[j]) {
        const float p = expf(v[j] - m) / s;
        hs += p * logf(fmaxf(p, 1e-9f));
      }
    }
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) hs += __shfl_xor(hs, o, 16);
    hs = -hs;
  }
  float psel[8];
  int isel[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    psel[k] = 0.f;
    isel[k] = 0;
    if (k >= K) continue;
    float bv = -INFINITY;
#pragma unroll
    for (int j = 0; j < NV; ++j)
      if (live[j]) bv = fmaxf(bv, v[j]);
    bv = row_max_dpp(bv);
    int bi = INT_MAX;  // stays so when only NaN logits are left
#pragma unroll
    for (int j = NV - 1; j >= 0; --j) {
      const unsigned at = static_cast<unsigned>(__ballot(live[j] && v[j] == bv) >> row0) & 0xffffu;
      if (at) bi = 16 * j + __builtin_ctz(at);
    }
#pragma unroll
    for (int j = 0; j < NV; ++j)
      if (sub + 16 * j == bi) live[j] = false;
    psel[k] = expf(bv - m) / s;
    isel[k] = bi;
  }
  if (sub != 0) return;
  int kd = K;
  if (kmin > 0) {
    const float hn = E > 1 ? hs / logf(static_cast<float>(E)) : 0.f;
    const float kf = rintf(static_cast<float>(kmin) + static_cast<float>(K - kmin) * hn);
    kd = static_cast<int>(fminf(fmaxf(kf, static_cast<float>(kmin)), static_cast<float>(K)));
  }
  float sum = 0.f;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    if (k < K) {
      psel[k] = k < kd ? psel[k] : 0.f;
      sum += psel[k];
    }
  }
  const bool norm = kmin > 0 || renorm;
  const float denom = kmin > 0 ? fmaxf(sum, 1e-9f) : sum;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    if (k < K) {
      w_out[k] = norm ? psel[k] / denom : psel[k];
      id_out[k] = isel[k];
    }
  }
}
