// GRPO group-normalised advantages.
//
// One wave per sample.  A sample's group is every row whose prompt key equals
// its own (exact row equality, as torch.unique(prompts, dim=0) groups them).
// Lane l takes the samples j = l (mod 64): it loads their keys, adds its own
// matches up in double, and a butterfly joins the lanes, so the result depends
// on the grouping alone and not on how the keys were compared.  Group sums are
// rounded once to fp32, where the reference uses an fp32 matrix-vector product;
// the two agree to the last fp32 ulp of the sum.
//
// How keys are compared:
// * single-element keys (group ids): directly, 64 a load;
// * longer keys (prompt token rows) with a workspace: each row is hashed once
//   (adv_hash_kernel), each sample finds the first row of its hash and compares
//   itself with that one row in full (adv_leader_kernel), and the row's index
//   is the group id that the sums are formed over: B K reads instead of one row
//   comparison per pair, which prompts that share their first tokens (a chat
//   template) all reach.  Rows that only share a hash stay apart: the comparison
//   decides, the hash selects.
// * longer keys without a workspace: the first elements 64 at a time, rows that
//   agree there in full by the whole wave.
//
// Semantics: nemo_rl/algorithms/utils.py:118-234
// (calculate_baseline_and_std_per_prompt) and
// nemo_rl/algorithms/advantage_estimator.py:106-145
// (GRPOAdvantageEstimator.compute_advantage).

#include <cfloat>

#include "common.h"

namespace mirl {
namespace {

struct AdvArgs {
  const int64_t* prompts;
  int64_t B, K, ps;
  const float* rewards;
  const float* srew;
  const float* valid;
  int loo, normalize;
  float* adv;
  float* baseline_out;
  float* std_out;
  uint8_t* trivial_out;
};

__device__ __forceinline__ float wave_min(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fminf(v, __shfl_xor(v, off, kWave));
  return v;
}

// Key loads in flight per lane: the scans are chains of L2 round trips (2048 prompt
// rows of 512 tokens, three launches: 26 us with one load a trip, 20 us with four).
constexpr int kAdvUnroll = 4;

// The advantage of sample i, formed by one whole wave; bit u of match(j0) is the
// lane's answer to whether sample j0 + 64 u + lane is in i's group (0 from B on).
template <class Match>
__device__ __forceinline__ void sample_advantage(const AdvArgs& A, int64_t i, int lane, Match&& match) {
  const float* __restrict__ rewards = A.rewards;
  const float* __restrict__ srew = A.srew;
  const float* __restrict__ valid = A.valid;
  const int loo = A.loo, normalize = A.normalize;
  double nd = 0.0, srv = 0.0, sqv = 0.0, sq2v = 0.0;
  float cmin = INFINITY, cmax = -INFINITY;
  for (int64_t j0 = 0; j0 < A.B; j0 += kAdvUnroll * kWave) {
    for (unsigned m = match(j0); m != 0; m &= m - 1) {
      const int64_t j = j0 + (__ffs((int)m) - 1) * kWave + lane;
      const float vj = valid ? valid[j] : 1.f;
      const float rj = rewards[j];
      const float qj = srew ? srew[j] : rj;
      nd += (double)vj;
      if (!(loo && j == i)) {
        srv += (double)(rj * vj);
        sqv += (double)(qj * vj);
        sq2v += (double)((qj * qj) * vj);
        if (vj != 0.f) {
          cmin = fminf(cmin, qj);
          cmax = fmaxf(cmax, qj);
        }
      }
    }
  }
  const float n = (float)wave_sum(nd);
  srv = wave_sum(srv);
  sqv = wave_sum(sqv);
  sq2v = wave_sum(sq2v);
  cmin = wave_min(cmin);
  cmax = wave_max(cmax);
  if (lane != 0) return;
  const float ri = rewards[i];
  float base, sd = 0.f;
  bool trivial = true;
  if (n <= 1.f) {
    base = ri;
  } else {
    const float nv = n - (loo ? 1.f : 0.f);
    base = (float)srv / nv;
    const float qbar = srew ? (float)sqv / nv : base;
    const float sq = (float)sq2v / nv;
    trivial = (cmin == cmax);
    sd = sqrtf((sq - qbar * qbar) * (nv / (nv - 1.f)));
    if (isnan(sd)) sd = 0.f;
    else if (isinf(sd)) sd = sd > 0.f ? FLT_MAX : -FLT_MAX;
  }
  float a = ri - base;
  if (normalize && sd > 0.f && !trivial) a = a / (sd + 1e-6f);
  A.adv[i] = a;
  if (A.baseline_out) A.baseline_out[i] = base;
  if (A.std_out) A.std_out[i] = sd;
  if (A.trivial_out) A.trivial_out[i] = trivial ? 1 : 0;
}

constexpr int kAdvWaves = 4;  // samples (waves) per workgroup of 256 threads

__device__ __forceinline__ int64_t wave_sample() {
  return (int64_t)blockIdx.x * kAdvWaves + threadIdx.x / kWave;
}

// Bit u: j + 64 u < end and its key equals `mine` (a load past the end reads the
// last key).
template <class T, class Load>
__device__ __forceinline__ unsigned equal_keys(int64_t j, int64_t end, T mine, Load&& load) {
  T k[kAdvUnroll];
#pragma unroll
  for (int u = 0; u < kAdvUnroll; ++u) {
    const int64_t ju = j + u * kWave;
    k[u] = load(ju < end ? ju : end - 1);
  }
  unsigned m = 0;
#pragma unroll
  for (int u = 0; u < kAdvUnroll; ++u) m |= (unsigned)(j + u * kWave < end && k[u] == mine) << u;
  return m;
}

// Rows a and b of K elements equal?  Every lane of the wave gets the answer.
__device__ __forceinline__ bool rows_equal(const int64_t* a, const int64_t* b, int64_t K, int lane) {
  uint64_t diff = 0;
#pragma unroll 4
  for (int64_t k = lane; k < K; k += kWave) diff |= (uint64_t)(a[k] ^ b[k]);
  return __ballot(diff != 0) == 0ull;
}

// Scalar keys (T = int64_t: group ids of stride `stride`; int32_t: the leaders).
// Bound by latency up to a few thousand samples (B / 64 coalesced key loads per
// wave, all of them cache hits), then by the B^2 keys read: 7 us for 1024 ids (one
// thread per sample walking all keys: 142), 36 us for 8192 (1087; in one group of
// 8192, 89 and 2215).
template <class T>
__global__ __launch_bounds__(256) void adv_scalar_kernel(AdvArgs A, const T* __restrict__ keys,
                                                         int64_t stride) {
  const int64_t i = wave_sample();
  if (i >= A.B) return;  // whole waves leave together
  const int lane = threadIdx.x % kWave;
  const T mine = keys[i * stride];
  sample_advantage(A, i, lane, [&](int64_t j0) {
    return equal_keys(j0 + lane, A.B, mine, [&](int64_t j) { return keys[j * stride]; });
  });
}

// Prompt rows compared directly (no workspace).  Each row that agrees in its first
// element costs a dependent round trip per 64 x 4 elements: 7 us for 8 rows of 512
// tokens, 11 us for 16, 20 us for 32, 57 us for 16 of 4096, against 13-16 us for the three
// hashed launches.
__global__ __launch_bounds__(256) void adv_rows_kernel(AdvArgs A) {
  const int64_t i = wave_sample();
  if (i >= A.B) return;
  const int lane = threadIdx.x % kWave;
  const int64_t* pi = A.prompts + i * A.ps;
  const int64_t p0 = pi[0];
  sample_advantage(A, i, lane, [&](int64_t j0) {
    const unsigned first =
        equal_keys(j0 + lane, A.B, p0, [&](int64_t j) { return A.prompts[j * A.ps]; });
    unsigned mine = 0;
#pragma unroll 1
    for (int u = 0; u < kAdvUnroll; ++u) {
      uint64_t cand = __ballot((first >> u) & 1u);
      while (cand != 0) {
        const int b = __ffsll((unsigned long long)cand) - 1;
        cand &= cand - 1;
        const int64_t j = j0 + u * kWave + b;
        if ((j == i || rows_equal(pi, A.prompts + j * A.ps, A.K, lane)) && lane == b) mine |= 1u << u;
      }
    }
    return mine;
  });
}

// hash[i] of row i: the sum over k of element k mixed with its position (the
// finaliser of Steele, Lea and Flood, "Fast splittable pseudorandom number
// generators", 2014).  One workgroup of NT threads per row, so that a row's loads
// are in flight together.  It reads the B K keys once (8.4 MB in 4-9 us); hash,
// leaders and sums together: 2048 rows of 512 tokens that share their first token
// 4481 -> 20 us, 8192 rows 29.1 ms -> 82 us, 512 rows of 1024 1069 -> 16 us.
template <int NT>
__global__ __launch_bounds__(NT) void adv_hash_kernel(const int64_t* __restrict__ prompts, int64_t K,
                                                      int64_t ps, uint64_t* __restrict__ hash) {
  const int64_t* p = prompts + (int64_t)blockIdx.x * ps;
  uint64_t h = 0;
#pragma unroll 4
  for (int64_t k = threadIdx.x; k < K; k += NT) {
    uint64_t z = (uint64_t)p[k] + (uint64_t)(k + 1) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    h += z ^ (z >> 31);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) h += __shfl_xor((unsigned long long)h, off, kWave);
  if constexpr (NT > kWave) {
    __shared__ uint64_t part[NT / kWave];
    if (threadIdx.x % kWave == 0) part[threadIdx.x / kWave] = h;
    __syncthreads();
    h = 0;
    for (int w = 0; w < NT / kWave; ++w) h += part[w];
  }
  if (threadIdx.x == 0) hash[blockIdx.x] = h;
}

// leader[i] = the first row equal to row i: among the rows of its hash, in
// ascending order, the first that a full comparison confirms (row i itself at
// the latest).
__global__ __launch_bounds__(256) void adv_leader_kernel(const int64_t* __restrict__ prompts, int64_t B,
                                                         int64_t K, int64_t ps,
                                                         const uint64_t* __restrict__ hash,
                                                         int32_t* __restrict__ leader) {
  const int64_t i = wave_sample();
  if (i >= B) return;
  const int lane = threadIdx.x % kWave;
  const uint64_t mine = hash[i];
  int64_t found = i;
  for (int64_t j0 = 0; j0 < i && found == i; j0 += kAdvUnroll * kWave) {
    const unsigned same = equal_keys(j0 + lane, i, mine, [&](int64_t j) { return hash[j]; });
    for (int u = 0; u < kAdvUnroll && found == i; ++u) {
      uint64_t cand = __ballot((same >> u) & 1u);
      while (cand != 0) {
        const int64_t c = j0 + u * kWave + __ffsll((unsigned long long)cand) - 1;
        cand &= cand - 1;
        if (rows_equal(prompts + i * ps, prompts + c * ps, K, lane)) {
          found = c;
          break;
        }
      }
    }
  }
  if (lane == 0) leader[i] = (int32_t)found;
}

}  // namespace
}  // namespace mirl

using namespace mirl;

extern "C" int64_t mirl_grpo_advantage_workspace_bytes(int64_t B, int64_t K) {
  // a 64-bit hash and a 32-bit leader per sample; group ids need neither
  return (B > 0 && K > 1) ? B * 12 : 0;
}

static int grpo_advantage(const int64_t* prompts, int64_t B, int64_t K, int64_t prompt_stride,
                          const float* rewards, const float* std_rewards, const float* valid_mask,
                          int leave_one_out, int normalize, float* adv, float* baseline, float* std,
                          uint8_t* trivial, void* workspace, const char* what, void* stream) {
  MIRL_REQUIRE(B >= 0 && K > 0, "invalid shape B=%lld K=%lld", (long long)B, (long long)K);
  if (B == 0) return MIRL_OK;
  MIRL_REQUIRE(prompts && rewards && adv, "null pointer argument");
  AdvArgs a{prompts, B, K, prompt_stride, rewards, std_rewards, valid_mask, leave_one_out, normalize,
            adv, baseline, std, trivial};
  hipStream_t st = static_cast<hipStream_t>(stream);
  const unsigned blocks = (unsigned)((B + kAdvWaves - 1) / kAdvWaves);
  if (K == 1) {
    hipLaunchKernelGGL(adv_scalar_kernel<int64_t>, dim3(blocks), dim3(256), 0, st, a, prompts,
                       prompt_stride);
  } else if (workspace != nullptr) {
    MIRL_REQUIRE(B < (int64_t(1) << 31), "too many samples (%lld)", (long long)B);
    MIRL_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 7u) == 0, "the workspace must be 8-byte aligned");
    uint64_t* hash = static_cast<uint64_t*>(workspace);
    int32_t* leader = reinterpret_cast<int32_t*>(hash + B);
    if (K <= 4 * kWave)
      hipLaunchKernelGGL(adv_hash_kernel<64>, dim3((unsigned)B), dim3(64), 0, st, prompts, K,
                         prompt_stride, hash);
    else
      hipLaunchKernelGGL(adv_hash_kernel<256>, dim3((unsigned)B), dim3(256), 0, st, prompts, K,
                         prompt_stride, hash);
    hipLaunchKernelGGL(adv_leader_kernel, dim3(blocks), dim3(256), 0, st, prompts, B, K, prompt_stride,
                       hash, leader);
    hipLaunchKernelGGL(adv_scalar_kernel<int32_t>, dim3(blocks), dim3(256), 0, st, a, leader, (int64_t)1);
  } else {
    hipLaunchKernelGGL(adv_rows_kernel, dim3(blocks), dim3(256), 0, st, a);
  }
  return check_launch(what);
}

extern "C" int mirl_grpo_advantage(const int64_t* prompts, int64_t B, int64_t K,
                                   int64_t prompt_stride, const float* rewards,
                                   const float* std_rewards, const float* valid_mask,
                                   int leave_one_out, int normalize,
                                   float* adv, float* baseline, float* std, uint8_t* trivial,
                                   void* stream) {
  clear_error();
  return grpo_advantage(prompts, B, K, prompt_stride, rewards, std_rewards, valid_mask, leave_one_out,
                        normalize, adv, baseline, std, trivial, nullptr, "mirl_grpo_advantage", stream);
}

extern "C" int mirl_grpo_advantage_ws(const int64_t* prompts, int64_t B, int64_t K,
                                      int64_t prompt_stride, const float* rewards,
                                      const float* std_rewards, const float* valid_mask,
                                      int leave_one_out, int normalize, float* adv, float* baseline,
                                      float* std, uint8_t* trivial, void* workspace, void* stream) {
  clear_error();
  MIRL_REQUIRE(workspace != nullptr || mirl_grpo_advantage_workspace_bytes(B, K) == 0, "null workspace");
  return grpo_advantage(prompts, B, K, prompt_stride, rewards, std_rewards, valid_mask, leave_one_out,
                        normalize, adv, baseline, std, trivial, workspace, "mirl_grpo_advantage_ws", stream);
}
