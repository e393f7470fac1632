// policy.hip — one rollout step of the policy (and optionally the value) in
// one launch: GpuPolicy::forward (src/biped/gpu_policy.rs:210-248) with the
// trainer's sampling (src/bin/biped_train_gpu.rs:910-930). At a rollout's
// few thousand rows the per-layer GEMM launches are latency-bound; here a
// block takes kPolicyRows rows through every layer with the activations in
// LDS, reading each layer's weights from L2 in the fragment-major copy that
// zk_policy_pack writes (a wavefront's load of one tile's 16-wide chunk is
// 1 KB of consecutive floats instead of 64 bytes of each of 16 weight rows).
//
// Every value is computed as on the multi-launch path: the normalisation is
// Normalizer::normalize's expression (ppo.rs:198-205), each layer sums its
// reduction index in 16-wide chunks with lane group s of MFMA step c on
// index k0 + 4 s + c (the order of the tiled and narrow fp32 GEMM kernels), adds
// the bias after the sum and applies ELU to the hidden layers, and the
// log-probability adds its terms in component order. Layer launches on fp32
// kernels (chunks of up to 2,048 rows) give the same bits; those that take the
// three-piece kernels agree to rounding.
#pragma once
#include "common.hip"

namespace zk {

constexpr int kPolicyPitch = kPolicyMaxWidth + 4;  // LDS row pitch of an activation tile
constexpr int kPolicyWaves = kPolicyThreads / 64;
constexpr int kPolicyMaxTiles = kPolicyMaxWidth / 16 / kPolicyWaves;  // 16-column tiles per wave
// float4 weight chunks a wavefront keeps in flight: one tile takes them as a
// ring of four chunks, two tiles as rings of two, within the 64 VGPRs of two
// blocks per CU. Eight (98 VGPRs, one block per CU) measured no faster: 23.7 vs
// 22.9 us per step at 64 rows, 45.8 vs 40.7 at 4,096.
constexpr int kPolicyDepth = 4;
static_assert(kPolicyRows == 16 && kPolicyWaves == kPolicyRows && kPolicyThreads >= 32 * kPolicyRows,
              "one 16-row MFMA tile; a wavefront per input row; a 32-lane group per row");
static_assert(kPolicyMaxTiles <= 2, "one or two tiles per wavefront");

// This lane's float4 of a tile's chunk c: 32-bit byte offsets from the uniform
// base, one register per address.
__device__ __forceinline__ float4 policy_chunk(const float* Wp, unsigned w, int c) {
  return *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(Wp) + (w + 1024u * c));
}

// A wavefront's nu tiles of one layer, src [16 x 16 kc] in LDS times the packed
// chunks at w[u] (bytes from Wp). Issue the first chunks of its tiles, which stay in
// flight over the code between the layers ...
__device__ __forceinline__ void policy_prime(float4 (&ring)[kPolicyDepth], const float* Wp, const unsigned (&w)[2], int nu,
                                             int kc) {
#pragma unroll
  for (int i = 0; i < kPolicyDepth; ++i) {
    const int j = nu == 2 ? i / 2 : i;
    ring[i] = policy_chunk(Wp, nu == 2 ? w[i & 1] : w[0], min(j, kc - 1));
  }
}

// ... then multiply chunk by chunk, each slot refilled D chunks ahead as soon as
// it is read (past the end: the last chunk again, never used).
template <int TU>
__device__ __forceinline__ void policy_sum(floatx4 (&acc)[2], float4 (&ring)[kPolicyDepth], const float* Wp,
                                           const unsigned (&w)[2], int kc, const float* src) {
  constexpr int D = kPolicyDepth / TU;
  auto step = [&](int c, int j) {
    const float4 a = *reinterpret_cast<const float4*>(src + 16 * c);
#pragma unroll
    for (int u = 0; u < TU; ++u) {
      const float4 b = ring[j * TU + u];
      acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, acc[u], 0, 0, 0);
      acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, acc[u], 0, 0, 0);
      acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, acc[u], 0, 0, 0);
      acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, acc[u], 0, 0, 0);
    }
  };
  int c0 = 0;
  for (; c0 + D < kc; c0 += D) {
#pragma unroll
    for (int j = 0; j < D; ++j) {
      step(c0 + j, j);
      const int c = min(c0 + j + D, kc - 1);
#pragma unroll
      for (int u = 0; u < TU; ++u) ring[j * TU + u] = policy_chunk(Wp, w[u], c);
      __builtin_amdgcn_sched_barrier(0);  // else all refills move behind the last product
    }
  }
#pragma unroll
  for (int j = 0; j < D; ++j)
    if (c0 + j < kc) step(c0 + j, j);
}

// What bounds it: up to a few hundred rows a block is alone on its CU and its
// 0.93 MB of weights (headline actor) arrive one dependent round of loads
// after another; the fp32 MFMAs alone take 12 us, and 24 us at 4,096 rows (two
// blocks per CU). The loads therefore run as a ring that is refilled slot by
// slot, a layer's first chunks and its bias are on their way over the barrier of
// the layer before (issued before that layer's epilogue they cost four spilled
// registers: with the loads of idle wavefronts 4,096 rows of 48-128-128-8 nets 13.4 us,
// now 11.5), and the input rows and log_std travel with the normaliser's
// statistics. A step of both headline nets: 28.3 -> 22.0 us at 64 rows, 51 -> 38.3 us
// at 4,096.
__device__ void policy_body(const PolicyArgs& p) {
  __shared__ __align__(16) float act[2][kPolicyRows * kPolicyPitch];
  __shared__ float s_mu[kPolicyMaxWidth], s_sd[kPolicyMaxWidth];
  __shared__ float s_term[kPolicyThreads];
  __shared__ float s_ls[32], s_sdv[32];
  const PolicyNet& q = p.net[blockIdx.y];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const long long r0 = (long long)blockIdx.x * kPolicyRows;
  const int nr = (int)min((long long)kPolicyRows, p.rows - r0);
  const int od = q.dims[0];
  const int k0w = (od + 15) & ~15;  // layer 0's reduction width (zero past od)

  // This wave's 16-column tiles of a layer: slots wave, wave + kPolicyWaves < nt,
  // slot s on tile (s + rot) % nt, rotated per block so that concurrent
  // blocks read different weight tiles (measured within 1 % of no rotation).
  float4 ring[kPolicyDepth];
  int tile[2];
  unsigned woff[2];
  float bias[2];
  int nu = 0;
  auto begin_layer = [&](int l) {
    const int nt = (q.dims[l + 1] + 15) / 16;
    const int kc = (l == 0 ? k0w : q.dims[l]) / 16;
    const int rot = (int)(blockIdx.x % (unsigned)nt);
    nu = wave + kPolicyWaves < nt ? 2 : wave < nt ? 1 : 0;  // uniform over the wavefront
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int s = wave + kPolicyWaves * u + rot;
      tile[u] = u >= nu ? 0 : s >= nt ? s - nt : s;
      woff[u] = 4u * (tile[u] * kc * 256 + 4 * lane);
    }
    // The biases first: the ring's own order of arrival then stays exact.
    const float* bl = p.params + q.b_off[l];
#pragma unroll
    for (int u = 0; u < 2; ++u) bias[u] = bl[(unsigned)min(16 * tile[u] + lr, q.dims[l + 1] - 1)];
    const float* Wp = q.wp + q.wp_off[l];
    if (nu > 0) policy_prime(ring, Wp, woff, nu, kc);
  };
  begin_layer(0);
  const bool sampling = blockIdx.y == 0 && p.sample;

  // Inputs, a row per wavefront: rows past nr and columns in [od, k0w) are zero.
  // The row's loads go out before the wait for the normaliser's statistics.
  constexpr int kIn = kPolicyMaxWidth / 64;
  float xin[kIn];
#pragma unroll
  for (int i = 0; i < kIn; ++i) {
    const int c = lane + 64 * i;
    xin[i] = wave < nr && c < od ? q.x[(r0 + wave) * q.ldx + c] : 0.f;
  }
  if (sampling && t < p.A) {
    s_ls[t] = p.log_std[t];
    s_sdv[t] = expf(s_ls[t]);
  }
  if (q.norm) {
    const float count = q.norm[2 * od];
    for (int c = t; c < od; c += kPolicyThreads) {
      s_mu[c] = q.norm[c];
      s_sd[c] = sqrtf(fmaxf(q.norm[od + c] / count, 1e-8f));
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < kIn; ++i) {
    const int c = lane + 64 * i;
    if (c >= k0w) break;
    float v = xin[i];
    if (q.norm && wave < nr && c < od) v = clampf((v - s_mu[c]) / s_sd[c], -5.0f, 5.0f);
    act[0][wave * kPolicyPitch + c] = v;
  }
  __syncthreads();

  int cur = 0;
  for (int l = 0; l < q.L; ++l) {
    const int kc = (l == 0 ? k0w : q.dims[l]) / 16;
    const int N = q.dims[l + 1];
    const bool last = l == q.L - 1;
    const float* Wp = q.wp + q.wp_off[l];
    const float* src = act[cur] + lr * kPolicyPitch + 4 * lg;
    float* dst = act[cur ^ 1];
    floatx4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    if (nu == 2)
      policy_sum<2>(acc, ring, Wp, woff, kc, src);
    else if (nu == 1)
      policy_sum<1>(acc, ring, Wp, woff, kc, src);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int n = 16 * tile[u] + lr;
      if (u >= nu || n >= N) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 4 * lg + r;
        const float v = last ? acc[u][r] + bias[u] : elu(acc[u][r] + bias[u]);
        dst[row * kPolicyPitch + n] = v;
        if (last && q.out && row < nr) q.out[(r0 + row) * q.ldo + n] = v;
      }
    }
    if (!last) begin_layer(l + 1);  // its first weights travel over the barrier
    __syncthreads();
    cur ^= 1;
  }

  // Sampling (as zk_sample_g32): a 32-lane group per row, lane k on component
  // k; the row's logp terms added in component order by its first lane.
  if (!sampling) return;
  const int A = p.A;
  const int g = t / 32, k = t % 32;
  const long long r = r0 + g;
  float term = 0.f;
  if (g < nr && k < A) {
    const float mu = act[cur][g * kPolicyPitch + k];
    const float a = mu + s_sdv[k] * p.eps[r * p.lde + k];
    p.action[r * p.lda + k] = a;
    const float d = (a - mu) / s_sdv[k];
    term = -0.5f * d * d - s_ls[k] - kLogSqrt2Pi;
  }
  s_term[t] = term;
  __syncthreads();
  if (k == 0 && g < nr) {
    float lp = 0.f;
    for (int j = 0; j < A; ++j) lp += s_term[g * 32 + j];
    p.logp[r] = lp;
  }
}

// One float4 of the packed weights per thread (the layout is described with
// PolicyPackArgs). The segment is found by comparing against every
// segment's start with constant indices, so the arguments stay in scalar
// registers.
__device__ void policy_pack_body(const PolicyPackArgs& a) {
  const long long i = (long long)blockIdx.x * kThreads + threadIdx.x;
  if (i >= a.nq) return;
  long long src = 0, dst = 0, q0 = 0;
  int ldw = 0, N = 0, K = 0, kc = 1;
#pragma unroll
  for (int s = 0; s < kPolicyPackSegs; ++s)
    if (s < a.nseg && i >= a.seg[s].q0) {
      src = a.seg[s].src;
      dst = a.seg[s].dst;
      q0 = a.seg[s].q0;
      ldw = a.seg[s].ldw;
      N = a.seg[s].N;
      K = a.seg[s].K;
      kc = a.seg[s].kc;
    }
  const long long j = i - q0;
  const int lane = (int)(j & 63);
  const long long b = j >> 6;
  const int n = 16 * (int)(b / kc) + (lane & 15);
  const int k = 16 * (int)(b % kc) + 4 * (lane >> 4);
  float4 v = {0.f, 0.f, 0.f, 0.f};
  if (n < N && k < K) {
    // k < K <= ldw with k and ldw multiples of 4: the float4 stays in the row.
    v = *reinterpret_cast<const float4*>(a.params + src + (long long)n * ldw + k);
    if (k + 1 >= K) v.y = 0.f;
    if (k + 2 >= K) v.z = 0.f;
    if (k + 3 >= K) v.w = 0.f;
  }
  *reinterpret_cast<float4*>(a.dst + dst + 4 * j) = v;
}

}  // namespace zk

// Held to eight waves per SIMD (two 16-wave blocks per CU, at most 64 VGPRs).
extern "C" __global__ __launch_bounds__(zk::kPolicyThreads) __attribute__((amdgpu_waves_per_eu(8)))
void zk_policy(zk::PolicyArgs p) {
  zk::policy_body(p);
}

extern "C" __global__ __launch_bounds__(zk::kThreads) void zk_policy_pack(zk::PolicyPackArgs a) {
  zk::policy_pack_body(a);
}
