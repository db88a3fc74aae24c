// One token a request of the linear recurrences (linear_scan.hip has the mathematics), with what stands before and behind
// them, in fewer launches: a decode step's kernels take some 4 us each whatever they compute.
//
//   state space   conv_silu_state and linear_scan in one launch, a block a head and request; the channels of B and C that
//                 all heads of a group read are convolved by each of them, and the carried inputs stay as they are until
//                 the second launch, which norms and gates the read-outs (one group a row) and moves them up.
//   time mixing   the decays' second product, linear_scan with its bonus and the read-out's norm and gate in one.
//
// A lane holds four neighbouring columns of every RG-th row of S; all loads that depend on nothing but the request's slot go
// out together, and rows meet once (lanes, then waves through LDS).  What bounds them is two dependent rounds of loads and
// three barriers.  Against the launches one by one, two layers of state space (64 heads of 128 x 64) and one of time mixing (32
// heads of 64 x 64), four launches fewer in a step of 1 / 4 / 8 / 16 / 32 / 64 requests: 24 / 27 / 31 / 44 / 68 / 98 us less, so
// steps of any number of requests take them (a prompt of 5,569 tokens and 16 steps of four requests 9,685 -> 9,257 us).
#include "common.h"

constexpr int kStepTaps = 4;

__device__ __forceinline__ float step_silu(float v) { return v / (1.f + expf(-v)); }

struct SpaceStepArgs {
  const float* proj;               // [tokens, ld]: z | x | B | C | step sizes (x at x_off)
  long ld;
  const void* taps;                // [channels, 4]
  const float* conv_bias;
  float* state;                    // a slot's row: [3, channels] carried inputs, the heads' matrices at state_off
  long slot_stride, state_off;
  const int* cu_seqlens;
  const int* slot_of_seq;
  const float* step_bias;
  const float* a_log;
  const float* skip;
  const float* norm;
  float* y;                        // [tokens, inner]
  void* out;
  int heads, groups, channels, inner, x_off;
  float eps;
};

template <typename T, int K, int V>
__global__ void __launch_bounds__(512) space_step_kernel(SpaceStepArgs p) {
  constexpr int VL = V / 4, RG = 512 / VL, RPT = K / RG, CH = V + 2 * K, WAVES = 512 / kWave;
  static_assert(RPT >= 1 && CH <= 512 && VL <= kWave, "the block holds a head");
  __shared__ float conv[CH];                       // x | B | C
  __shared__ __attribute__((aligned(16))) float part[WAVES][V];
  const int h = blockIdx.x, seq = blockIdx.y, tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int t = p.cu_seqlens[seq], end = p.cu_seqlens[seq + 1], slot = p.slot_of_seq[seq];
  if (t == end) return;
  float* y = p.y + (size_t)t * p.inner + (size_t)h * V;
  if (slot < 0) {
    if (tid < V) y[tid] = 0.f;
    return;
  }
  const float* row = p.proj + (size_t)t * p.ld;
  const float* tail = p.state + (size_t)slot * p.slot_stride;
  float* S0 = p.state + (size_t)slot * p.slot_stride + p.state_off + (size_t)h * K * V;
  const int group = h / (p.heads / p.groups);
  float in[kStepTaps], bias = 0.f;
  Four<T> w4;
  if (tid < CH) {
    const int c = tid < V ? h * V + tid : tid < V + K ? p.inner + group * K + tid - V : p.inner + (p.groups + group) * K + tid - V - K;
    in[3] = row[p.x_off + c];
#pragma unroll
    for (int j = 0; j < kStepTaps - 1; ++j) in[j] = tail[(size_t)j * p.channels + c];
    w4 = reinterpret_cast<const Four<T>*>(p.taps)[c];
    bias = p.conv_bias[c];
  }
  const float z = row[p.x_off + p.channels + h] + p.step_bias[h], alog = p.a_log[h], skip = p.skip[h];
  const int col = tid % VL * 4, row0 = tid / VL;
  float4 S[RPT];
#pragma unroll
  for (int i = 0; i < RPT; ++i) S[i] = *reinterpret_cast<const float4*>(S0 + (size_t)(row0 + RG * i) * V + col);
  if (tid < CH) {
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < kStepTaps; ++j) s = fmaf(to_f32(w4.at[j]), in[j], s);
    conv[tid] = step_silu(s + bias);
  }
  const float step = z > 20.f ? z : log1pf(expf(z));
  const float decay = expf(-expf(alog) * step);
  __syncthreads();
  float v[4], acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = conv[col + e] * step;
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const float k = conv[V + row0 + RG * i], r = conv[V + K + row0 + RG * i];
    float* s = &S[i].x;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      s[e] = decay * s[e] + k * v[e];
      acc[e] = fmaf(r, s[e], acc[e]);
    }
    *reinterpret_cast<float4*>(S0 + (size_t)(row0 + RG * i) * V + col) = S[i];
  }
#pragma unroll
  for (int off = VL; off < kWave; off *= 2)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] += __shfl_xor(acc[e], off);
  if (lane < VL) *reinterpret_cast<float4*>(&part[wave][col]) = float4{acc[0], acc[1], acc[2], acc[3]};
  __syncthreads();
  if (tid < V) {
    float o = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) o += part[w][tid];
    y[tid] = o + skip * conv[tid];
  }
}

// grid (requests, 1 + channels / 1,024): the first block of a request norms and gates its row, the others move its channels up.
template <typename T>
__global__ void __launch_bounds__(1024) space_step_out_kernel(SpaceStepArgs p) {
  __shared__ float scratch[16];
  const int seq = blockIdx.x, tid = threadIdx.x;
  const int t = p.cu_seqlens[seq], end = p.cu_seqlens[seq + 1], slot = p.slot_of_seq[seq];
  if (t == end) return;
  if (blockIdx.y > 0) {
    const int c = (blockIdx.y - 1) * 1024 + tid;
    if (slot < 0 || c >= p.channels) return;
    float* tail = p.state + (size_t)slot * p.slot_stride + c;
    const float b = tail[p.channels], d = tail[2 * (size_t)p.channels], x = p.proj[(size_t)t * p.ld + p.x_off + c];
    tail[0] = b;
    tail[p.channels] = d;
    tail[2 * (size_t)p.channels] = x;
    return;
  }
  constexpr int MOST = 4;                          // groups of four entries a thread: rows of up to 16,384
  float v[MOST][4], ss = 0.f;
#pragma unroll
  for (int j = 0; j < MOST; ++j) {
    const int i = (tid + j * 1024) * 4;
    if (i >= p.inner) continue;
    float g[4];
    reinterpret_cast<const Four<float>*>(p.y + (size_t)t * p.inner + i)->to(v[j]);
    reinterpret_cast<const Four<float>*>(p.proj + (size_t)t * p.ld + i)->to(g);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[j][e] *= step_silu(g[e]);
      ss += v[j][e] * v[j][e];
    }
  }
  const float inv = 1.f / sqrtf(block_sum(ss, scratch) / (float)p.inner + p.eps);
#pragma unroll
  for (int j = 0; j < MOST; ++j) {
    const int i = (tid + j * 1024) * 4;
    if (i >= p.inner) continue;
    float w[4];
    reinterpret_cast<const Four<float>*>(p.norm + i)->to(w);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[j][e] = v[j][e] * inv * w[e];
    reinterpret_cast<Four<T>*>((T*)p.out + (size_t)t * p.inner + i)->from(v[j]);
  }
}

// 1 if the kernels take these sizes: heads of 64 or 128 rows by 64 columns, one group of the read-out's norm.
ATOM_EXPORT int atom_space_step_supports(int heads, int groups, int dim, int vdim, int taps, int norm_groups) {
  return heads > 0 && heads <= 65535 && groups > 0 && heads % groups == 0 && (dim == 64 || dim == 128) && vdim == 64 &&
         taps == kStepTaps && norm_groups == 1 && (long)heads * vdim <= 16384;
}

// Requests bring one token each, or none.  proj: z (heads vdim columns) | x | B | C | step sizes, x at x_off; taps and out of
// the type `dtype`.
ATOM_EXPORT int atom_space_step(const float* proj, long ld, int x_off, const void* taps, const float* conv_bias, int dtype,
                                float* state, long slot_stride, long state_off, const int* cu_seqlens, const int* slot_of_seq,
                                int num_seqs, const float* step_bias, const float* a_log, const float* skip, const float* norm,
                                float eps, float* y, void* out, int heads, int groups, int dim, int vdim, hipStream_t stream) {
  if (!atom_space_step_supports(heads, groups, dim, vdim, kStepTaps, 1)) return ATOM_UNSUPPORTED;
  if ((unsigned)dtype > 1u) return ATOM_BAD_DTYPE;
  const int inner = heads * vdim, channels = inner + 2 * groups * dim;
  if (num_seqs < 0 || x_off < 0 || ld < inner || ld < (long)x_off + channels + heads) return ATOM_BAD_SHAPE;
  if (state_off < (long)(kStepTaps - 1) * channels || slot_stride < state_off + (long)inner * dim) return ATOM_BAD_SHAPE;
  if (!proj || !taps || !conv_bias || !state || !cu_seqlens || !slot_of_seq || !step_bias || !a_log || !skip || !norm || !y || !out)
    return ATOM_BAD_SHAPE;
  // rows of S, and of what the second kernel reads, go 16 bytes at a time
  if (slot_stride % 4 || state_off % 4 || ld % 4 ||
      (((uintptr_t)proj | (uintptr_t)state | (uintptr_t)taps | (uintptr_t)norm | (uintptr_t)y | (uintptr_t)out) & 15))
    return ATOM_UNSUPPORTED;
  if (num_seqs == 0) return ATOM_OK;
  if (num_seqs > 65535) return ATOM_TOO_LARGE;
  const SpaceStepArgs p{proj, ld, taps, conv_bias, state, slot_stride, state_off, cu_seqlens, slot_of_seq, step_bias, a_log,
                        skip, norm, y, out, heads, groups, channels, inner, x_off, eps};
  const dim3 grid(heads, num_seqs), after(num_seqs, 1 + (channels + 1023) / 1024);
  ATOM_DISPATCH_DTYPE(dtype, {
    if (dim == 128) hipLaunchKernelGGL((space_step_kernel<T, 128, 64>), grid, dim3(512), 0, stream, p);
    else hipLaunchKernelGGL((space_step_kernel<T, 64, 64>), grid, dim3(512), 0, stream, p);
    hipLaunchKernelGGL((space_step_out_kernel<T>), after, dim3(1024), 0, stream, p);
  });
  return launch_status();
}

// ------------------------------------------------------------------ time mixing

constexpr int kMix = 64;           // rows and columns of a head
constexpr int kMixRank = 128;      // the largest inner size of the decays' product

struct MixStepArgs {
  const float* r; const float* k; const float* v; const float* g;   // [tokens, heads * 64]
  const float* squashed;           // [tokens, rank]
  const void* decay2;              // [heads * 64, rank]
  const float* decay_bias;
  const float* bonus;
  const float* norm;
  float* state;
  long slot_stride, state_off;
  const int* cu_seqlens;
  const int* slot_of_seq;
  void* out;                       // [tokens, heads * 64]
  int heads, rank;
  float eps;
};

template <typename T>
__global__ void __launch_bounds__(256) mix_step_kernel(MixStepArgs p) {
  constexpr int VL = kMix / 4, RG = 256 / VL, RPT = kMix / RG, WAVES = 256 / kWave;
  __shared__ float rs[kMix], ks[kMix], vs[kMix], dec[kMix], sq[kMixRank];
  __shared__ __attribute__((aligned(16))) float part[WAVES][kMix];
  const int h = blockIdx.x, seq = blockIdx.y, tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int t = p.cu_seqlens[seq], end = p.cu_seqlens[seq + 1], slot = p.slot_of_seq[seq];
  if (t == end) return;
  const size_t at = ((size_t)t * p.heads + h) * kMix;
  T* out = (T*)p.out + at;
  if (slot < 0) {
    if (tid < kMix) out[tid] = from_f32<T>(0.f);
    return;
  }
  float* S0 = p.state + (size_t)slot * p.slot_stride + p.state_off + (size_t)h * kMix * kMix;
  const int col = tid % VL * 4, row0 = tid / VL;
  // r, k and v by a wave each; the fourth keeps the gate for the end.  The decays' product: four threads a row.
  const float mine = (wave == 0 ? p.r : wave == 1 ? p.k : wave == 2 ? p.v : p.g)[at + lane];
  const float sq_in = tid < p.rank ? p.squashed[(size_t)t * p.rank + tid] : 0.f;
  const float u = p.bonus[(size_t)h * kMix + lane], weight = p.norm[(size_t)h * kMix + lane];
  const float bias = p.decay_bias[(size_t)h * kMix + tid / 4];
  constexpr int EACH = 16 / sizeof(T), PIECES = kMixRank / 4 / EACH;
  struct alignas(16) Piece { T at[EACH]; };
  Piece w2[PIECES];
  const int quarter = p.rank / 4;
  const T* from = (const T*)p.decay2 + ((size_t)h * kMix + tid / 4) * p.rank + tid % 4 * quarter;
#pragma unroll
  for (int i = 0; i < PIECES; ++i)
    if (i * EACH < quarter) w2[i] = *reinterpret_cast<const Piece*>(from + i * EACH);
  float4 S[RPT];
#pragma unroll
  for (int i = 0; i < RPT; ++i) S[i] = *reinterpret_cast<const float4*>(S0 + (size_t)(row0 + RG * i) * kMix + col);
  if (wave < 3) (wave == 0 ? rs : wave == 1 ? ks : vs)[lane] = mine;
  if (tid < p.rank) sq[tid] = sq_in;
  __syncthreads();
  float raw = 0.f;
#pragma unroll
  for (int i = 0; i < PIECES; ++i)
    if (i * EACH < quarter)
#pragma unroll
      for (int e = 0; e < EACH; ++e) raw = fmaf(to_f32(w2[i].at[e]), sq[tid % 4 * quarter + i * EACH + e], raw);
  raw += __shfl_xor(raw, 1);
  raw += __shfl_xor(raw, 2);
  if (tid % 4 == 0) dec[tid / 4] = expf(-expf(raw + bias));
  const float own = wave_sum(rs[lane] * u * ks[lane]);   // the token's own part of the read-out, by v
  __syncthreads();
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int r = row0 + RG * i;
    const float rr = rs[r], kk = ks[r], d = dec[r];
    float* s = &S[i].x;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      acc[e] = fmaf(rr, s[e], acc[e]);
      s[e] = d * s[e] + kk * vs[col + e];
    }
    *reinterpret_cast<float4*>(S0 + (size_t)r * kMix + col) = S[i];
  }
#pragma unroll
  for (int off = VL; off < kWave; off *= 2)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] += __shfl_xor(acc[e], off);
  if (lane < VL) *reinterpret_cast<float4*>(&part[wave][col]) = float4{acc[0], acc[1], acc[2], acc[3]};
  __syncthreads();
  if (wave == 3) {                                       // the wave that has the gate
    float o = own * vs[lane];
#pragma unroll
    for (int w = 0; w < WAVES; ++w) o += part[w][lane];
    const float inv = 1.f / sqrtf(wave_sum(o * o) / (float)kMix + p.eps);
    out[lane] = from_f32<T>(o * inv * weight * step_silu(mine));
  }
}

// 1 if the kernel takes these sizes: heads of 64 by 64, ranks of 32 to 128 in steps of 32.
ATOM_EXPORT int atom_mix_step_supports(int heads, int dim, int rank) {
  return heads > 0 && heads <= 65535 && dim == kMix && rank >= 32 && rank <= kMixRank && rank % 32 == 0;
}

// Requests bring one token each, or none; decay2 and out of the type `dtype`.
ATOM_EXPORT int atom_mix_step(const float* r, const float* k, const float* v, const float* g, const float* squashed,
                              const void* decay2, int dtype, const float* decay_bias, const float* bonus, const float* norm,
                              float* state, long slot_stride, long state_off, const int* cu_seqlens, const int* slot_of_seq,
                              int num_seqs, void* out, int heads, int dim, int rank, float eps, hipStream_t stream) {
  if (!atom_mix_step_supports(heads, dim, rank)) return ATOM_UNSUPPORTED;
  if ((unsigned)dtype > 1u) return ATOM_BAD_DTYPE;
  if (num_seqs < 0 || state_off < 0 || slot_stride < state_off + (long)heads * dim * dim) return ATOM_BAD_SHAPE;
  if (!r || !k || !v || !g || !squashed || !decay2 || !decay_bias || !bonus || !norm || !state || !cu_seqlens || !slot_of_seq || !out)
    return ATOM_BAD_SHAPE;
  if (slot_stride % 4 || state_off % 4 || (((uintptr_t)state | (uintptr_t)decay2) & 15)) return ATOM_UNSUPPORTED;
  if (num_seqs == 0) return ATOM_OK;
  if (num_seqs > 65535) return ATOM_TOO_LARGE;
  const MixStepArgs p{r, k, v, g, squashed, decay2, decay_bias, bonus, norm, state, slot_stride, state_off, cu_seqlens,
                      slot_of_seq, out, heads, rank, eps};
  ATOM_DISPATCH_DTYPE(dtype, hipLaunchKernelGGL((mix_step_kernel<T>), dim3(heads, num_seqs), dim3(256), 0, stream, p));
  return launch_status();
}
