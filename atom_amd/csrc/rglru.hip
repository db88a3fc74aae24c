// The real-gated linear recurrence, token by token and channel by channel, in float32:
//
//   r = sigmoid(gr + br);  i = sigmoid(gi + bi);  log a = -scale * r * softplus(lam);  a = exp(log a)
//   S <- a S + sqrt(1 - a^2) (i u);   out = S * gelu_tanh(y)
//
// gr and gi are the gates' small products (before their biases), u the convolved input branch, y the other branch
// before its activation.  S [channels] sits in a request's state row at state_off and starts from what the slot
// holds (zero for a new request).  1 - a^2 is formed as -expm1(2 log a), which keeps its digits when a is near 1.
//
// Requests are walked through the step's device arrays, so prompt portions, single tokens and padded rows
// (slot < 0: nothing of the state is touched, zeros are written) run the same kernels.
//
// Short requests (up to 64 tokens each): one kernel, a thread owns a channel of a request and walks its tokens; the
// loads of the tokens ahead do not depend on S, so they are in flight while the chain runs.
// Longer ones: the recurrence is linear in S, so a run of 64 tokens acts on it as S -> A S + B with A the product
// of the run's decays and B what the run leaves of a zero state.  A first kernel forms (A, B) of every run (and
// copies the state S had before the step aside), a second one starts every run from the state before the step
// folded through the runs ahead of it, and walks the run's tokens.  Both have a block per (128 channels, request,
// run), so a prompt fills the chip instead of one wave per 64 channels walking all of it.
#include "common.h"

__device__ __forceinline__ float gelu_tanh_y(float z) {
  const float inner = 0.7978845608028654f * (z + 0.044715f * z * z * z);
  return 0.5f * z * (1.f + tanhf(inner));
}

struct Step {
  float a, b;
};

// One token's decay and input: S <- a S + b.
__device__ __forceinline__ Step token_step(float gr, float gi, float u, float rb, float ib, float rate) {
  const float r = 1.f / (1.f + expf(-(gr + rb)));
  const float g = 1.f / (1.f + expf(-(gi + ib)));
  const float log_a = rate * r;
  Step s;
  s.a = expf(log_a);
  s.b = sqrtf(-expm1f(2.f * log_a)) * (g * u);
  return s;
}

constexpr int kScanRun = 64;

// grid (channel blocks, requests, runs).  ab [requests, runs, 2, channels]; s0 [requests, channels].
__global__ void __launch_bounds__(128)
rglru_runs_kernel(const float* __restrict__ u, const float* __restrict__ gr, const float* __restrict__ gi,
                  const float* __restrict__ br, const float* __restrict__ bi, const float* __restrict__ lam,
                  const float* __restrict__ state, long slot_stride, long state_off, const int* __restrict__ cu_seqlens,
                  const int* __restrict__ slot_of_seq, float* __restrict__ ab, float* __restrict__ s0, int channels,
                  float scale) {
  const int c = blockIdx.x * 128 + threadIdx.x;
  const int seq = blockIdx.y, run = blockIdx.z, runs = gridDim.z;
  if (c >= channels) return;
  const int slot = slot_of_seq[seq];
  if (slot < 0) return;
  if (run == 0) s0[(size_t)seq * channels + c] = state[(size_t)slot * slot_stride + state_off + c];
  const int begin = cu_seqlens[seq], end = cu_seqlens[seq + 1];
  const int first = begin + run * kScanRun;
  if (first >= end) return;
  const int last = first + kScanRun < end ? first + kScanRun : end;
  const float l = lam[c];
  const float rate = -scale * (l > 20.f ? l : log1pf(expf(l)));
  const float rb = br[c], ib = bi[c];
  float A = 1.f, B = 0.f;
#pragma unroll 4
  for (int t = first; t < last; ++t) {
    const size_t at = (size_t)t * channels + c;
    const Step s = token_step(gr[at], gi[at], u[at], rb, ib, rate);
    A *= s.a;
    B = fmaf(s.a, B, s.b);
  }
  float* dst = ab + ((size_t)seq * runs + run) * 2 * channels + c;
  dst[0] = A;
  dst[channels] = B;
}

template <typename TO>
__global__ void __launch_bounds__(128)
rglru_scan_runs_kernel(const float* __restrict__ u, const float* __restrict__ gr, const float* __restrict__ gi,
                       const float* __restrict__ br, const float* __restrict__ bi, const float* __restrict__ lam,
                       const float* __restrict__ y, int ld_y, int y_off, float* __restrict__ state, long slot_stride,
                       long state_off, const int* __restrict__ cu_seqlens, const int* __restrict__ slot_of_seq,
                       const float* __restrict__ ab, const float* __restrict__ s0, TO* __restrict__ out, int channels,
                       float scale) {
  const int c = blockIdx.x * 128 + threadIdx.x;
  const int seq = blockIdx.y, run = blockIdx.z, runs = gridDim.z;
  if (c >= channels) return;
  const int begin = cu_seqlens[seq], end = cu_seqlens[seq + 1];
  const int first = begin + run * kScanRun;
  if (first >= end) return;
  const int last = first + kScanRun < end ? first + kScanRun : end;
  const int slot = slot_of_seq[seq];
  if (slot < 0) {
    for (int t = first; t < last; ++t) out[(size_t)t * channels + c] = from_f32<TO>(0.f);
    return;
  }
  float S = s0[(size_t)seq * channels + c];
  const float* src = ab + (size_t)seq * runs * 2 * channels + c;
  for (int j = 0; j < run; ++j) S = fmaf(src[(size_t)j * 2 * channels], S, src[(size_t)j * 2 * channels + channels]);
  const float l = lam[c];
  const float rate = -scale * (l > 20.f ? l : log1pf(expf(l)));
  const float rb = br[c], ib = bi[c];
#pragma unroll 4
  for (int t = first; t < last; ++t) {
    const size_t at = (size_t)t * channels + c;
    const Step s = token_step(gr[at], gi[at], u[at], rb, ib, rate);
    S = fmaf(s.a, S, s.b);
    out[at] = from_f32<TO>(S * gelu_tanh_y(y[(size_t)t * ld_y + y_off + c]));
  }
  if (last == end) state[(size_t)slot * slot_stride + state_off + c] = S;
}

template <typename TO>
__global__ void __launch_bounds__(128)
rglru_scan_kernel(const float* __restrict__ u, const float* __restrict__ gr, const float* __restrict__ gi,
                  const float* __restrict__ br, const float* __restrict__ bi, const float* __restrict__ lam,
                  const float* __restrict__ y, int ld_y, int y_off, float* __restrict__ state, long slot_stride,
                  long state_off, const int* __restrict__ cu_seqlens, const int* __restrict__ slot_of_seq,
                  TO* __restrict__ out, int channels, float scale) {
  const int c = blockIdx.x * 128 + threadIdx.x;
  const int seq = blockIdx.y;
  if (c >= channels) return;
  const int begin = cu_seqlens[seq], end = cu_seqlens[seq + 1];
  const int slot = slot_of_seq[seq];
  if (slot < 0) {
    for (int t = begin; t < end; ++t) out[(size_t)t * channels + c] = from_f32<TO>(0.f);
    return;
  }
  float* sp = state + (size_t)slot * slot_stride + state_off + c;
  float S = *sp;
  const float l = lam[c];
  const float rate = -scale * (l > 20.f ? l : log1pf(expf(l)));
  const float rb = br[c], ib = bi[c];
#pragma unroll 4
  for (int t = begin; t < end; ++t) {
    const size_t at = (size_t)t * channels + c;
    const Step s = token_step(gr[at], gi[at], u[at], rb, ib, rate);
    S = fmaf(s.a, S, s.b);
    out[at] = from_f32<TO>(S * gelu_tanh_y(y[(size_t)t * ld_y + y_off + c]));
  }
  *sp = S;
}

ATOM_EXPORT int atom_rglru_scan(const float* u, const float* gr, const float* gi, const float* br, const float* bi,
                                const float* lam, const float* y, int ld_y, int y_off, float* state, long slot_stride,
                                long state_off, const int* cu_seqlens, const int* slot_of_seq, int num_seqs, void* out,
                                int out_dtype, int channels, float scale, int max_q_len, float* workspace,
                                long workspace_floats, hipStream_t stream) {
  if (channels <= 0 || num_seqs < 0 || y_off < 0 || y_off + channels > ld_y) return ATOM_BAD_SHAPE;
  if (state_off < 0 || slot_stride < state_off + channels) return ATOM_BAD_SHAPE;
  if (u == nullptr || gr == nullptr || gi == nullptr || br == nullptr || bi == nullptr || lam == nullptr ||
      y == nullptr || state == nullptr || cu_seqlens == nullptr || slot_of_seq == nullptr || out == nullptr)
    return ATOM_BAD_SHAPE;
  if (num_seqs == 0) return ATOM_OK;
  if (num_seqs > 65535 || max_q_len < 0) return ATOM_TOO_LARGE;
  if (max_q_len > kScanRun && workspace != nullptr) {
    // runs of 64 tokens side by side; the workspace holds the states before the step, then every run's (A, B)
    const int runs = (max_q_len + kScanRun - 1) / kScanRun;
    if (runs > 65535) return ATOM_TOO_LARGE;
    if (workspace_floats < (long)num_seqs * channels * (1 + 2 * (long)runs)) return ATOM_BAD_SHAPE;
    float* s0 = workspace;
    float* ab = workspace + (size_t)num_seqs * channels;
    dim3 grid((channels + 127) / 128, num_seqs, runs), block(128);
    hipLaunchKernelGGL(rglru_runs_kernel, grid, block, 0, stream, u, gr, gi, br, bi, lam, state, slot_stride, state_off,
                       cu_seqlens, slot_of_seq, ab, s0, channels, scale);
    ATOM_DISPATCH_DTYPE(out_dtype, hipLaunchKernelGGL((rglru_scan_runs_kernel<T>), grid, block, 0, stream, u, gr, gi, br,
                                                       bi, lam, y, ld_y, y_off, state, slot_stride, state_off, cu_seqlens,
                                                       slot_of_seq, ab, s0, (T*)out, channels, scale));
    return launch_status();
  }
  dim3 grid((channels + 127) / 128, num_seqs), block(128);
  ATOM_DISPATCH_DTYPE(out_dtype, hipLaunchKernelGGL((rglru_scan_kernel<T>), grid, block, 0, stream, u, gr, gi, br, bi,
                                                     lam, y, ld_y, y_off, state, slot_stride, state_off, cu_seqlens,
                                                     slot_of_seq, (T*)out, channels, scale));
  return launch_status();
}

// ------------------------------------------------------------------ a decode step: one token a request
//
// From the projection's columns to the gated output in two launches instead of four (convolution, the gates' two products,
// the scan; each some 4 us of a decode step whatever it does).  The first forms both gates' products; every one of its
// blocks convolves the inputs of its channels anew (four values a channel) and nothing is moved up, so the second, which has
// a channel a thread, finds the carried inputs as they were, convolves its own channel, and alone moves them up.
// Width 2,048 in 8 blocks of 256, two such layers, a step of 1 / 4 / 8 requests: 12 / 20 / 24 us less than with four launches (four
// token tables' gates in their products' epilogue 3.4 / 4.6 / 8.8 more).  Steps of more requests keep the four: every block of the
// first launch convolves all requests anew.

constexpr int kStepTaps = 4;
constexpr int kStepSeqs = 8;       // the most requests of a step
constexpr int kStepCols = 8;       // channels of a block whose gates it forms

struct RglruStep {
  const float* proj;               // [tokens, ld]: the input branch, then the other at y_off
  long ld;
  const void* taps;                // [channels, 4]
  const float* conv_bias;
  float* state;                    // a slot's row: [3, channels] carried inputs, S at state_off
  long slot_stride, state_off;
  const int* cu_seqlens;
  const int* slot_of_seq;
  const void* ra;                  // [blocks, part, part]
  const void* ri;
  const float* br;
  const float* bi;
  const float* lam;
  float* gates;                    // [2, tokens, channels]
  void* out;
  int num_seqs, tokens, channels, part, y_off;
  float scale;
};

// The convolved input of channel c, and (win) what the request carries of it.
template <typename T>
__device__ __forceinline__ float convolved(const RglruStep& p, int t, int slot, int c, float (&win)[kStepTaps]) {
  const float* tail = p.state + (size_t)slot * p.slot_stride;
  win[kStepTaps - 1] = p.proj[(size_t)t * p.ld + c];
#pragma unroll
  for (int j = 0; j < kStepTaps - 1; ++j) win[j] = tail[(size_t)j * p.channels + c];
  const Four<T> w = reinterpret_cast<const Four<T>*>(p.taps)[c];
  float s = 0.f;
#pragma unroll
  for (int j = 0; j < kStepTaps; ++j) s = fmaf(to_f32(w.at[j]), win[j], s);
  return s + p.conv_bias[c];
}

// grid (part / 8, blocks); PL: weights of a row that a lane holds, part / 64.  A wave forms four of the block's sixteen
// products (8 channels, 2 gates), each of a row of weights with every request's channels.
template <typename T, int PL>
__global__ void __launch_bounds__(256) rglru_step_gates_kernel(RglruStep p) {
  constexpr int PART = PL * kWave, OUTS = 2 * kStepCols / 4;
  __shared__ float us[kStepSeqs][PART];
  struct alignas(PL * sizeof(T)) Lane { T at[PL]; };
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int c0 = blockIdx.y * PART;
  Lane w[OUTS];
#pragma unroll
  for (int o = 0; o < OUTS; ++o) {
    const int which = wave * OUTS + o, col = blockIdx.x * kStepCols + which % kStepCols;
    w[o] = *reinterpret_cast<const Lane*>((const T*)(which < kStepCols ? p.ra : p.ri) + ((size_t)c0 + col) * PART + lane * PL);
  }
  for (int s = 0; s < p.num_seqs; ++s) {
    const int t = p.cu_seqlens[s], slot = p.slot_of_seq[s];
    if (slot < 0 || p.cu_seqlens[s + 1] == t) continue;
    for (int c = tid; c < PART; c += 256) {
      float win[kStepTaps];
      us[s][c] = convolved<T>(p, t, slot, c0 + c, win);
    }
  }
  __syncthreads();
  for (int s = 0; s < p.num_seqs; ++s) {
    const int t = p.cu_seqlens[s];
    if (p.slot_of_seq[s] < 0 || p.cu_seqlens[s + 1] == t) continue;
    float u[PL];
#pragma unroll
    for (int e = 0; e < PL; ++e) u[e] = us[s][lane * PL + e];
#pragma unroll
    for (int o = 0; o < OUTS; ++o) {
      const int which = wave * OUTS + o, col = blockIdx.x * kStepCols + which % kStepCols;
      float sum = 0.f;
#pragma unroll
      for (int e = 0; e < PL; ++e) sum = fmaf(u[e], to_f32(w[o].at[e]), sum);
      sum = wave_sum(sum);
      if (lane == 0) p.gates[((size_t)(which < kStepCols ? 0 : p.tokens) + t) * p.channels + c0 + col] = sum;
    }
  }
}

template <typename T>
__global__ void __launch_bounds__(64) rglru_step_kernel(RglruStep p) {
  const int c = blockIdx.x * 64 + threadIdx.x, s = blockIdx.y;
  const int t = p.cu_seqlens[s], slot = p.slot_of_seq[s];
  if (c >= p.channels || p.cu_seqlens[s + 1] == t) return;
  T* out = (T*)p.out + (size_t)t * p.channels + c;
  if (slot < 0) {
    *out = from_f32<T>(0.f);
    return;
  }
  float* row = p.state + (size_t)slot * p.slot_stride;
  const float l = p.lam[c], S0 = row[p.state_off + c], y = p.proj[(size_t)t * p.ld + p.y_off + c];
  const float gr = p.gates[(size_t)t * p.channels + c], gi = p.gates[((size_t)p.tokens + t) * p.channels + c];
  float win[kStepTaps];
  const float u = convolved<T>(p, t, slot, c, win);
  const float rate = -p.scale * (l > 20.f ? l : log1pf(expf(l)));
  const Step step = token_step(gr, gi, u, p.br[c], p.bi[c], rate);
  const float S = fmaf(step.a, S0, step.b);
  *out = from_f32<T>(S * gelu_tanh_y(y));
  row[p.state_off + c] = S;
#pragma unroll
  for (int j = 0; j < kStepTaps - 1; ++j) row[(size_t)j * p.channels + c] = win[j + 1];
}

// 1 if the kernels take these sizes.
ATOM_EXPORT int atom_rglru_step_supports(int num_seqs, int channels, int part, int taps) {
  return num_seqs >= 1 && num_seqs <= kStepSeqs && taps == kStepTaps && (part == 64 || part == 128 || part == 256 || part == 512) &&
         channels > 0 && channels % part == 0 && channels / part <= 65535;
}

// Requests bring one token each, or none; taps, ra, ri and out of the type `dtype`, whose tensors begin at multiples of 16 bytes.
ATOM_EXPORT int atom_rglru_step(const float* proj, long ld, int y_off, const void* taps, const float* conv_bias, int dtype,
                                float* state, long slot_stride, long state_off, const int* cu_seqlens, const int* slot_of_seq,
                                int num_seqs, int tokens, const void* ra, const void* ri, const float* br, const float* bi,
                                const float* lam, float* gates, void* out, int channels, int part, float scale,
                                hipStream_t stream) {
  if (!atom_rglru_step_supports(num_seqs, channels, part, kStepTaps)) return ATOM_UNSUPPORTED;
  if ((unsigned)dtype > 1u) return ATOM_BAD_DTYPE;
  if (ld < channels || y_off < 0 || y_off + channels > ld || tokens < 0 || tokens > num_seqs) return ATOM_BAD_SHAPE;
  if (state_off < (long)(kStepTaps - 1) * channels || slot_stride < state_off + channels) return ATOM_BAD_SHAPE;
  if (!proj || !taps || !conv_bias || !state || !cu_seqlens || !slot_of_seq || !ra || !ri || !br || !bi || !lam || !gates || !out)
    return ATOM_BAD_SHAPE;
  if (((uintptr_t)taps | (uintptr_t)ra | (uintptr_t)ri) & 15) return ATOM_BAD_SHAPE;
  if (tokens == 0) return ATOM_OK;
  const RglruStep p{proj, ld, taps, conv_bias, state, slot_stride, state_off, cu_seqlens, slot_of_seq, ra, ri, br, bi, lam,
                    gates, out, num_seqs, tokens, channels, part, y_off, scale};
  const dim3 grid(part / kStepCols, channels / part);
#define GO(PL) hipLaunchKernelGGL((rglru_step_gates_kernel<T, PL>), grid, dim3(256), 0, stream, p)
  ATOM_DISPATCH_DTYPE(dtype, {
    switch (part) {
      case 64: GO(1); break;
      case 128: GO(2); break;
      case 256: GO(4); break;
      default: GO(8); break;
    }
    hipLaunchKernelGGL((rglru_step_kernel<T>), dim3((channels + 63) / 64, num_seqs), dim3(64), 0, stream, p);
  });
#undef GO
  return launch_status();
}
