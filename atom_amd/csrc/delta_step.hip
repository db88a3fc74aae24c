// One token of the gated delta rule, from the projection's columns to the gated read-out, in one launch: what
// conv_silu_state, the two low-rank products (where the mixer has them), delta_prepare, delta_rule and delta_out do one
// after the other for prompts (delta_rule.hip has the mathematics).
//
// A decode step's kernels are each a launch, a wait for what the one before wrote through another die's cache, and an end,
// about 4 us whatever they compute; the state of 128 x 128 a head is read and written once either way.  A block takes a
// q/k head of a request with the value heads it serves, because these share the carried inputs of the convolution: the
// block that reads them is the only one that does and may move them up in place.  All loads that depend on nothing but the
// request's slot go out together, ahead of the first barrier.
//
// S is [dim, vdim]; a lane holds four neighbouring columns of every RG-th row.  Both products with the decayed state,
// S^T k and S^T q, come from one pass over it, o = S_new^T q = (g S)^T q + u (k . q), so that rows meet (lanes, then
// waves through LDS) once a token.
//
// What bounds it is that chain: two dependent rounds of loads, four barriers.  Against the launches one by one, heads of 128 x
// 128, two a q/k head, a layer and step of 1 / 4 / 8 / 16 / 32 / 64 requests, us less: 8 q/k heads with a decay a head (four
// launches) 4.2 / 8.0 / 14 / 24 / 39 / 66; with decays per channel and both low-rank products (six) 6.1 / 16 / 25 / 31 / 49 / 78;
// 4 q/k heads so 8.5 / 11 / 15 / 21 / 33 / 52 (runs of 16 steps: 6,888 -> 6,735 us with one such layer, 7,944 -> 7,620 with two).
// So steps of any number of requests take it.
#include "common.h"

constexpr int kStepThreads = 1024;
constexpr int kStepWaves = kStepThreads / kWave;
constexpr int kStepTaps = 4;
constexpr int kStepRank = 64;      // the largest inner size of a low-rank decay or gate

struct DeltaStepArgs {
  const float* proj;               // [tokens, ld]: q | k | v inputs of the convolution, and what the offsets below name
  long ld;
  const void* taps;                // [channels, 4]
  float* state;                    // a slot's row: [3, channels] carried inputs, ..., the heads' matrices at state_off
  long slot_stride, state_off;
  const int* cu_seqlens;
  const int* slot_of_seq;
  const void* decay2;              // [decays, decay_rank] or null: the raw decays are columns of proj
  const void* gate2;               // [heads * vdim, gate_rank] or null
  const float* a_log;
  const float* dt_bias;
  const float* norm;
  void* y;                         // [tokens, heads * vdim]
  int beta_off, decay_off, decay_rank, gate_off, gate_rank;
  int heads, kv_heads, channels, act;
  float eps;
};

// N: key and value channels of a head; G: value heads of a q/k head; CHANNEL: a decay per key channel.
template <typename T, int N, int G, bool CHANNEL>
__global__ void __launch_bounds__(kStepThreads) delta_step_kernel(DeltaStepArgs p) {
  constexpr int VL = N / 4;                      // lanes of a row of S
  constexpr int RG = kStepThreads / VL;          // rows that are held side by side
  constexpr int RPT = N / RG;                    // rows of a lane
  constexpr int CH = (2 + G) * N;                // channels of the block: q | k | v of its heads
  constexpr int ND = G * (CHANNEL ? N : 1);      // decays
  constexpr int NG = G * N;                      // gates, columns of the read-out
  static_assert(RPT >= 1 && CH <= kStepThreads && NG <= kStepThreads, "the block holds a q/k head");
  __shared__ __attribute__((aligned(16))) float conv[CH];
  __shared__ float low[2][kStepRank];
  __shared__ float dec[ND], gates[NG];
  __shared__ __attribute__((aligned(16))) float part[kStepWaves][G][2][N];
  __shared__ __attribute__((aligned(16))) float us[NG];
  __shared__ float os[NG];
  const int kvh = blockIdx.x, seq = blockIdx.y;
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int t = p.cu_seqlens[seq], end = p.cu_seqlens[seq + 1], slot = p.slot_of_seq[seq];
  if (t == end) return;
  T* y = (T*)p.y + (size_t)t * p.heads * N + (size_t)kvh * NG;
  if (slot < 0) {                                // a padded row: nothing is read or kept
    if (tid < NG) y[tid] = from_f32<T>(0.f);
    return;
  }
  const float* row = p.proj + (size_t)t * p.ld;
  float* tail = p.state + (size_t)slot * p.slot_stride;
  float* S0 = tail + p.state_off + (size_t)kvh * G * N * N;

  // the convolution's inputs, one channel a thread
  float in[kStepTaps];
  Four<T> w4;
  int ch = 0;
  if (tid < CH) {
    ch = tid < N ? kvh * N + tid : tid < 2 * N ? (p.kv_heads + kvh) * N + tid - N : 2 * p.kv_heads * N + kvh * NG + tid - 2 * N;
    in[3] = row[ch];
#pragma unroll
    for (int j = 0; j < kStepTaps - 1; ++j) in[j] = tail[(size_t)j * p.channels + ch];
    w4 = reinterpret_cast<const Four<T>*>(p.taps)[ch];
  }
  // the inner vectors of low-rank decays and gates, or the decays and gates themselves
  const int low_at = tid - (kStepThreads - 2 * kStepRank);
  float low_in = 0.f;
  if (low_at >= 0) {
    const int i = low_at % kStepRank;
    if (low_at < kStepRank ? i < p.decay_rank : i < p.gate_rank) low_in = row[(low_at < kStepRank ? p.decay_off : p.gate_off) + i];
  }
  const float dec_in = tid < ND && p.decay_rank == 0 ? row[p.decay_off + kvh * ND + tid] : 0.f;
  const float gate_in = tid < NG && p.gate_rank == 0 ? row[p.gate_off + kvh * NG + tid] : 0.f;
  const float bias_in = tid < ND ? p.dt_bias[kvh * ND + tid] : 0.f;
  const float alog_in = tid < ND ? p.a_log[kvh * G + tid / (ND / G)] : 0.f;
  const float beta_in = tid < NG ? row[p.beta_off + kvh * G + tid / N] : 0.f;
  // rows of the second products: two threads a row, half of its terms each (none where the rank is 0)
  constexpr int HALF = kStepRank / 2, EACH = 16 / sizeof(T), PIECES = HALF / EACH;
  constexpr int ITEMS = kStepThreads / 2, PASSES = (ND + NG + ITEMS - 1) / ITEMS;
  struct alignas(16) Piece { T at[EACH]; };
  Piece w2[PASSES][PIECES];
#pragma unroll
  for (int s = 0; s < PASSES; ++s) {
    const int item = tid / 2 + s * ITEMS;
    const bool gate = item >= ND;
    const int rank = item >= ND + NG ? 0 : gate ? p.gate_rank : p.decay_rank;
    const T* from = gate ? (const T*)p.gate2 + ((size_t)kvh * NG + item - ND) * rank : (const T*)p.decay2 + ((size_t)kvh * ND + item) * rank;
#pragma unroll
    for (int i = 0; i < PIECES; ++i)
      if (i * EACH < rank / 2) w2[s][i] = *reinterpret_cast<const Piece*>(from + tid % 2 * (rank / 2) + i * EACH);
  }
  const int col = tid % VL * 4, row0 = tid / VL;
  float4 S[G][RPT];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int i = 0; i < RPT; ++i) S[g][i] = *reinterpret_cast<const float4*>(S0 + ((size_t)g * N + row0 + RG * i) * N + col);

  if (low_at >= 0) low[low_at / kStepRank][low_at % kStepRank] = low_in;
  if (tid < CH) {
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < kStepTaps; ++j) s = fmaf(to_f32(w4.at[j]), in[j], s);
    conv[tid] = s / (1.f + expf(-s));
#pragma unroll
    for (int j = 0; j < kStepTaps - 1; ++j) tail[(size_t)j * p.channels + ch] = in[j + 1];
  }
  __syncthreads();

  const auto decay_of = [](float raw, float bias, float alog) {
    const float z = raw + bias;
    const float sp_z = z > 20.f ? z : log1pf(expf(z));
    return expf(-expf(alog) * sp_z);
  };
  if (tid < ND && p.decay_rank == 0) dec[tid] = decay_of(dec_in, bias_in, alog_in);
  if (tid < NG && p.gate_rank == 0) gates[tid] = gate_in;
  if (p.decay_rank > 0 || p.gate_rank > 0) {
#pragma unroll
    for (int s = 0; s < PASSES; ++s) {
      const int item = tid / 2 + s * ITEMS;
      const bool gate = item >= ND;
      const int rank = item >= ND + NG ? 0 : gate ? p.gate_rank : p.decay_rank;
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < PIECES; ++i)
        if (i * EACH < rank / 2)
#pragma unroll
          for (int e = 0; e < EACH; ++e)
            sum = fmaf(to_f32(w2[s][i].at[e]), low[gate ? 1 : 0][tid % 2 * (rank / 2) + i * EACH + e], sum);
      sum += __shfl_xor(sum, 1);
      if (rank > 0 && tid % 2 == 0) {
        if (gate) gates[item - ND] = sum;
        else dec[item] = decay_of(sum, p.dt_bias[kvh * ND + item], p.a_log[kvh * G + item / (ND / G)]);
      }
    }
  }
  // every wave finds the lengths of q and k and their product itself: no barrier of its own
  float qq = 0.f, kk = 0.f, qk = 0.f;
#pragma unroll
  for (int i = lane; i < N; i += kWave) {
    const float a = conv[i], b = conv[N + i];
    qq += a * a;
    kk += b * b;
    qk += a * b;
  }
  const float fq = (1.f / sqrtf((float)N)) / sqrtf(wave_sum(qq) + 1e-6f);
  const float fk = 1.f / sqrtf(wave_sum(kk) + 1e-6f);
  const float kq = wave_sum(qk) * fq * fk;
  __syncthreads();

  float kr[RPT];
#pragma unroll
  for (int i = 0; i < RPT; ++i) kr[i] = conv[N + row0 + RG * i] * fk;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    float a[4] = {0.f, 0.f, 0.f, 0.f}, b[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      const float d = CHANNEL ? dec[g * N + row0 + RG * i] : dec[g];
      const float qr = conv[row0 + RG * i] * fq;
      float* s = &S[g][i].x;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[e] *= d;
        a[e] = fmaf(s[e], kr[i], a[e]);
        b[e] = fmaf(s[e], qr, b[e]);
      }
    }
#pragma unroll
    for (int off = VL; off < kWave; off *= 2)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        a[e] += __shfl_xor(a[e], off);
        b[e] += __shfl_xor(b[e], off);
      }
    if (lane < VL) {
      *reinterpret_cast<float4*>(&part[wave][g][0][col]) = float4{a[0], a[1], a[2], a[3]};
      *reinterpret_cast<float4*>(&part[wave][g][1][col]) = float4{b[0], b[1], b[2], b[3]};
    }
  }
  __syncthreads();
  if (tid < NG) {
    const int g = tid / N, c = tid % N;
    float a = 0.f, b = 0.f;
#pragma unroll
    for (int w = 0; w < kStepWaves; ++w) {
      a += part[w][g][0][c];
      b += part[w][g][1][c];
    }
    const float beta = 1.f / (1.f + expf(-beta_in));
    const float u = beta * (conv[2 * N + tid] - a);
    us[tid] = u;
    os[tid] = fmaf(u, kq, b);
  }
  __syncthreads();
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const float4 u = *reinterpret_cast<const float4*>(&us[g * N + col]);
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      float4 s = S[g][i];
      s.x = fmaf(kr[i], u.x, s.x);
      s.y = fmaf(kr[i], u.y, s.y);
      s.z = fmaf(kr[i], u.z, s.z);
      s.w = fmaf(kr[i], u.w, s.w);
      *reinterpret_cast<float4*>(S0 + ((size_t)g * N + row0 + RG * i) * N + col) = s;
    }
  }
  if (wave < G) {   // the read-out's norm and gate, a wave a head
    float ss = 0.f;
#pragma unroll
    for (int i = lane; i < N; i += kWave) ss += os[wave * N + i] * os[wave * N + i];
    const float rstd = 1.f / sqrtf(wave_sum(ss) / (float)N + p.eps);
#pragma unroll
    for (int i = lane; i < N; i += kWave) {
      const float g = gates[wave * N + i];
      const float sig = 1.f / (1.f + expf(-g));
      y[wave * N + i] = from_f32<T>(os[wave * N + i] * rstd * p.norm[i] * (p.act == 0 ? g * sig : sig));
    }
  }
}

// 1 if the kernel takes these heads.  The inner size of a low-rank decay or gate (0: none) is a multiple of 16 up to 64.
ATOM_EXPORT int atom_delta_step_supports(int heads, int kv_heads, int dim, int vdim, int taps, int decay_rank, int gate_rank) {
  if (heads <= 0 || kv_heads <= 0 || heads % kv_heads || heads / kv_heads > 2 || heads > 65535) return 0;
  if (dim != vdim || (dim != 64 && dim != 128) || taps != kStepTaps) return 0;
  return decay_rank >= 0 && decay_rank <= kStepRank && decay_rank % 16 == 0 && gate_rank >= 0 && gate_rank <= kStepRank &&
         gate_rank % 16 == 0;
}

// Requests bring one token each, or none.  proj float32 [tokens, ld]; taps, decay2, gate2 and y of the type `dtype`.
ATOM_EXPORT int atom_delta_step(const float* proj, long ld, const void* taps, int dtype, float* state, long slot_stride,
                                long state_off, const int* cu_seqlens, const int* slot_of_seq, int num_seqs, int beta_off,
                                int decay_off, int decay_rank, const void* decay2, int gate_off, int gate_rank,
                                const void* gate2, int per_channel, const float* a_log, const float* dt_bias,
                                const float* norm, float eps, void* y, int heads, int kv_heads, int dim, int act,
                                hipStream_t stream) {
  if (!atom_delta_step_supports(heads, kv_heads, dim, dim, kStepTaps, decay_rank, gate_rank)) return ATOM_UNSUPPORTED;
  if ((unsigned)act > 1u) return ATOM_UNSUPPORTED;   // 0: SiLU of the gate, 1: its sigmoid
  if ((unsigned)dtype > 1u) return ATOM_BAD_DTYPE;
  const int channels = (2 * kv_heads + heads) * dim;
  const int decays = decay_rank ? decay_rank : heads * (per_channel ? dim : 1), gates = gate_rank ? gate_rank : heads * dim;
  if (num_seqs < 0 || ld < channels || beta_off < 0 || decay_off < 0 || gate_off < 0 || beta_off + heads > ld ||
      decay_off + decays > ld || gate_off + gates > ld)
    return ATOM_BAD_SHAPE;
  if (state_off < (long)(kStepTaps - 1) * channels || slot_stride < state_off + (long)heads * dim * dim) return ATOM_BAD_SHAPE;
  if (!proj || !taps || !state || !cu_seqlens || !slot_of_seq || !a_log || !dt_bias || !norm || !y) return ATOM_BAD_SHAPE;
  if ((decay_rank && !decay2) || (gate_rank && !gate2)) return ATOM_BAD_SHAPE;
  // rows of S and of the second products are read 16 bytes at a time
  if (slot_stride % 4 || state_off % 4 || (((uintptr_t)state | (uintptr_t)taps | (uintptr_t)decay2 | (uintptr_t)gate2) & 15))
    return ATOM_BAD_SHAPE;
  if (num_seqs == 0) return ATOM_OK;
  if (num_seqs > 65535) return ATOM_TOO_LARGE;
  const DeltaStepArgs p{proj, ld, taps, state, slot_stride, state_off, cu_seqlens, slot_of_seq, decay2, gate2, a_log, dt_bias,
                        norm, y, beta_off, decay_off, decay_rank, gate_off, gate_rank, heads, kv_heads, channels, act, eps};
  const dim3 grid(kv_heads, num_seqs), block(kStepThreads);
#define GO(NV, GV, CV) hipLaunchKernelGGL((delta_step_kernel<T, NV, GV, CV>), grid, block, 0, stream, p)
#define GO_DECAY(NV, GV)             \
  do {                               \
    if (per_channel) GO(NV, GV, true); \
    else GO(NV, GV, false);          \
  } while (0)
  const int pick = (dim == 128 ? 2 : 0) + (heads / kv_heads == 2 ? 1 : 0);
  ATOM_DISPATCH_DTYPE(dtype, switch (pick) {
    case 0: GO_DECAY(64, 1); break;
    case 1: GO_DECAY(64, 2); break;
    case 2: GO_DECAY(128, 1); break;
    default: GO_DECAY(128, 2); break;
  });
#undef GO_DECAY
#undef GO
  return launch_status();
}
