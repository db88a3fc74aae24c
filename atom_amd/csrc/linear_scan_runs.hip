// A linear recurrence with one decay per head over runs of 64 tokens, as products of the matrix cores' float32
// instructions.  With c_t the sum of the logarithms of a run's decays up to token t, S the state before the run, k_t, r_t,
// v_t as in linear_scan.hip and dt_t the step sizes,
//
//   what the run adds     B = sum_t exp(c_end - c_t) dt_t k_t v_t^T
//   its outputs           o_t = exp(c_t) S^T r_t + sum_{i <= t} exp(c_t - c_i) dt_i (r_t . k_i) v_i   (+ skip v_t)
//
// in three launches: B of every run; per request the states before its runs (and the one after the last, which goes to the
// slot); the outputs.  The scores r_t . k_i do not depend on the head where heads share r and k: a block takes several
// such heads, stages r and k and forms the scores once, and brings one head's v and state while it works on the head
// before.
//
// Everything is float32; the logarithms are summed in float64 and kept as two floats, so that a difference of two of them
// is as exact as the decays' own products are.  An infinity or a NaN of a token reaches that token and those behind it only,
// as in the walk token by token: a wave whose 16 tokens' values hold any takes their triangle term by term, because a zero
// above the diagonal times such a value is not zero.
//
// Requests of one run (64 tokens or fewer) are left to the walk token by token, which follows for them alone: they take it
// without longer ones beside them too, so a token's result does not depend on those, and a single token does not pay for a
// run (64 heads of 128 x 64, 512 tokens beside 24 single ones: 175 us with runs for all, 115 so; beside three of 40 tokens 73
// and 95).
//
// Against a walk of the runs token by token (which it replaces for these sizes): 5,569 tokens of 64 heads of 128 x 64,
// 99 + 81 + 203 us for the three launches, 263 + 80 + 486 so.  At the smallest, 65 tokens of 32 heads, 30 us and 77.
// The first and the last are bound by their blocks' waits between the stages of a head (they run at 0.37 and 0.26 of the float32
// rate of the matrix cores), the middle one by the bytes of the states (2.1 MB a run of 64 heads, read and written).
#include "linear_scan.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kRun = 64;         // tokens of a run
constexpr int kCols = 64;        // value columns of a block
constexpr int kMaxK = 128;       // key channels at most
constexpr int kVRow = kCols + 4; // floats of a staged row: rows 4 apart lie 16 banks apart
constexpr int kGRow = kRun + 4;
constexpr int kFormThreads = 256;
constexpr int kReadThreads = 512;

// Where a token stands in its run, for one head.
struct RunTimes {
  float hi[kRun], lo[kRun];   // c_t
  float step[kRun];           // dt_t (0 behind the run's end)
  float grown[kRun];          // exp(c_t)
  float end;                  // exp(c_end)
};

// One wave fills `times` for head h and a run of n tokens; `raw` is its lane's raw step size.  Returns the lane's c_t.
__device__ __forceinline__ double run_times(const ScanArgs& a, RunTimes& times, int h, int n, float raw) {
  const int lane = threadIdx.x % kWave;
  float step = 0.f;
  double c = 0.0;
  if (lane < n) {
    const float z = raw + a.w_bias[h];
    step = z > 20.f ? z : log1pf(expf(z));
    const float l = expf(a.a_log[h]) * step;
    c = l > 110.f ? -110.0 : -(double)l;   // e^-110 is zero in float32; larger ones would take the digits of those behind
  }
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const double before = __shfl_up(c, off, kWave);
    if (lane >= off) c += before;
  }
  const float hi = (float)c;
  times.hi[lane] = hi;
  times.lo[lane] = (float)(c - (double)hi);
  times.step[lane] = step;
  times.grown[lane] = expf(hi);
  return c;
}

// n rows of `wide` floats (a multiple of 4) at src, ld apart, into rows of `stride` floats; rows n .. 63 become zeros.
template <int THREADS>
__device__ __forceinline__ void stage_rows(float* dst, int stride, const float* src, long ld, int n, int wide) {
  const int per = wide / 4;
  for (int e = threadIdx.x; e < kRun * per; e += THREADS) {
    const int row = e / per, c = (e - row * per) * 4;
    float4 v = {0.f, 0.f, 0.f, 0.f};
    if (row < n) v = *reinterpret_cast<const float4*>(src + (size_t)row * ld + c);
    *reinterpret_cast<float4*>(dst + row * stride + c) = v;
  }
}

// grid (places, H / heads, column blocks): B and exp(c_end) of `heads` heads that share their keys, one after the other.
__global__ void __launch_bounds__(kFormThreads) scan_form_kernel(ScanArgs a, int heads) {
  extern __shared__ __align__(16) float lds[];
  __shared__ RunTimes times;
  const int K = a.K, V = a.V, ks = K + 4;
  float* k_rows = lds;                  // [64][ks]
  float* v_rows = lds + kRun * ks;      // [64][kVRow]
  int seq, run, runs;
  if (!scan_place(a, blockIdx.x, seq, run, runs) || runs < 2) return;
  if (a.slot_of_seq[seq] < 0) return;
  const int t0 = a.cu_seqlens[seq] + run * kRun, n = min(kRun, a.cu_seqlens[seq + 1] - t0);
  const size_t place = (size_t)(a.cu_seqlens[seq] / kRun + seq + run);
  const int h0 = blockIdx.y * heads, col0 = blockIdx.z * kCols;
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave, side = lane % 16, quarter = lane / 16;
  stage_rows<kFormThreads>(k_rows, ks, a.k + (size_t)t0 * a.ldk + (size_t)(h0 / a.k_div) * K, a.ldk, n, K);
  constexpr int VN = kRun * kCols / 4 / kFormThreads;
  float4 v_next[VN];
  float raw_next = 0.f;
  const auto fetch = [&](int h) {
#pragma unroll
    for (int u = 0; u < VN; ++u) {
      const int e = tid + u * kFormThreads, row = e / (kCols / 4), c = e % (kCols / 4) * 4;
      v_next[u] = float4{0.f, 0.f, 0.f, 0.f};
      if (row < n && col0 + c < V)
        v_next[u] = *reinterpret_cast<const float4*>(a.v + (size_t)(t0 + row) * a.ldv + (size_t)h * V + col0 + c);
    }
    if (wave == 0 && lane < n) raw_next = a.w[(size_t)(t0 + lane) * a.ldw + h];
  };
  fetch(h0);
  for (int hh = 0; hh < heads; ++hh) {
    const int h = h0 + hh;
    if (hh) __syncthreads();            // the head before has been read
#pragma unroll
    for (int u = 0; u < VN; ++u) {
      const int e = tid + u * kFormThreads;
      *reinterpret_cast<float4*>(v_rows + e / (kCols / 4) * kVRow + e % (kCols / 4) * 4) = v_next[u];
    }
    if (wave == 0) {
      const double c = run_times(a, times, h, n, raw_next), end = __shfl(c, kWave - 1, kWave);
      times.grown[lane] = expf((float)(end - c)) * times.step[lane];   // here: what of the token is left at the end
      if (lane == 0) times.end = expf((float)end);
    }
    __syncthreads();
    if (hh + 1 < heads) fetch(h + 1);
    const size_t at = place * a.H + h;
    if (tid == 0 && col0 == 0) a.run_decay[at] = times.end;
    for (int rt = wave; rt * 16 < K; rt += kFormThreads / kWave) {
      f32x4 acc[kCols / 16];
#pragma unroll
      for (int j = 0; j < kCols / 16; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
      for (int u = 0; u < kRun / 4; ++u) {
        const int t = 16 * (u / 4) + 4 * quarter + u % 4;   // this lane's token of the four
        const float x = k_rows[t * ks + 16 * rt + side] * times.grown[t];
#pragma unroll
        for (int j = 0; j < kCols / 16; ++j)
          acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, v_rows[t * kVRow + 16 * j + side], acc[j], 0, 0, 0);
      }
      float* B = a.run_state + at * K * V;
#pragma unroll
      for (int j = 0; j < kCols / 16; ++j) {
        const int col = col0 + 16 * j + side;
        if (col < V)
#pragma unroll
          for (int i = 0; i < 4; ++i) B[(size_t)(16 * rt + 4 * quarter + i) * V + col] = acc[j][i];
      }
    }
  }
}

// Per request and four neighbouring entries of S: the state before every run takes the place of its B, the state behind
// the last goes to the slot.
__global__ void __launch_bounds__(256) scan_join_kernel(ScanArgs a) {
  const int seq = blockIdx.x, h = blockIdx.y;
  const int e = (blockIdx.z * 256 + threadIdx.x) * 4;
  if (e >= a.K * a.V) return;
  const int slot = a.slot_of_seq[seq];
  const int t0 = a.cu_seqlens[seq], len = a.cu_seqlens[seq + 1] - t0;
  if (slot < 0 || len <= kRun) return;
  const int runs = (len + kRun - 1) / kRun;
  const size_t first = ((size_t)(t0 / kRun + seq) * a.H + h), state = (size_t)a.K * a.V;
  float* B = a.run_state + first * state + e;
  const float* decay = a.run_decay + first;
  float* own = a.state + (size_t)slot * a.slot_stride + a.state_off + (size_t)h * state + e;
  float S[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) S[i] = own[i];
  constexpr int kAhead = 4;
  for (int j0 = 0; j0 < runs; j0 += kAhead) {
    float4 b[kAhead];
    float d[kAhead];
#pragma unroll
    for (int c = 0; c < kAhead; ++c) {
      const int j = min(j0 + c, runs - 1);
      b[c] = *reinterpret_cast<const float4*>(B + (size_t)j * a.H * state);
      d[c] = decay[(size_t)j * a.H];
    }
#pragma unroll
    for (int c = 0; c < kAhead; ++c) {
      if (j0 + c < runs) {
        *reinterpret_cast<float4*>(B + (size_t)(j0 + c) * a.H * state) = float4{S[0], S[1], S[2], S[3]};
        S[0] = d[c] * S[0] + b[c].x;
        S[1] = d[c] * S[1] + b[c].y;
        S[2] = d[c] * S[2] + b[c].z;
        S[3] = d[c] * S[3] + b[c].w;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) own[i] = S[i];
}

// grid (places, H / heads, column blocks): the outputs of `heads` heads that share r and k, one after the other.  A wave
// owns 16 tokens and 32 columns.
__global__ void __launch_bounds__(kReadThreads) scan_read_kernel(ScanArgs a, int heads) {
  extern __shared__ __align__(16) float lds[];
  __shared__ RunTimes times;
  const int K = a.K, V = a.V, ks = K + 4;
  float* r_rows = lds;                        // [64][ks]
  float* scores = r_rows + kRun * ks;         // [64][kGRow]
  float* v_rows = scores + kRun * kGRow;      // [64][kVRow]
  float* s_rows = v_rows + kRun * kVRow;      // [K][kVRow]; the keys [64][ks] until the scores are formed
  int seq, run, runs;
  if (!scan_place(a, blockIdx.x, seq, run, runs) || runs < 2) return;
  const int t0 = a.cu_seqlens[seq] + run * kRun, n = min(kRun, a.cu_seqlens[seq + 1] - t0);
  const size_t place = (size_t)(a.cu_seqlens[seq] / kRun + seq + run);
  const int h0 = blockIdx.y * heads, col0 = blockIdx.z * kCols;
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave, side = lane % 16, quarter = lane / 16;
  if (a.slot_of_seq[seq] < 0) {               // padding: its output is never read
    for (int e = tid; e < n * heads * kCols; e += kReadThreads) {
      const int c = col0 + e % kCols, h = h0 + e / kCols % heads;
      if (c < V) a.out[(size_t)(t0 + e / kCols / heads) * a.ldo + (size_t)h * V + c] = 0.f;
    }
    return;
  }
  constexpr int VN = kRun * kCols / 4 / kReadThreads, SN = kMaxK * kCols / 4 / kReadThreads;
  float4 v_next[VN], s_next[SN];
  float raw_next = 0.f;
  const auto fetch = [&](int h) {
#pragma unroll
    for (int u = 0; u < SN; ++u) {
      const int e = tid + u * kReadThreads, row = e / (kCols / 4), c = e % (kCols / 4) * 4;
      s_next[u] = float4{0.f, 0.f, 0.f, 0.f};
      if (row < K && col0 + c < V)
        s_next[u] = *reinterpret_cast<const float4*>(a.run_state + (place * a.H + h) * K * V + (size_t)row * V + col0 + c);
    }
#pragma unroll
    for (int u = 0; u < VN; ++u) {
      const int e = tid + u * kReadThreads, row = e / (kCols / 4), c = e % (kCols / 4) * 4;
      v_next[u] = float4{0.f, 0.f, 0.f, 0.f};
      if (row < n && col0 + c < V)
        v_next[u] = *reinterpret_cast<const float4*>(a.v + (size_t)(t0 + row) * a.ldv + (size_t)h * V + col0 + c);
    }
    if (wave == 0 && lane < n) raw_next = a.w[(size_t)(t0 + lane) * a.ldw + h];
  };
  stage_rows<kReadThreads>(r_rows, ks, a.r + (size_t)t0 * a.ldr + (size_t)(h0 / a.r_div) * K, a.ldr, n, K);
  stage_rows<kReadThreads>(s_rows, ks, a.k + (size_t)t0 * a.ldk + (size_t)(h0 / a.k_div) * K, a.ldk, n, K);
  fetch(h0);
  __syncthreads();
  // the scores, tiles on and below the diagonal: tile (1, 0) is number 1, (1, 1) 2, (2, 0) 3, ...
  for (int tile = wave; tile < 10; tile += kReadThreads / kWave) {
    const int mt = tile >= 6 ? 3 : tile >= 3 ? 2 : tile >= 1 ? 1 : 0, nt = tile - mt * (mt + 1) / 2;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int u = 0; u < K / 16; ++u) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(r_rows + (16 * mt + side) * ks + 16 * u + 4 * quarter);
      const f32x4 y = *reinterpret_cast<const f32x4*>(s_rows + (16 * nt + side) * ks + 16 * u + 4 * quarter);
#pragma unroll
      for (int t = 0; t < 4; ++t) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[t], y[t], acc, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) scores[(16 * mt + 4 * quarter + i) * kGRow + 16 * nt + side] = acc[i];
  }
  const int mt = wave / 2, j0 = wave % 2 * 2;
  const int row = 16 * mt + side;             // the token whose scores this lane brings
  for (int hh = 0; hh < heads; ++hh) {
    const int h = h0 + hh;
    __syncthreads();                          // the keys, and the head before, have been read
#pragma unroll
    for (int u = 0; u < SN; ++u) {
      const int e = tid + u * kReadThreads;
      if (e / (kCols / 4) < K) *reinterpret_cast<float4*>(s_rows + e / (kCols / 4) * kVRow + e % (kCols / 4) * 4) = s_next[u];
    }
#pragma unroll
    for (int u = 0; u < VN; ++u) {
      const int e = tid + u * kReadThreads;
      *reinterpret_cast<float4*>(v_rows + e / (kCols / 4) * kVRow + e % (kCols / 4) * 4) = v_next[u];
    }
    if (wave == 0) run_times(a, times, h, n, raw_next);
    __syncthreads();
    if (hh + 1 < heads) fetch(h + 1);
    f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    for (int u = 0; u < K / 16; ++u) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(r_rows + row * ks + 16 * u + 4 * quarter);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const float* s = s_rows + (16 * u + 4 * quarter + t) * kVRow + 16 * j0 + side;
        acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[t], s[0], acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[t], s[16], acc[1], 0, 0, 0);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float grown = times.grown[16 * mt + 4 * quarter + i];
      acc[0][i] *= grown;
      acc[1][i] *= grown;
    }
    const float hi = times.hi[row], lo = times.lo[row];
    // the diagonal tile's values hold no infinity or NaN: their products with zero are zeros
    float zeros = 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const float* v = v_rows + (16 * mt + 4 * quarter + t) * kVRow + 16 * j0 + side;
      zeros += fmaf(v[0], 0.f, v[16] * 0.f);
    }
    const bool whole = __builtin_expect(__all(zeros == 0.f), 1);
    const int tiles = whole ? mt + 1 : mt;
    for (int u = 0; u < tiles; ++u) {
      const f32x4 g = *reinterpret_cast<const f32x4*>(scores + row * kGRow + 16 * u + 4 * quarter);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int i = 16 * u + 4 * quarter + t;
        const float x = i <= row ? g[t] * times.step[i] * expf((hi - times.hi[i]) + (lo - times.lo[i])) : 0.f;
        const float* v = v_rows + i * kVRow + 16 * j0 + side;
        acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, v[0], acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, v[16], acc[1], 0, 0, 0);
      }
    }
    if (!whole) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = 16 * mt + 4 * quarter + r;
#pragma unroll 1
        for (int i = 16 * mt; i <= t; ++i) {
          const float x = scores[t * kGRow + i] * times.step[i] * expf((times.hi[t] - times.hi[i]) + (times.lo[t] - times.lo[i]));
          const float* v = v_rows + i * kVRow + 16 * j0 + side;
          acc[0][r] += x * v[0];
          acc[1][r] += x * v[16];
        }
      }
    }
    const float skip = a.skip != nullptr ? a.skip[h] : 0.f;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int c = 16 * (j0 + j) + side;
      if (col0 + c < V)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int t = 16 * mt + 4 * quarter + i;
          if (t < n) a.out[(size_t)(t0 + t) * a.ldo + (size_t)h * V + col0 + c] = acc[j][i] + skip * v_rows[t * kVRow + c];
        }
    }
  }
}

// One decay per head formed from raw steps, r and k shared by the same heads, whole tiles of channels and columns, rows
// that begin at multiples of 16 bytes.
bool scan_runs_takes(const ScanArgs& a) {
  const uintptr_t ends = (uintptr_t)a.r | (uintptr_t)a.k | (uintptr_t)a.v | (uintptr_t)a.run_state;
  return a.run_len == kRun && a.w_mode == 2 && a.bonus == nullptr && a.v_scale == nullptr && a.r_div == a.k_div &&
         a.K % 16 == 0 && a.K >= 64 && a.K <= kMaxK && a.V % 16 == 0 && a.ldr % 4 == 0 && a.ldk % 4 == 0 && a.ldv % 4 == 0 &&
         ends % 16 == 0;
}

int scan_runs_launch(const ScanArgs& a, long need, int tokens, hipStream_t stream) {
  const int blocks_v = (a.V + kCols - 1) / kCols;
  // heads a block: as many as share r and k, up to eight, while every CU keeps two blocks (a request of several runs leaves
  // at most every second one part empty)
  const long busy = min(need, 2L * tokens / kRun);
  int heads = 8;
  while (heads > 1 && (a.r_div % heads || busy * (a.H / heads) * blocks_v < 2L * device_cus())) heads /= 2;
  const dim3 grid((unsigned)need, a.H / heads, blocks_v);
  if (need > 0x7fffffL || a.H > 65535 || blocks_v > 65535) return ATOM_TOO_LARGE;
  const size_t form = (size_t)kRun * (a.K + 4 + kVRow) * sizeof(float);
  const size_t read = ((size_t)kRun * (a.K + 4 + kGRow + kVRow) + (size_t)max(a.K * kVRow, kRun * (a.K + 4))) * sizeof(float);
  const int most = 120 * 1024;
  static bool allowed = false;
  if (!allowed) {
    if (hipFuncSetAttribute((const void*)scan_form_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, most) != hipSuccess ||
        hipFuncSetAttribute((const void*)scan_read_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, most) != hipSuccess)
      return ATOM_LAUNCH_FAILED;
    allowed = true;
  }
  hipLaunchKernelGGL(scan_form_kernel, grid, dim3(kFormThreads), form, stream, a, heads);
  hipLaunchKernelGGL(scan_join_kernel, dim3(a.num_seqs, a.H, (a.K * a.V / 4 + 255) / 256), dim3(256), 0, stream, a);
  hipLaunchKernelGGL(scan_read_kernel, grid, dim3(kReadThreads), read, stream, a, heads);
  return launch_status();
}
