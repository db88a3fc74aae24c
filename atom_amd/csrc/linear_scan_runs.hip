// A linear recurrence with one decay per head over runs of 64 tokens, as products of the matrix cores' float32
// instructions.  With c_t the sum of the logarithms of a run's decays up to token t, S the state before the run, k_t, r_t,
// v_t as in linear_scan.hip and dt_t the step sizes,
//
//   what the run adds     B = sum_t exp(c_end - c_t) dt_t k_t v_t^T
//   its outputs           o_t = exp(c_t) S^T r_t + sum_{i <= t} exp(c_t - c_i) dt_i (r_t . k_i) v_i   (+ skip v_t)
//
// in three launches: the decays of every run and head; per request the states before its runs (and the one after the last, which
// goes to the slot), run by run; the outputs of all runs side by side.  The scores r_t . k_i do not depend on the head where
// heads share r and k: a block takes several such heads and forms the scores once.
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
// Heads of 128 x 64, the three launches against forming B of every run, joining them into states in a second launch and
// reading by blocks that staged a head at a time (and a walk token by token before that: 263 + 80 + 486 us), us: 5,569 tokens of
// four requests, 64 heads 6 + 105 + 137 and 99 + 81 + 202; one request of 2,048, 64 heads 5 + 42 + 61 and 51 + 22 + 78, 32 heads
// 5 + 39 + 45 and 30 + 13 + 48; 70 tokens of 32 heads 4 + 6 + 12 and 10 + 4 + 14; eight of 1,000, 128 heads 13 + 238 + 352 and
// 269 + 204 + 578.  The states of the runs were written, read, written and read again (2.1 MB a run of 64 heads); the walk writes
// them once, and they stand as the reading lanes take them.  What bounds the walk is issuing a run's loads, stores and LDS
// accesses beside its 32 or 64 matrix instructions a wave (1.2 and 1.8 us a run, the instructions 0.4 and 0.85), the reading
// its products (0.4 of the float32 rate of the matrix cores) and what a block does before its first head.
#include "linear_scan.h"
#include <type_traits>

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kRun = 64;         // tokens of a run
constexpr int kCols = 64;        // value columns of a reading block
constexpr int kMaxK = 128;       // key channels at most
constexpr int kMaxHeads = 8;     // heads of a reading block at most
constexpr int kWRow = 64 + 4;    // floats of a row the walk stages: rows 4 apart lie 16 banks apart
constexpr int kWalkThreads = 256;
constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;
constexpr double kLog2E = 1.4426950408889634;

// Where the tokens of a run stand in it, for one head; in memory kScanRunTimes floats a (place, head).
struct RunTimes {
  float hi[kRun], lo[kRun];   // c_t to base 2; of the last token behind the run's end
  float step[kRun];           // dt_t (0 behind the run's end)
  float left[kRun];           // dt_t times what is left of token t at the run's end
};
static_assert(sizeof(RunTimes) == kScanRunTimes * sizeof(float));

// grid (places, H / 4): a wave a run and head.
__global__ void __launch_bounds__(256) scan_times_kernel(ScanArgs a) {
  int seq, run, runs;
  if (!scan_place(a, blockIdx.x, seq, run, runs) || runs < 2 || a.slot_of_seq[seq] < 0) return;
  const int lane = threadIdx.x % kWave, h = blockIdx.y * 4 + threadIdx.x / kWave;
  if (h >= a.H) return;
  const int t0 = a.cu_seqlens[seq] + run * kRun, n = min(kRun, a.cu_seqlens[seq + 1] - t0);
  float step = 0.f;
  double c = 0.0;
  if (lane < n) {
    const float z = a.w[(size_t)(t0 + lane) * a.ldw + h] + a.w_bias[h];
    step = z > 20.f ? z : log1pf(expf(z));
    const float l = expf(a.a_log[h]) * step;
    c = kLog2E * (l > 110.f ? -110.0 : -(double)l);   // e^-110 is zero in float32; larger ones would take the digits of those behind
  }
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const double before = __shfl_up(c, off, kWave);
    if (lane >= off) c += before;
  }
  const double end = __shfl(c, kWave - 1, kWave);
  RunTimes& to = reinterpret_cast<RunTimes*>(a.run_decay)[((size_t)(a.cu_seqlens[seq] / kRun + seq + run)) * a.H + h];
  const float hi = (float)c;
  to.hi[lane] = hi;
  to.lo[lane] = (float)(c - (double)hi);
  to.step[lane] = step;
  to.left[lane] = exp2f((float)(end - c)) * step;
}

// The state before a run stands in memory as the lanes that read it take it: by tiles of 16 channels x 16 columns, tile
// (i, j) with V / 16 tiles in a row being 64 lanes' four floats, lane (side, quarter) column `side`, channels 4 quarter ...
__device__ __forceinline__ size_t state_tile(const ScanArgs& a, size_t place, int h, int i, int j) {
  return (place * a.H + h) * a.K * a.V + (size_t)(i * (a.V / 16) + j) * 256;
}

// Per request and head the states before its runs, and the one behind the last, which goes to the slot.  No entry of the state
// depends on another one: a block owns 64 channels x 32 CT columns of them, a wave 2 x CT tiles in registers, and walks the
// request's runs; the rows of the runs ahead wait in registers and, the next run's, in the other of two LDS buffers.
// grid (H x requests, blocks of columns and channels).
template <int CT>
__global__ void __launch_bounds__(kWalkThreads, 2) scan_walk_kernel(ScanArgs a) {
  constexpr int C = 32 * CT, VRow = C + 4;
  __shared__ __align__(16) float k_rows[2][kRun * kWRow], v_rows[2][kRun * VRow];
  __shared__ __align__(16) float left[2][kRun];
  const int h = blockIdx.x % a.H, seq = blockIdx.x / a.H;
  const int slot = a.slot_of_seq[seq];
  const int t0 = a.cu_seqlens[seq], len = a.cu_seqlens[seq + 1] - t0;
  if (slot < 0 || len <= kRun) return;
  const int runs = (len + kRun - 1) / kRun;
  const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave), side = lane % 16, quarter = lane / 16;
  const int K = a.K, V = a.V, blocks_v = (V + C - 1) / C;
  const int ch0 = blockIdx.y / blocks_v * 64, col0 = blockIdx.y % blocks_v * C;
  const int i0 = wave / 2 * 32, j0 = wave % 2 * 16 * CT;     // the wave's first channel and column of the block's
  const size_t first = (size_t)(t0 / kRun + seq);
  const RunTimes* times = reinterpret_cast<const RunTimes*>(a.run_decay) + first * a.H + h;
  // What a thread brings: groups of four floats of k and of v, a row to neighbouring threads.  (No branch around a load, or the
  // compiler waits for all of them: rows behind the request's end are its last one and become zeros on their way into LDS,
  // channels and columns behind the head's are its first ones and are not kept.)
  constexpr int NK = kRun * 64 / 4 / kWalkThreads, NV = kRun * C / 4 / kWalkThreads;
  const int kc4 = tid % 16 * 4, krow = tid / 16, vc4 = tid % (C / 4) * 4, vrow = tid / (C / 4);
  const float* kp = a.k + (size_t)t0 * a.ldk + (size_t)(h / a.k_div) * K;
  const float* vp = a.v + (size_t)t0 * a.ldv + (size_t)h * V;
  const unsigned kc = ch0 + kc4 < K ? ch0 + kc4 : 0, vc = col0 + vc4 < V ? col0 + vc4 : 0, ldk = (unsigned)a.ldk, ldv = (unsigned)a.ldv;
  f32x4 kn[2][NK], vn[2][NV];
  float left_next[2], hi_next[2], lo_next[2];   // (lane 63's hi and lo are the run's end: a scalar load's wait would be one for all of LDS)
  const auto fetch_times = [&](int run, auto which) {
    constexpr int set = which;
    const RunTimes& of = times[(size_t)run * a.H];
    left_next[set] = of.left[lane];
    hi_next[set] = of.hi[lane];
    lo_next[set] = of.lo[lane];
  };
  const auto fetch = [&](int run, int u, auto which) {   // group u of the thread's into register set `which`
    constexpr int set = which;
    const int last = len - 1 - run * kRun;
    if (u < NK) {
      const unsigned t = min(krow + u * (kWalkThreads / 16), last);
      kn[set][u] = *reinterpret_cast<const f32x4*>(kp + (size_t)run * kRun * a.ldk + (t * ldk + kc));
    }
    if (u < NV) {
      const unsigned t = min(vrow + u * (kWalkThreads * 4 / C), last);
      vn[set][u] = *reinterpret_cast<const f32x4*>(vp + (size_t)run * kRun * a.ldv + (t * ldv + vc));
    }
  };
  float* own = a.state + (size_t)slot * a.slot_stride + a.state_off + (size_t)h * K * V;
  f32x4 S[2][CT];
  const auto live = [&](int x, int y) { return ch0 + i0 + 16 * x < K && col0 + j0 + 16 * y < V; };   // (whole tiles)
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < CT; ++y) {
      S[x][y] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (live(x, y))
#pragma unroll
        for (int r = 0; r < 4; ++r) S[x][y][r] = own[(size_t)(ch0 + i0 + 16 * x + 4 * quarter + r) * V + col0 + j0 + 16 * y + side];
    }
  float end[2];
  const auto stage = [&](int run, int u, auto which) {   // group u of run `run` into buffer `which`
    constexpr int set = which;
    const auto put = [&](f32x4& x, int row, float* at) {
      if (len < (run + 1) * kRun) {
        const bool in = run * kRun + row < len;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = in ? x[e] : 0.f;
      }
      *reinterpret_cast<f32x4*>(at) = x;
    };
    if (u < NK) {
      const int row = krow + u * (kWalkThreads / 16);
      put(kn[set][u], row, &k_rows[set][row * kWRow + kc4]);
    }
    if (u < NV) {
      const int row = vrow + u * (kWalkThreads * 4 / C);
      put(vn[set][u], row, &v_rows[set][row * VRow + vc4]);
    }
  };
  const auto stage_times = [&](auto which) {
    constexpr int set = which;
    left[set][lane] = left_next[set];             // (all waves the same)
    end[set] = exp2f(__shfl(hi_next[set] + lo_next[set], kRun - 1, kWave));
  };
  constexpr std::integral_constant<int, 0> even;
  constexpr std::integral_constant<int, 1> odd;
#pragma unroll
  for (int u = 0; u < NK; ++u) fetch(0, u, even);
  fetch_times(0, even);
#pragma unroll
  for (int u = 0; u < NK; ++u) fetch(1, u, odd);   // (there are two runs at least)
  fetch_times(1, odd);
  __builtin_amdgcn_s_waitcnt(0x0f70);        // vmcnt(0): what is asked for so far is waited for once, and not in every run
#pragma unroll
  for (int u = 0; u < NK; ++u) {
    stage(0, u, even);
    fetch(min(2, runs - 1), u, even);
  }
  stage_times(even);
  fetch_times(min(2, runs - 1), even);
  __syncthreads();
  float* tiles = a.run_state + state_tile(a, first, h, (ch0 + i0) / 16, (col0 + j0) / 16) + 4 * lane;
  const size_t per_run = (size_t)a.H * K * V;
  // A run from buffer `which`.  Storing the state before it, staging the next run and asking for the third further on are dealt
  // out among the products: put before them they took half of a run's 1.9 us.
  const auto walk = [&](int run, auto which, auto other) {
    constexpr int buffer = which;
    const int next = min(run + 1, runs - 1), third = min(run + 3, runs - 1);
    const auto piece = [&](int step) {
      if (step < 2 * CT) {
        if (live(step / CT, step % CT))
          *reinterpret_cast<f32x4*>(tiles + (step / CT * (V / 16) + step % CT) * 256) = S[step / CT][step % CT];
      } else if (step >= 4 && step < 4 + NK) {
        stage(next, step - 4, other);
      } else if (step == 4 + NK) {
        stage_times(other);
      } else if (step > 4 + NK && step < 5 + 2 * NK) {
        fetch(third, step - 5 - NK, other);
      } else if (step == 5 + 2 * NK) {
        fetch_times(third, other);
      }
    };
    static_assert(NV <= NK && 5 + 2 * NK < 16);
    const float* kr = k_rows[buffer] + i0 + side;
    const float* vr = v_rows[buffer] + j0 + side;
    f32x4 add[2][CT];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < CT; ++y) add[x][y] = f32x4{0.f, 0.f, 0.f, 0.f};
    float k[2][2][4], v[2][CT][4];                   // a step's entries, read while the step before is multiplied
    f32x4 f[2];
    const auto read = [&](int u) {
      f[u % 2] = *reinterpret_cast<const f32x4*>(&left[buffer][16 * u + 4 * quarter]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int t = 16 * u + 4 * quarter + e;
#pragma unroll
        for (int x = 0; x < 2; ++x) k[u % 2][x][e] = kr[t * kWRow + 16 * x];
#pragma unroll
        for (int y = 0; y < CT; ++y) v[u % 2][y][e] = vr[t * VRow + 16 * y];
      }
    };
    read(0);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (u + 1 < 4) read(u + 1);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        __builtin_amdgcn_sched_barrier(0);
        piece(4 * u + e);
#pragma unroll
        for (int y = 0; y < CT; ++y) {
          const float by = v[u % 2][y][e] * f[u % 2][e];
#pragma unroll
          for (int x = 0; x < 2; ++x) add[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[u % 2][x][e], by, add[x][y], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < CT; ++y)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[x][y][r] = end[buffer] * S[x][y][r] + add[x][y][r];
    tiles += per_run;
    __syncthreads();             // the next run's rows are there, this one's have been read
  };
  int run = 0;
  for (; run + 1 < runs; run += 2) {
    walk(run, even, odd);
    walk(run + 1, odd, even);
  }
  if (run < runs) walk(run, even, odd);
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < CT; ++y)
      if (live(x, y))
#pragma unroll
        for (int r = 0; r < 4; ++r) own[(size_t)(ch0 + i0 + 16 * x + 4 * quarter + r) * V + col0 + j0 + 16 * y + side] = S[x][y][r];
}

// n rows of K floats at src, ld apart, into rows of K + 4 floats; rows n .. 63 become zeros.
template <int K>
__device__ __forceinline__ void stage_rows(float* dst, const float* src, long ld, int n) {
  constexpr int per = K / 4;
  for (int e = threadIdx.x; e < kRun * per; e += kThreads) {
    const int row = e / per, c = (e - row * per) * 4;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (row < n) v = *reinterpret_cast<const f32x4*>(src + (size_t)row * ld + c);
    *reinterpret_cast<f32x4*>(dst + row * (K + 4) + c) = v;
  }
}

constexpr int kTriangle = 10;    // tiles of 16 x 16 tokens on and below the diagonal: (0, 0), (1, 0), (1, 1), (2, 0), ...
constexpr int kTile = 256;       // floats of a tile as the matrix cores' lanes take it: lane (side, quarter) row `side`, 4 quarter ...

template <int K>
struct ReadLds {
  static constexpr int R = K + 4;
  static constexpr int r = 0;                                // [64][R]
  static constexpr int keys = r + kRun * R;                  // [64][R]; once the scores are formed: these, and two heads' weights
  static constexpr int scores = keys;
  static constexpr int weights = scores + kTriangle * kTile;
  static constexpr int times = keys + (kRun * R > 3 * kTriangle * kTile ? kRun * R : 3 * kTriangle * kTile);
  static constexpr int total = times + kMaxHeads * 3 * kRun; // hi, lo, step
};

// grid (places, H / heads, column blocks): the outputs of `heads` heads (up to eight) that share r and k, one after the other.
// A wave owns 16 columns and all tokens of the run; a head's state and values come straight into the registers that the products
// take them from, while the head before is worked on.  The weights of the run's tokens (scores, steps and decays) are the same
// for all columns: the waves form the next head's together, in LDS.  77 KB of LDS: two blocks a CU.
template <int K>
__global__ void __launch_bounds__(kThreads, 2) scan_read_kernel(ScanArgs a, int heads) {
  using At = ReadLds<K>;
  extern __shared__ __align__(16) float lds[];
  float *r_rows = lds + At::r, *keys = lds + At::keys, *scores = lds + At::scores, *weights = lds + At::weights, *times = lds + At::times;
  int seq, run, runs;
  if (!scan_place(a, blockIdx.x, seq, run, runs) || runs < 2) return;
  const int V = a.V;
  const int t0 = a.cu_seqlens[seq] + run * kRun, n = min(kRun, a.cu_seqlens[seq + 1] - t0);
  const size_t place = (size_t)(a.cu_seqlens[seq] / kRun + seq + run);
  const int h0 = blockIdx.y * heads, col0 = blockIdx.z * kCols;
  const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave), side = lane % 16, quarter = lane / 16;
  if (a.slot_of_seq[seq] < 0) {               // padding: its output is never read
    for (int e = tid; e < n * heads * kCols; e += kThreads) {
      const int c = col0 + e % kCols, h = h0 + e / kCols % heads;
      if (c < V) a.out[(size_t)(t0 + e / kCols / heads) * a.ldo + (size_t)h * V + c] = 0.f;
    }
    return;
  }
  const int j = wave, col = col0 + 16 * j + side;
  const bool has = col0 + 16 * j < V;         // (whole tiles of columns)
  f32x4 S[K / 16];
  float v[16];
  const float* vp = a.v + (size_t)t0 * a.ldv + (has ? col : 0);
  const auto fetch_state = [&](int h, int u) {
    S[u] = *reinterpret_cast<const f32x4*>(a.run_state + state_tile(a, place, h, u, has ? col0 / 16 + j : 0) + 4 * lane);
  };
  const auto fetch_values = [&](int h) {
#pragma unroll
    for (int t = 0; t < 16; ++t)
      v[t] = vp[(unsigned)(min(16 * (t / 4) + 4 * quarter + t % 4, n - 1) * (int)a.ldv + h * V)];
  };
#pragma unroll
  for (int u = 0; u < K / 16; ++u) fetch_state(h0, u);
  fetch_values(h0);
  const float skips = a.skip != nullptr && lane < heads ? a.skip[h0 + lane] : 0.f;
  for (int e = tid; e < heads * 3 * kRun; e += kThreads) {
    const int hh = e / (3 * kRun);
    times[e] = a.run_decay[(place * a.H + h0 + hh) * kScanRunTimes + e - hh * 3 * kRun];
  }
  stage_rows<K>(r_rows, a.r + (size_t)t0 * a.ldr + (size_t)(h0 / a.r_div) * K, a.ldr, n);
  stage_rows<K>(keys, a.k + (size_t)t0 * a.ldk + (size_t)(h0 / a.k_div) * K, a.ldk, n);
  __syncthreads();
  // the scores.  Their rows are the lanes' sides: a lane's four lie side by side
  const auto place_of = [](int t, int& mt, int& nt) {
    mt = t >= 6 ? 3 : t >= 3 ? 2 : t >= 1 ? 1 : 0;
    nt = t - mt * (mt + 1) / 2;
  };
  constexpr int kMine = (kTriangle + kWaves - 1) / kWaves;
  f32x4 tile[kMine];
#pragma unroll
  for (int x = 0; x < kMine; ++x) {
    tile[x] = f32x4{0.f, 0.f, 0.f, 0.f};
    int mt, nt;
    place_of(min(wave + x * kWaves, kTriangle - 1), mt, nt);
#pragma unroll 4
    for (int u = 0; u < K / 16; ++u) {
      const f32x4 rr = *reinterpret_cast<const f32x4*>(r_rows + (16 * mt + side) * At::R + 16 * u + 4 * quarter);
      const f32x4 kk = *reinterpret_cast<const f32x4*>(keys + (16 * nt + side) * At::R + 16 * u + 4 * quarter);
#pragma unroll
      for (int t = 0; t < 4; ++t) tile[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[t], rr[t], tile[x], 0, 0, 0);
    }
  }
  __syncthreads();                            // the keys have been read
#pragma unroll
  for (int x = 0; x < kMine; ++x)
    if (wave + x * kWaves < kTriangle) *reinterpret_cast<f32x4*>(scores + (wave + x * kWaves) * kTile + 4 * lane) = tile[x];
  // token t's weight of token i: score, step and decay; zero above the diagonal
  const auto form_weights = [&](int hh, int x) {
    const float *his = times + hh * 3 * kRun, *los = his + kRun, *steps = los + kRun;
    {
      if (wave + x * kWaves < kTriangle) {    // (the wave's own scores)
        int mt, nt;
        place_of(wave + x * kWaves, mt, nt);
        const int row = 16 * mt + side, col = 16 * nt + 4 * quarter;
        const float hi = his[row], lo = los[row];
        const f32x4 step = *reinterpret_cast<const f32x4*>(steps + col);
        const f32x4 h4 = *reinterpret_cast<const f32x4*>(his + col), l4 = *reinterpret_cast<const f32x4*>(los + col);
        f32x4 w;
#pragma unroll
        for (int t = 0; t < 4; ++t)
          w[t] = col + t <= row ? tile[x][t] * step[t] * __builtin_amdgcn_exp2f((hi - h4[t]) + (lo - l4[t])) : 0.f;
        *reinterpret_cast<f32x4*>(weights + (hh & 1) * kTriangle * kTile + (wave + x * kWaves) * kTile + 4 * lane) = w;
      }
    }
  };
#pragma unroll
  for (int x = 0; x < kMine; ++x) form_weights(0, x);
  for (int hh = 0; hh < heads; ++hh) {
    const int h = h0 + hh, next = h0 + min(hh + 1, heads - 1);
    const float *his = times + hh * 3 * kRun, *los = his + kRun, *steps = los + kRun;
    const float* mine = weights + (hh & 1) * kTriangle * kTile;
    __syncthreads();                          // this head's weights are there, those of the head before have been used
    f32x4 acc[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
    f32x4 x[2][4];
    const auto read = [&](int u) {
#pragma unroll
      for (int m = 0; m < 4; ++m) x[u % 2][m] = *reinterpret_cast<const f32x4*>(r_rows + (16 * m + side) * At::R + 16 * u + 4 * quarter);
    };
    read(0);
#pragma unroll
    for (int u = 0; u < K / 16; ++u) {
      if (u + 1 < K / 16) read(u + 1);
      __builtin_amdgcn_sched_barrier(0);
      if (u < kMine && hh + 1 < heads) form_weights(hh + 1, u);
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int m = 0; m < 4; ++m) acc[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[u % 2][m][t], S[u][t], acc[m], 0, 0, 0);
      fetch_state(next, u);
    }
    const float skip = __shfl(skips, hh, kWave);
    f32x4 g[2];
    g[0] = *reinterpret_cast<const f32x4*>(mine + 4 * lane);
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      const f32x4 hi4 = *reinterpret_cast<const f32x4*>(his + 16 * mt + 4 * quarter);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[mt][i] *= __builtin_amdgcn_exp2f(hi4[i]);
      // the diagonal tile's values: where they hold no infinity or NaN their products with zero are zeros
      const float zeros = fmaf(v[4 * mt], 0.f, v[4 * mt + 1] * 0.f) + fmaf(v[4 * mt + 2], 0.f, v[4 * mt + 3] * 0.f);
      const bool whole = __builtin_expect(__all(zeros == 0.f), 1);
#pragma unroll
      for (int u = 0; u <= mt; ++u) {
        constexpr auto number = [](int m, int n) { return m * (m + 1) / 2 + n; };
        const int now = number(mt, u);
        if (now + 1 < kTriangle) g[(now + 1) % 2] = *reinterpret_cast<const f32x4*>(mine + (now + 1) * kTile + 4 * lane);
        if (u < mt || whole)
#pragma unroll
          for (int t = 0; t < 4; ++t) acc[mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(g[now % 2][t], v[4 * u + t], acc[mt], 0, 0, 0);
      }
      if (!whole) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int t = 16 * mt + 4 * quarter + r;
#pragma unroll 1
          for (int i = 16 * mt; i <= min(t, n - 1); ++i) {
            const int q = i - 16 * mt;
            const float w = mine[(mt * (mt + 1) / 2 + mt) * kTile + (q / 4 * 16 + 4 * quarter + r) * 4 + q % 4];
            acc[mt][r] += w * vp[(size_t)i * a.ldv + (size_t)h * V];
          }
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = 16 * mt + 4 * quarter + i;
        if (has && t < n) a.out[(size_t)(t0 + t) * a.ldo + (size_t)h * V + col] = acc[mt][i] + skip * v[4 * mt + i];
      }
    }
    fetch_values(next);
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

template <int K>
static int launch_read(const ScanArgs& a, const dim3& grid, int heads, hipStream_t stream) {
  constexpr size_t bytes = ReadLds<K>::total * sizeof(float);
  static bool allowed = false;
  if (!allowed) {
    if (hipFuncSetAttribute((const void*)scan_read_kernel<K>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess)
      return ATOM_LAUNCH_FAILED;
    allowed = true;
  }
  hipLaunchKernelGGL(scan_read_kernel<K>, grid, dim3(kThreads), bytes, stream, a, heads);
  return launch_status();
}

int scan_runs_launch(const ScanArgs& a, long need, int tokens, hipStream_t stream) {
  const int blocks_v = (a.V + kCols - 1) / kCols;
  // heads a block, of those that share r and k: what a block does before its first head is about a head's time, and two blocks a
  // CU work at a time (5,569 tokens of four requests, 64 heads: 157 us with eight a block, which is one round and a half, 137 with four)
  const long busy = min(need, (long)tokens / kRun + 1), slots = 2L * device_cus();
  int heads = 1;
  double least = 0.0;
  for (int some = kMaxHeads; some >= 1; some /= 2) {
    if (a.r_div % some) continue;
    const long rounds = (busy * (a.H / some) * blocks_v + slots - 1) / slots;
    const double time = rounds * (some + 0.8);
    if (least == 0.0 || time < least) heads = some, least = time;
  }
  const dim3 grid((unsigned)need, a.H / heads, blocks_v);
  // columns a block of the walk: 64, or 32 where blocks of 64 would leave CUs idle (one request of 2,048 tokens, 64 heads of
  // 128 x 64: 42 us with 32 and 58 with 64)
  const int blocks_k = (a.K + 63) / 64;
  const bool narrow = min((long)a.num_seqs, tokens / (kRun + 1L)) * a.H * blocks_k * blocks_v < device_cus();
  const int squares = blocks_k * (narrow ? (a.V + 31) / 32 : blocks_v);
  if (need > 0x7fffffL || a.H > 65535 || squares > 65535 || (long)a.H * a.num_seqs > 0x7fffffffL) return ATOM_TOO_LARGE;
  hipLaunchKernelGGL(scan_times_kernel, dim3((unsigned)need, (a.H + 3) / 4), dim3(256), 0, stream, a);
  hipLaunchKernelGGL(narrow ? scan_walk_kernel<1> : scan_walk_kernel<2>, dim3((unsigned)(a.H * a.num_seqs), squares), dim3(kWalkThreads), 0, stream, a);
  switch (a.K) {
    case 64: return launch_read<64>(a, grid, heads, stream);
    case 80: return launch_read<80>(a, grid, heads, stream);
    case 96: return launch_read<96>(a, grid, heads, stream);
    case 112: return launch_read<112>(a, grid, heads, stream);
    case 128: return launch_read<128>(a, grid, heads, stream);
    default: return ATOM_UNSUPPORTED;
  }
}
