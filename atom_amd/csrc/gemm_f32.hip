// y[M, N] = x[M, K] * w[N, K]^T (+ bias[N]) in true float32: the matrix cores' float32 instructions, every product
// and every sum in 32 bits.  X and W may be float32 or bfloat16 independently (read, widened, multiplied in float32).
//
// K is walked 16 terms at a time.  The 16 are summed apart and join the sum of their slice; K is cut into 8 slices, whose
// sums are added four and four in order, then the two.  That order is the same whatever M is and whichever tile and kernel
// a launch uses, so a row's result does not depend on its batch.
//
// A block is 8 waves, one a slice, all on the same output tile of 16 MT rows and 16 NT columns; a wave reads its
// operands straight from memory into the registers that the matrix instructions take, DEPTH steps ahead of their use
// (no LDS before the slices meet: at 64 x 64 a step's 8 KB feed 64 instructions of 32 cycles, so the caches keep up).
// Few rows are bound by the weights' bytes: one row by 24,576 x 4,096 takes 71 us, 5.6 TB/s.  Many are bound by what the
// loads cost (16 rows of 64 bytes an instruction) and take the kernel with LDS below where its tiles fill the chip, bound by
// the float32 rate of the matrix cores.  (The multiply-add kernel of 64 x 64 tiles that these replaced: the products of two
// 8B layers at 465 rows, once, and at 2 rows, four times, with the heads, took 44 ms, 7.0 now.)
#include "common.h"
#include "lds_loads.h"

constexpr int kSlices = 8;      // slices of K, and waves of a block
constexpr int kStep = 16;       // terms summed apart
constexpr int kXcds = 8;        // dies of the chip, each with an L2 of its own
constexpr int kSide = 16;       // rows and columns of a matrix instruction

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef bf16_t bf16x4 __attribute__((ext_vector_type(4)));

struct GemmF32Params {
  const void* x;
  const void* w;
  const float* bias;
  void* y;
  int m, n, k;
  int row_tiles, tiles;
  int y_bf16;
  int inter;   // SiLU-gate: w holds `inter` gate rows, then as many up rows (n = 2 inter); 0: a plain product
};

// The row of w that stands at column `at` of the output tiles: with a gate every 16 columns are 8 gate rows and the up rows
// of the same 8 columns of y, so that both meet in one place.
__device__ __forceinline__ int row_of_w(const GemmF32Params& p, int at) {
  if (p.inter == 0) return min(at, p.n - 1);
  return min(at / kSide * 8 + at % 8, p.inter - 1) + (at % kSide < 8 ? 0 : p.inter);
}

__device__ __forceinline__ float silu_times(float gate, float up) { return gate / (1.f + expf(-gate)) * up; }

// How a row's terms are read, four at a time.  kWhole: K is a multiple of 16 and rows begin at multiples of four elements in
// memory.  kAny: any K from 4 on and any rows, with loads that need no more than their elements' alignment; the four that would
// reach behind the row's end are its last four, which last_terms moves into place before they are used.  kTerms: term by
// term, for the K below 4.  (4,096 columns at 2,048 rows, K 4,095, bfloat16 x: 1,867 us term by
// term, 795 with loads of four; one row 36 and 17.)
enum Loads : int { kTerms, kAny, kWhole };
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
typedef bf16_t bf16x4_any __attribute__((ext_vector_type(4), aligned(2)));

template <typename T, int LOADS>
__device__ __forceinline__ f32x4 four_terms(const T* __restrict__ row, int k0, int k) {
  f32x4 v;
  if constexpr (LOADS == kTerms) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = k0 + i < k ? to_f32(row[k0 + i]) : 0.f;
  } else if constexpr (sizeof(T) == 4) {
    if constexpr (LOADS == kWhole) v = *reinterpret_cast<const f32x4*>(row + k0);
    else v = *reinterpret_cast<const f32x4_any*>(row + min(k0, k - 4));
  } else {
    bf16x4 h;
    if constexpr (LOADS == kWhole) h = *reinterpret_cast<const bf16x4*>(row + k0);
    else h = *reinterpret_cast<const bf16x4_any*>(row + min(k0, k - 4));
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = to_f32(h[i]);
  }
  return v;
}

// The terms from k0 on of what four_terms<kAny> read: `late` (1 to 3, or more for none) of the four were read too early, and
// zeros stand behind the row's end.
__device__ __forceinline__ void last_terms(f32x4& v, int late) {
  if (late & 1) v = f32x4{v[1], v[2], v[3], 0.f};
  if (late & 2) v = f32x4{v[2], v[3], 0.f, 0.f};
  if (late > 3) v = f32x4{0.f, 0.f, 0.f, 0.f};
}

template <typename TX, typename TW, int MT, int NT, int DEPTH, int LOADS>
__global__ void __launch_bounds__(kSlices* kWave)
gemm_f32_kernel(GemmF32Params p) {
  __shared__ float met[kSlices][MT * kSide * kSide];
  const int tid = threadIdx.x;
  const int wave = tid / kWave;
  const int lane = tid % kWave;
  const int side = lane % kSide;       // the row of x and the row of w whose terms this lane brings
  const int quarter = lane / kSide;    // which 4 of a step's 16 terms
  // blocks go to the chip's XCDs in turn: each XCD gets a range of columns, with all their rows one after the other, so
  // that weights are read into one L2 only
  const int tile = blockIdx.x % kXcds * (gridDim.x / kXcds) + blockIdx.x / kXcds;
  if (tile >= p.tiles) return;
  const int row0 = tile % p.row_tiles * (MT * kSide);
  const int col0 = tile / p.row_tiles * (NT * kSide);
  // rows and columns beyond the end read the last one; their results are not written
  const TX* xr[MT];
  const TW* wr[NT];
#pragma unroll
  for (int i = 0; i < MT; ++i) xr[i] = (const TX*)p.x + (size_t)min(row0 + i * kSide + side, p.m - 1) * p.k;
#pragma unroll
  for (int j = 0; j < NT; ++j) wr[j] = (const TW*)p.w + (size_t)row_of_w(p, col0 + j * kSide + side) * p.k;

  const int steps = (p.k + kStep - 1) / kStep;
  const int share = (steps + kSlices - 1) / kSlices;
  const int begin = min(wave * share, steps);
  const int count = __builtin_amdgcn_readfirstlane(min(begin + share, steps) - begin);

  const int ends = __builtin_amdgcn_readfirstlane(p.k / kStep - begin);   // kAny: the step that the row ends in

  f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // The largest tile asks for a later step's operands in every step, the last ones for the last step's again: with loads
  // in all paths alike the compiler knows how many are in flight and waits for the oldest only (1,024 x 4,096 x 4,096:
  // 388 us without, 336 with).  The small tiles are bound by what the loads cost and ask for nothing twice.
  constexpr bool kSteady = MT * NT >= 16;
  f32x4 a[DEPTH][MT], b[DEPTH][NT];
  const auto fetch = [&](int d, int step) {
    const int at = min(begin + min(step, max(count - 1, 0)), steps - 1) * kStep + quarter * 4;
#pragma unroll
    for (int j = 0; j < NT; ++j) b[d][j] = four_terms<TW, LOADS>(wr[j], at, p.k);
#pragma unroll
    for (int i = 0; i < MT; ++i) a[d][i] = four_terms<TX, LOADS>(xr[i], at, p.k);
  };
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) {
    if (kSteady || d < count) fetch(d, d);
    __builtin_amdgcn_sched_barrier(0);
  }
  for (int base = 0; base < count; base += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      if (base + d < count) {
        if constexpr (LOADS == kAny) {
          if (base + d == ends) {
            const int late = max(p.k / kStep * kStep + quarter * 4 - (p.k - 4), 0);
#pragma unroll
            for (int i = 0; i < MT; ++i) last_terms(a[d][i], late);
#pragma unroll
            for (int j = 0; j < NT; ++j) last_terms(b[d][j], late);
          }
        }
        // term by term over all tiles: an instruction's sum is needed only MT NT instructions later
        f32x4 part[MT][NT];
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
              part[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                  a[d][i][t], b[d][j][t], t ? part[i][j] : f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[i][j][t] += part[i][j][t];
      }
      __builtin_amdgcn_sched_barrier(0);
      if (kSteady || base + d + DEPTH < count) fetch(d, base + d + DEPTH);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // the slices' sums meet, 16 columns at a time
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    if (j) __syncthreads();
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int t = 0; t < 4; ++t) met[wave][(i * kSide + quarter * 4 + t) * kSide + side] = acc[i][j][t];
    __syncthreads();
    const auto sum_of = [&](int e) {
      float sum = 0.f;
#pragma unroll
      for (int half = 0; half < kSlices; half += kSlices / 2) {
        float part = met[half][e];
#pragma unroll
        for (int s = 1; s < kSlices / 2; ++s) part += met[half + s][e];
        sum = half ? sum + part : part;
      }
      return sum;
    };
    if (p.inter != 0) {
      for (int e = tid; e < MT * kSide * 8; e += kSlices * kWave) {
        const int r = row0 + e / 8, c = (col0 + j * kSide) / 2 + e % 8;
        if (r >= p.m || c >= p.inter) continue;
        float gate = sum_of(e / 8 * kSide + e % 8), up = sum_of(e / 8 * kSide + 8 + e % 8);
        if (p.bias != nullptr) gate += p.bias[c], up += p.bias[p.inter + c];
        ((float*)p.y)[(size_t)r * p.inter + c] = silu_times(gate, up);
      }
      continue;
    }
    for (int e = tid; e < MT * kSide * kSide; e += kSlices * kWave) {
      const int r = row0 + e / kSide, c = col0 + j * kSide + e % kSide;
      if (r >= p.m || c >= p.n) continue;
      float sum = sum_of(e);
      if (p.bias != nullptr) sum += p.bias[c];
      if (p.y_bf16)
        ((bf16_t*)p.y)[(size_t)r * p.n + c] = from_f32<bf16_t>(sum);
      else
        ((float*)p.y)[(size_t)r * p.n + c] = sum;
    }
  }
}

// Many rows, float32 operands, K a multiple of 16: tiles of 64 rows and 128 columns whose operands go through LDS, in whole
// cache lines straight from memory.  A block is two groups of four waves, each with four of the slices, a wave with 32 x 64
// of the tile.  A stage is 32 terms of the tile's 192 rows, double buffered; the eight 16-byte pieces of a row change
// places by its row number, so that the 16 rows a wave reads at once lie in different banks.  465 rows by 24,576 x 4,096
// take 932 us, 100 TFLOP/s (1,039 in tiles of 64 x 64 without LDS), by 4,096 x 4,096 157 (177); 1,024 rows 110 TFLOP/s
// (102).
constexpr int kWideRows = 64, kWideCols = 128, kWideStage = 32;
constexpr int kStageFloats = (kWideRows + kWideCols) * kWideStage;

__global__ void __launch_bounds__(kSlices* kWave) gemm_f32_wide_kernel(GemmF32Params p) {
  extern __shared__ __align__(16) float wide[];   // [group][buffer][kStageFloats]
  const int tile = blockIdx.x % kXcds * (gridDim.x / kXcds) + blockIdx.x / kXcds;
  if (tile >= p.tiles) return;
  const int row0 = tile % p.row_tiles * kWideRows;
  const int col0 = tile / p.row_tiles * kWideCols;
  const int tid = threadIdx.x, lane = tid % kWave, side = lane % kSide, quarter = lane / kSide;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave), group = wave / 4, w4 = wave % 4;
  const int r0 = w4 % 2 * 32, c0 = kWideRows + w4 / 2 * 64;   // the wave's first row and column among the staged rows

  const int steps = p.k / kStep;
  const int share = (steps + kSlices - 1) / kSlices;
  const int low = min(steps, 4 * share);
  const int count = group ? steps - low : low;      // this group's steps
  const int stages = (low + 1) / 2;
  const int k0 = group ? low * kStep : 0;

  // piece `lane % 8` of row 8 (6 w4 + j) + lane / 8 in LDS holds the row's piece of that number turned by the row
  constexpr int LOADS = (kWideRows + kWideCols) / 8 / 4;
  const float* from[LOADS];
  int at[LOADS];
#pragma unroll
  for (int j = 0; j < LOADS; ++j) {
    const int r = 8 * (LOADS * w4 + j) + lane / 8;
    from[j] = r < kWideRows ? (const float*)p.x + (size_t)min(row0 + r, p.m - 1) * p.k
                            : (const float*)p.w + (size_t)row_of_w(p, col0 + r - kWideRows) * p.k;
    at[j] = k0 + (lane % 8 ^ (r >> 1 & 7)) * 4;
  }
  float* mine = wide + group * 2 * kStageFloats;
  const auto fetch = [&](int buffer, int stage) {
#pragma unroll
    for (int j = 0; j < LOADS; ++j)   // pieces behind the row's end: its last again, never used
      load_to_lds(from[j] + min(at[j] + stage * kWideStage, p.k - 4),
                  lds_address(mine + buffer * kStageFloats + (LOADS * w4 + j) * 8 * kWideStage));
  };
  const auto piece = [&](const float* buffer, int r, int half) {
    return *reinterpret_cast<const f32x4*>(buffer + r * kWideStage + ((4 * half + quarter) ^ (r >> 1 & 7)) * 4);
  };
  f32x4 acc[2][4], total[2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = total[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  fetch(0, 0);
  int until = share;                                // steps until the slice ends
  for (int stage = 0; stage < stages; ++stage) {
    arrived();
    lds_barrier();                                  // the stage is there, the one before has been read
    if (stage + 1 < stages) fetch(stage + 1 & 1, stage + 1);
    const float* buffer = mine + (stage & 1) * kStageFloats;
    f32x4 a2[2][2], b2[2][4];                       // both halves' operands at once: one wait for LDS a stage
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
      for (int i = 0; i < 2; ++i) a2[half][i] = piece(buffer, r0 + 16 * i + side, half);
#pragma unroll
      for (int j = 0; j < 4; ++j) b2[half][j] = piece(buffer, c0 + 16 * j + side, half);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      if (2 * stage + half < count) {
        const f32x4(&a)[2] = a2[half];
        const f32x4(&b)[4] = b2[half];
        f32x4 part[2][4];
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
              part[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][t], b[j][t], t ? part[i][j] : f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[i][j][t] += part[i][j][t];
        if (--until == 0 || 2 * stage + half + 1 == count) {
          until = share;
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
#pragma unroll
              for (int t = 0; t < 4; ++t) total[i][j][t] += acc[i][j][t];
              acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
        }
      }
    }
  }

  // the second group's half of the sum joins the first's
  __syncthreads();
  float* met = wide + w4 * 32 * 64;                 // the wave's 32 x 64
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        float* there = met + (16 * i + 4 * quarter + t) * 64 + 16 * j + side;
        if (group) *there = total[i][j][t];
      }
  __syncthreads();
  if (group) return;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int at = col0 + c0 - kWideRows + 16 * j + side;
      const int c = p.inter == 0 ? at : at / kSide * 8 + side % 8;     // the column of y
      if (c >= (p.inter == 0 ? p.n : p.inter)) continue;               // (gate and up lanes of a column go together)
      const float bias = p.bias != nullptr ? p.bias[c + (p.inter != 0 && side >= 8 ? p.inter : 0)] : 0.f;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int r = row0 + r0 + 16 * i + 4 * quarter + t;
        if (r >= p.m) continue;
        float sum = total[i][j][t] + met[(16 * i + 4 * quarter + t) * 64 + 16 * j + side];
        if (p.bias != nullptr) sum += bias;
        if (p.inter != 0) {
          const float up = __shfl_xor(sum, 8);
          if (side < 8) ((float*)p.y)[(size_t)r * p.inter + c] = silu_times(sum, up);
        } else if (p.y_bf16) {
          ((bf16_t*)p.y)[(size_t)r * p.n + c] = from_f32<bf16_t>(sum);
        } else {
          ((float*)p.y)[(size_t)r * p.n + c] = sum;
        }
      }
    }
}

static int launch_gemm_f32_wide(GemmF32Params p, hipStream_t stream) {
  p.row_tiles = (p.m + kWideRows - 1) / kWideRows;
  const long tiles = (long)p.row_tiles * ((p.n + kWideCols - 1) / kWideCols);
  if (tiles > 0x3fffffL) return ATOM_TOO_LARGE;
  p.tiles = (int)tiles;
  constexpr int bytes = 4 * kStageFloats * sizeof(float);
  static bool allowed = false;
  if (!allowed) {
    if (hipFuncSetAttribute((const void*)gemm_f32_wide_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess)
      return ATOM_LAUNCH_FAILED;
    allowed = true;
  }
  hipLaunchKernelGGL(gemm_f32_wide_kernel, dim3((unsigned)(tiles + kXcds - 1) / kXcds * kXcds), dim3(kSlices * kWave), bytes,
                     stream, p);
  return launch_status();
}

template <typename TX, typename TW, int MT, int NT, int DEPTH>
static int launch_gemm_f32(GemmF32Params p, hipStream_t stream) {
  p.row_tiles = (p.m + MT * kSide - 1) / (MT * kSide);
  const long tiles = (long)p.row_tiles * ((p.n + NT * kSide - 1) / (NT * kSide));
  if (tiles > 0x3fffffL) return ATOM_TOO_LARGE;   // 2^31 threads
  p.tiles = (int)tiles;
  const dim3 grid((unsigned)(tiles + kXcds - 1) / kXcds * kXcds), block(kSlices * kWave);
  const bool whole = p.k % kStep == 0 && (uintptr_t)p.x % (4 * sizeof(TX)) == 0 && (uintptr_t)p.w % (4 * sizeof(TW)) == 0;
  if (whole)
    hipLaunchKernelGGL((gemm_f32_kernel<TX, TW, MT, NT, DEPTH, kWhole>), grid, block, 0, stream, p);
  else if (MT * NT < 16 || p.k >= 4)
    hipLaunchKernelGGL((gemm_f32_kernel<TX, TW, MT, NT, DEPTH, kAny>), grid, block, 0, stream, p);
  else if constexpr (MT * NT == 16)
    hipLaunchKernelGGL((gemm_f32_kernel<TX, TW, MT, NT, DEPTH, kTerms>), grid, block, 0, stream, p);
  return launch_status();
}

template <typename TX, typename TW>
static int choose_gemm_f32(const GemmF32Params& p, hipStream_t stream) {
  // Tiles two wide read x half as often, which pays from where there is one for most CUs on.  24,576 x 4,096, narrow and
  // wide: 16 rows 111 and 93 us, 32 rows 155 and 116; 4,096 x 12,288 (128
  // wide tiles): 32 rows 89 and 116 us.
  if (p.k < 4) return launch_gemm_f32<TX, TW, 4, 4, 2>(p, stream);
  const long cus = device_cus();
  const bool wide_fills = p.n / 32 >= cus * 3 / 4;
  if (p.m <= 16) {
    if (p.m > 4 && wide_fills) return launch_gemm_f32<TX, TW, 1, 2, 6>(p, stream);
    return launch_gemm_f32<TX, TW, 1, 1, 8>(p, stream);
  }
  if (p.m <= 32) {
    if (wide_fills) return launch_gemm_f32<TX, TW, 2, 2, 3>(p, stream);
    return launch_gemm_f32<TX, TW, 2, 1, 6>(p, stream);
  }
  // 64 rows: the width whose rounds over the CUs take least, a round's time being about 13, 22, 40 and, through LDS, 64
  // for 16, 32, 64 and 128 columns (465 rows by 6,144 x 4,096: 384 of the widest tiles are two rounds, 317 us, 768 tiles of
  // 64 three shorter ones, 272)
  const long rows = (p.m + 63) / 64;
  const auto cost = [&](int cols, int round) { return (rows * ((p.n + cols - 1) / cols) + cus - 1) / cus * round; };
  const long c1 = cost(16, 13), c2 = cost(32, 22), c4 = cost(64, 40), c8 = cost(128, 64);
  if constexpr (sizeof(TX) == 4 && sizeof(TW) == 4) {
    const bool whole = p.k % kStep == 0 && ((uintptr_t)p.x | (uintptr_t)p.w) % 16 == 0;
    if (p.m > 64 && whole && c8 <= c4 && c8 <= c2 && c8 <= c1) return launch_gemm_f32_wide(p, stream);
  }
  if (c1 <= c2 && c1 <= c4) return launch_gemm_f32<TX, TW, 4, 1, 4>(p, stream);
  if (c2 <= c4) return launch_gemm_f32<TX, TW, 4, 2, 3>(p, stream);
  return launch_gemm_f32<TX, TW, 4, 4, 2>(p, stream);
}

ATOM_EXPORT int atom_gemm_f32(const void* x, int x_dtype, const void* w, int w_dtype, const float* bias, void* y,
                              int y_dtype, int m, int n, int k, hipStream_t stream) {
  if (m < 0 || n <= 0 || k <= 0) return ATOM_BAD_SHAPE;
  if ((unsigned)x_dtype > 1u || (unsigned)w_dtype > 1u || (unsigned)y_dtype > 1u) return ATOM_BAD_DTYPE;
  if (m == 0) return ATOM_OK;
  const GemmF32Params p{x, w, bias, y, m, n, k, 0, 0, y_dtype == ATOM_BF16, 0};
  switch (x_dtype * 2 + w_dtype) {
    case 0: return choose_gemm_f32<float, float>(p, stream);
    case 1: return choose_gemm_f32<float, bf16_t>(p, stream);
    case 2: return choose_gemm_f32<bf16_t, float>(p, stream);
    default: return choose_gemm_f32<bf16_t, bf16_t>(p, stream);
  }
}

// y[M, inter] = silu(x wg^T + bg) * (x wu^T + bu), float32, for w of `inter` gate rows and then as many up rows: the sums of
// the plain product, gated where they are written instead of in a launch of their own that reads them back.
ATOM_EXPORT int atom_gemm_f32_gate(const void* x, int x_dtype, const void* w, int w_dtype, const float* bias, float* y, int m,
                                   int inter, int k, hipStream_t stream) {
  if (m < 0 || inter <= 0 || inter > 0x3fffffff || k <= 0) return ATOM_BAD_SHAPE;
  if ((unsigned)x_dtype > 1u || (unsigned)w_dtype > 1u) return ATOM_BAD_DTYPE;
  if (m == 0) return ATOM_OK;
  const GemmF32Params p{x, w, bias, y, m, 2 * inter, k, 0, 0, 0, inter};
  switch (x_dtype * 2 + w_dtype) {
    case 0: return choose_gemm_f32<float, float>(p, stream);
    case 1: return choose_gemm_f32<float, bf16_t>(p, stream);
    case 2: return choose_gemm_f32<bf16_t, float>(p, stream);
    default: return choose_gemm_f32<bf16_t, bf16_t>(p, stream);
  }
}
