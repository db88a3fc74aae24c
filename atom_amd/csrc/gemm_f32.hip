// y[M, N] = x[M, K] * w[N, K]^T (+ bias[N]) with float32 operands and float32 sums (X and W may be float32 or bfloat16
// independently), on the matrix cores' bfloat16 instructions, whose rate is sixteen times that of the float32 ones.
//
// A float32 value is the sum of three bfloat16 pieces, hi + mid + lo, each the rounded rest of what the pieces before it
// leave: 3 x 8 bits hold its 24.  A product of two values is the six products of pieces that reach its last bits (hi lo, lo
// hi, mid mid, hi mid, mid hi, hi hi; the three left out are below 2^-24 of it, a rounding of float32, at most, and a
// sixth of the sums' own roundings on average), each exact in float32 and added there.  An operand that is bfloat16 is one
// piece.  A float32 operand is split times 2^24, and the sums are taken back as they join: float32 values are multiples of
// 2^-149, so all pieces of any of them are then normal bfloat16 values (without that the pieces of operands below 2^-110 lose
// bits, which the results show where the other operand is large).  What this takes from the other end, operands from 2^104 and
// sums of 32 terms from 2^80 on, comes out as an infinity or a NaN, as infinities do themselves (a piece behind one is a NaN);
// results that are not finite are summed again by the float32 instructions.
//
// K is walked 32 terms at a time.  The 32 are summed apart, smallest pieces first, and join the sum of their slice; K is cut
// into 8 slices, whose sums are added four and four in order, then the two.  That order is the same whatever M is and
// whichever tile and kernel a launch uses, so a row's result does not depend on its batch.  Against float64 (random normal
// operands, 2-norm of the difference over that of the result): 9.9e-8 at K 4,096 (with one operand in bfloat16 the same, with
// both 9.6e-8) and 1.43e-7 at 12,288, where the float32 instructions' sums of 16 terms are 1.38e-7 and 2.00e-7 off.
//
// A block is 8 waves, one a slice, all on the same output tile of 16 MT rows and 16 NT columns; a wave reads its
// operands straight from memory into the registers that the matrix instructions take, DEPTH steps ahead of their use
// (no LDS before the slices meet).  Few rows are bound by the weights' bytes: one row by 24,576 x 4,096 takes 70 us, 5.8 TB/s
// (71 with the float32 instructions), 8 rows 72 (83), 32 rows 98 (117).  Many rows take the kernel with LDS below where its
// tiles fill the chip and K is a multiple of 32; else 465 rows by 24,576 x 4,112 take 804 us (952), by 4,096 x 4,112 133 (160).
// What splitting costs shows where the bytes come from caches or are few: one row by 1,024 x 1,024 5.3 us (4.9), x 1,040 5.7
// (4.9), by 4,096 x 4,096 read again and again 13.6 (12.8), 300 rows by 4,096 x 96 14.9 (12.2), by 4,096 x 8 1.2 times as long.
#include "common.h"
#include "lds_loads.h"

#include <type_traits>

constexpr int kSlices = 8;      // slices of K, and waves of a block
constexpr int kStep = 32;       // terms summed apart
constexpr int kLane = 8;        // of them, those a lane brings
constexpr int kXcds = 8;        // dies of the chip, each with an L2 of its own
constexpr int kSide = 16;       // rows and columns of a matrix instruction

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef bf16_t bf16x4 __attribute__((ext_vector_type(4)));
typedef bf16_t bf16x8 __attribute__((ext_vector_type(8)));

struct GemmF32Params {
  const void* x;
  const void* w;
  const float* bias;
  void* y;
  int m, n, k;
  int row_tiles, tiles;
  int y_bf16;
  const bf16_t* pieces;   // the wide kernel: x's pieces [m, k / 32, 3, 32]
  int inter;   // SiLU-gate: w holds `inter` gate rows, then as many up rows (n = 2 inter); 0: a plain product
};

// The row of w that stands at column `at` of the output tiles: with a gate every 16 columns are 8 gate rows and the up rows
// of the same 8 columns of y, so that both meet in one place.
__device__ __forceinline__ int row_of_w(int n, int inter, int at) {
  if (inter == 0) return min(at, n - 1);
  return min(at / kSide * 8 + at % 8, inter - 1) + (at % kSide < 8 ? 0 : inter);
}
__device__ __forceinline__ int row_of_w(const GemmF32Params& p, int at) { return row_of_w(p.n, p.inter, at); }

__device__ __forceinline__ float silu_times(float gate, float up) { return gate / (1.f + expf(-gate)) * up; }

// The pieces of a value; an operand that is bfloat16 has one.
template <typename T>
constexpr int kPieces = sizeof(T) == 4 ? 3 : 1;

constexpr float kUp = 0x1p24f;   // what a float32 operand is split times
template <typename T>
constexpr float kDown = sizeof(T) == 4 ? 0x1p-24f : 1.f;

// (Two values at a time, e and e + 1 of a lane's: the instruction that rounds takes two, and their widened pieces are its
// result's halves.)
__device__ __forceinline__ void pieces_of_two(float a, float b, bf16x8 (&p)[3], int e) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef bf16_t bf16x2 __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const bf16x2 both = __builtin_convertvector(f32x2{a, b}, bf16x2);
    p[i][e] = both[0];
    p[i][e + 1] = both[1];
    const unsigned bits = __builtin_bit_cast(unsigned, both);
    a -= __uint_as_float(bits << 16);
    b -= __uint_as_float(bits & 0xffff0000u);
  }
}

// The products of pieces that are formed, smallest first: (piece of x, piece of w).
template <int PX, int PW>
struct Products;
template <>
struct Products<3, 3> {
  static constexpr int count = 6, x[6] = {0, 2, 1, 0, 1, 0}, w[6] = {2, 0, 1, 1, 0, 0};
};
template <>
struct Products<3, 1> {
  static constexpr int count = 3, x[3] = {2, 1, 0}, w[3] = {0, 0, 0};
};
template <>
struct Products<1, 3> {
  static constexpr int count = 3, x[3] = {0, 0, 0}, w[3] = {2, 1, 0};
};
template <>
struct Products<1, 1> {
  static constexpr int count = 1, x[1] = {0}, w[1] = {0};
};

// The matrix instruction cuts its 32 products off below the largest one's last bits, downwards whatever their sign: a mean
// error of its own, the same in all rows, which an average over rows (of values, by attention) does not take down with it.
// Every other step of K is therefore formed from x's negatives and subtracted (without that 1.21e-7 and 1.87e-7 in the figures
// above, but 9.1e-7 for 4.6e-7 in attention's averages over 300 rows).
__device__ __forceinline__ unsigned flip_of(int step) { return step & 1 ? 0x80000000u : 0u; }
template <typename TX, typename TW>
__device__ __forceinline__ float factor_of(int step) {
  return step & 1 ? -kDown<TX> * kDown<TW> : kDown<TX> * kDown<TW>;
}

// How a row's terms are read, four at a time.  kWhole: K is a multiple of 32 and rows begin at multiples of 16 bytes in
// memory.  kAny: any K from 4 on and any rows, with loads that need no more than their elements' alignment; the four that would
// reach behind the row's end are its last four, which last_terms moves into place before they are used.  kTerms: term by
// term, for the K below 4.
enum Loads : int { kTerms, kAny, kWhole };
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
typedef bf16_t bf16x4_any __attribute__((ext_vector_type(4), aligned(2)));

// A lane's eight terms as they lie in memory: of a step's 32 terms from `k0` on lane quarter q brings four from 4 q on and four
// from 16 + 4 q on, so that the quarters' reads lie side by side.  Operands agree on that order, which is all it takes.
__device__ __forceinline__ int quad_at(int quarter, int h) { return 16 * h + 4 * quarter; }

template <typename T>
struct Terms {
  typedef typename std::conditional<sizeof(T) == 4, f32x4, bf16x4>::type Quad;
  typedef typename std::conditional<sizeof(T) == 4, f32x4_any, bf16x4_any>::type QuadAny;
  Quad q[2];

  template <int LOADS>
  __device__ __forceinline__ void read(const T* __restrict__ row, int k0, int quarter, int k) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int at = k0 + quad_at(quarter, h);
      if constexpr (LOADS == kWhole) {
        q[h] = *reinterpret_cast<const Quad*>(row + at);
      } else if constexpr (LOADS == kAny) {
        q[h] = *reinterpret_cast<const QuadAny*>(row + min(at, k - 4));
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) q[h][i] = at + i < k ? row[at + i] : from_f32<T>(0.f);
      }
    }
  }
  // After read<kAny> of the step from k0 on: four that were read too early (up to 3 places, or more for those that lie
  // behind the row's end altogether) move into place, with zeros behind them.
  __device__ __forceinline__ void last_terms(int k0, int quarter, int k) {
    const T zero = from_f32<T>(0.f);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int late = max(k0 + quad_at(quarter, h) - (k - 4), 0);
      if (late & 1) q[h] = Quad{q[h][1], q[h][2], q[h][3], zero};
      if (late & 2) q[h] = Quad{q[h][2], q[h][3], zero, zero};
      if (late > 3) q[h] = Quad{zero, zero, zero, zero};
    }
  }
  // `flip`: the sign bit, or 0; with it the pieces are those of the terms' negatives.  (float32: of the terms times kUp.)
  __device__ __forceinline__ void pieces(bf16x8 (&p)[kPieces<T>], unsigned flip = 0) const {
    if constexpr (sizeof(T) == 4) {
      const float up = __uint_as_float(__float_as_uint(kUp) ^ flip);
#pragma unroll
      for (int e = 0; e < kLane; e += 2) pieces_of_two(q[e / 4][e % 4] * up, q[e / 4][e % 4 + 1] * up, p, e);
    } else {
      typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
      const bf16x8 all = __builtin_shufflevector(q[0], q[1], 0, 1, 2, 3, 4, 5, 6, 7);
      p[0] = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, all) ^ (flip | flip >> 16));
    }
  }
};

// Whether a result is one of those that pieces may have spoilt.
__device__ __forceinline__ bool spoilt(float v) { return !(fabsf(v) < INFINITY); }

// 16 rows and columns summed by the float32 instructions, in the kernels' steps and slices: lane (side, quarter) brings row `side` of
// both operands and receives column `side` of rows 4 quarter .. + 3.  (One lane a result, term by term: 465 rows by 24,576 x 4,096
// 2,600 us with one row of NaN and 91 ms with nothing else.)
template <int LOADS, typename TX, typename TW>
__device__ __noinline__ f32x4 summed_again(const TX* x, const TW* w, int quarter, int k) {
  constexpr int DEPTH = 2;
  const int steps = (k + kStep - 1) / kStep, share = (steps + kSlices - 1) / kSlices;
  Terms<TX> a[DEPTH];
  Terms<TW> b[DEPTH];
  const auto fetch = [&](int d, int step) {
    if (step >= steps) return;
    a[d].template read<LOADS>(x, step * kStep, quarter, k);
    b[d].template read<LOADS>(w, step * kStep, quarter, k);
  };
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) fetch(d, d);
  f32x4 total = {0.f, 0.f, 0.f, 0.f}, half = total, sum = total;
  int until = share, slice = 0;
#pragma unroll 1
  for (int base = 0; base < steps; base += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      const int step = base + d;
      if (step >= steps) break;
      if (LOADS == kAny && step == k / kStep) {
        a[d].last_terms(step * kStep, quarter, k);
        b[d].last_terms(step * kStep, quarter, k);
      }
      f32x4 part = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int e = 0; e < kLane; ++e)
        part = __builtin_amdgcn_mfma_f32_16x16x4f32(to_f32(a[d].q[e / 4][e % 4]), to_f32(b[d].q[e / 4][e % 4]), part, 0, 0, 0);
      fetch(d, step + DEPTH);
      sum += part;
      if (--until == 0 || step + 1 == steps) {
        until = share;
        half += sum;
        sum = f32x4{0.f, 0.f, 0.f, 0.f};
        if (++slice == kSlices / 2 || step + 1 == steps) {
          total += half;
          half = f32x4{0.f, 0.f, 0.f, 0.f};
        }
      }
    }
  }
  return total;
}

// Row r, column c of what summed_again left in the wave's lanes.
__device__ __forceinline__ float picked(f32x4 sums, int r, int c) {
  float v = 0.f;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const float other = __shfl(sums[t], r / 4 * kSide + c);
    if (r % 4 == t) v = other;
  }
  return v;
}

template <typename TX, typename TW, int MT, int NT, int DEPTH, int LOADS>
__global__ void __launch_bounds__(kSlices* kWave)
gemm_f32_kernel(GemmF32Params p) {
  using Order = Products<kPieces<TX>, kPieces<TW>>;
  __shared__ float met[kSlices][MT * kSide * kSide];
  const int tid = threadIdx.x;
  const int wave = tid / kWave;
  const int lane = tid % kWave;
  const int side = lane % kSide;       // the row of x and the row of w whose terms this lane brings
  const int quarter = lane / kSide;    // which 8 of a step's 32 terms
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
  const int begin = __builtin_amdgcn_readfirstlane(min(wave * share, steps));
  const int count = __builtin_amdgcn_readfirstlane(min(begin + share, steps) - begin);
  const int ends = __builtin_amdgcn_readfirstlane(p.k / kStep - begin);   // kAny: the step that the row ends in

  f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  Terms<TX> a[DEPTH][MT];
  Terms<TW> b[DEPTH][NT];
  const auto fetch = [&](int d, int step) {
    const int at = (begin + step) * kStep;
#pragma unroll
    for (int j = 0; j < NT; ++j) b[d][j].template read<LOADS>(wr[j], at, quarter, p.k);
#pragma unroll
    for (int i = 0; i < MT; ++i) a[d][i].template read<LOADS>(xr[i], at, quarter, p.k);
  };
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) {
    if (d < count) fetch(d, d);
    __builtin_amdgcn_sched_barrier(0);
  }
  for (int base = 0; base < count; base += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      if (base + d < count) {
        if constexpr (LOADS == kAny) {
          if (base + d == ends) {
            const int at = p.k / kStep * kStep;
#pragma unroll
            for (int i = 0; i < MT; ++i) a[d][i].last_terms(at, quarter, p.k);
#pragma unroll
            for (int j = 0; j < NT; ++j) b[d][j].last_terms(at, quarter, p.k);
          }
        }
        const float factor = factor_of<TX, TW>(begin + base + d);
        bf16x8 ap[MT][kPieces<TX>];
#pragma unroll
        for (int i = 0; i < MT; ++i) a[d][i].pieces(ap[i], flip_of(begin + base + d));
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          bf16x8 bp[kPieces<TW>];
          b[d][j].pieces(bp);
          f32x4 part[MT];
#pragma unroll
          for (int t = 0; t < Order::count; ++t)
#pragma unroll
            for (int i = 0; i < MT; ++i)
              part[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ap[i][Order::x[t]], bp[Order::w[t]],
                                                                t ? part[i] : f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[i][j][t] = fmaf(part[i][t], factor, acc[i][j][t]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (base + d + DEPTH < count) fetch(d, base + d + DEPTH);
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
    const auto sum_of = [&](int e) {   // entry e % 16 of row e / 16
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
    // of the 16 rows that hold row r, which a whole wave asks for together
    const auto again = [&](int r) {
      return summed_again<LOADS>((const TX*)p.x + (size_t)min(row0 + r / kSide * kSide + side, p.m - 1) * p.k,
                          (const TW*)p.w + (size_t)row_of_w(p, col0 + j * kSide + side) * p.k, quarter, p.k);
    };
    if (p.inter != 0) {
      for (int e = tid; e < MT * kSide * 8; e += kSlices * kWave) {
        const int r = row0 + e / 8, c = (col0 + j * kSide) / 2 + e % 8;
        float gate = sum_of(e / 8 * kSide + e % 8), up = sum_of(e / 8 * kSide + 8 + e % 8);
        if constexpr (kPieces<TX> * kPieces<TW> > 1) {
          if (__any(spoilt(gate) || spoilt(up))) {
            const f32x4 sums = again(e / 8);
            const float g = picked(sums, e / 8 % kSide, e % 8), u = picked(sums, e / 8 % kSide, 8 + e % 8);
            if (spoilt(gate)) gate = g;
            if (spoilt(up)) up = u;
          }
        }
        if (r >= p.m || c >= p.inter) continue;
        if (p.bias != nullptr) gate += p.bias[c], up += p.bias[p.inter + c];
        ((float*)p.y)[(size_t)r * p.inter + c] = silu_times(gate, up);
      }
      continue;
    }
    for (int e = tid; e < MT * kSide * kSide; e += kSlices * kWave) {
      const int r = row0 + e / kSide, c = col0 + j * kSide + e % kSide;
      float sum = sum_of(e);
      if constexpr (kPieces<TX> * kPieces<TW> > 1) {
        if (__any(spoilt(sum))) {
          const float other = picked(again(e / kSide), e / kSide % kSide, e % kSide);
          if (spoilt(sum)) sum = other;
        }
      }
      if (r >= p.m || c >= p.n) continue;
      if (p.bias != nullptr) sum += p.bias[c];
      if (p.y_bf16)
        ((bf16_t*)p.y)[(size_t)r * p.n + c] = from_f32<bf16_t>(sum);
      else
        ((float*)p.y)[(size_t)r * p.n + c] = sum;
    }
  }
}

// Many rows, float32 operands, K a multiple of 32: tiles of 64 or 128 rows and 128 columns whose operands go through LDS, in
// whole cache lines straight from memory.  x comes in pieces, a row's twelve of a step side by side, made once by a kernel of its
// own; pieces of w are formed where it is multiplied.  A block is two groups of four waves, a wave with 64 x 32 of the tile, so that a step's splitting
// (two of w's 16-row parts) takes a third of the cycles of its 48 matrix instructions; in 32 x 64 it would take more than they
// do.  A stage is 32 terms of the tile's rows, double buffered; the 16-byte pieces of a row change places by its row number, so
// that the rows a wave reads at once lie in different banks.  While a stage is multiplied, the next one's operands are read from
// LDS and the stage behind that comes from memory: 56 KB for two groups of four slices each, 40 KB in tiles of 128 rows, at the
// 35 to 40 KB a microsecond that a CU draws, are what bounds it.  465 rows by 24,576 x 4,096 take 573 us in tiles of 128 rows (938
// with the float32 instructions; 645 in tiles of 64, timed when those were 595), by 4,096 x 4,096, where only the lower ones are a
// tile for every CU, 108 (164), by 4,096 x 12,288 299 (475); 1,024 rows by 24,576 1,120, 184 TFLOP/s (1,873; the float32
// instructions' rate is 157).  (w times 2^24 as it is split is 1 to 2 % of these.  With x's pieces in three planes, a plane's rows
// half a line a step, the four are 600, 112, 310 and 1,151.)
// Five stages in LDS with all eight waves on each (32 x 32 of 64 x 128 a wave) took 705, 120 and 340 at 465 rows.
constexpr int kWideCols = 128;

// ROWS 64: the block's halves take half of K each.  ROWS 128: they take 64 rows each and all of K, and the first four slices'
// sums wait in LDS.
template <int ROWS>
struct Wide {
  static constexpr int groups = 128 / ROWS;                            // of waves that share K
  static constexpr int xs = ROWS * kStep * 6;                          // bytes of x in a stage: rows of three times kStep pieces,
  static constexpr int stage = xs + kWideCols * kStep * 4;             // and of a stage, w behind them
  static constexpr int sums = ROWS * kWideCols * 4;                    // the sums of half of K
  static constexpr int bytes = groups == 2 ? 4 * stage : 2 * stage + sums;
  static_assert(bytes <= 160 * 1024 && bytes >= sums, "it all fits in LDS");
};

__global__ void __launch_bounds__(256) split_f32_kernel(const float* __restrict__ x, bf16_t* __restrict__ pieces, size_t eights,
                                                                  int steps) {
  const size_t at = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (at >= eights) return;
  Terms<float> v;   // four eights a step, in the order of the lanes' quarters
  v.read<kWhole>(x + at / 4 * kStep, 0, at % 4, kStep);
  bf16x8 p[3];
  v.pieces(p, flip_of(at / 4 % steps));
#pragma unroll
  for (int i = 0; i < 3; ++i) *reinterpret_cast<bf16x8*>(pieces + (at / 4 * 12 + 4 * i + at % 4) * kLane) = p[i];
}

// The place of row 16 i + 4 quarter + t, column 16 j + side among a wave's 64 x 32 sums in LDS.
__device__ __forceinline__ int place_of(int i, int j, int t, int quarter, int side) {
  return (16 * i + 4 * quarter + t) * 32 + 16 * j + side;
}

// The wide kernel's: of a wave's 64 x 32 sums in LDS, from row `row0` and column `col0` on, those that pieces may have spoilt.
// (Through LDS, so that the kernel has no registers to keep for it.)
__device__ __noinline__ void sum_again_wide(const float* x, const float* w, int m, int n, int k, int inter, float* sums, int row0, int col0) {
  const int lane = threadIdx.x % kWave, side = lane % kSide, quarter = lane / kSide;
#pragma unroll 1
  for (int i = 0; i < 4; ++i)
#pragma unroll 1
    for (int j = 0; j < 2; ++j) {
      float* own[4];
      bool any = false;
#pragma unroll
      for (int t = 0; t < 4; ++t) own[t] = sums + place_of(i, j, t, quarter, side), any = any || spoilt(*own[t]);
      if (!__any(any)) continue;
      const f32x4 again = summed_again<kWhole>(x + (size_t)min(row0 + 16 * i + side, m - 1) * k,
                                               w + (size_t)row_of_w(n, inter, col0 + 16 * j + side) * k, quarter, k);
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (spoilt(*own[t])) *own[t] = again[t];
    }
}

template <int ROWS>
__global__ void __launch_bounds__(kSlices* kWave) gemm_f32_wide_kernel(GemmF32Params p) {
  constexpr int GROUPS = Wide<ROWS>::groups, kStageBytes = Wide<ROWS>::stage;
  extern __shared__ __align__(16) char wide[];   // [group][buffer][kStageBytes]: x's pieces, then w
  const int tile = blockIdx.x % kXcds * (gridDim.x / kXcds) + blockIdx.x / kXcds;
  if (tile >= p.tiles) return;
  const int row0 = tile % p.row_tiles * ROWS;
  const int col0 = tile / p.row_tiles * kWideCols;
  const int tid = threadIdx.x, lane = tid % kWave, side = lane % kSide, quarter = lane / kSide;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave), w4 = wave % 4;
  const int group = GROUPS == 2 ? wave / 4 : 0, r0 = GROUPS == 2 ? 0 : wave / 4 * 64;   // the wave's share of K, or of the rows

  const int steps = p.k / kStep;
  const int share = (steps + kSlices - 1) / kSlices;
  const int low = GROUPS == 2 ? min(steps, 4 * share) : steps;
  const int count = group ? steps - low : low;      // this group's steps
  const int k0 = group ? low * kStep : 0;

  // Loads of a stage: x, whose rows have twelve 16-byte pieces a step side by side (their place in LDS turned, in fours, by the
  // row), then 8 rows of w each (piece `lane % 8`).
  constexpr int X_LOADS = 3 * ROWS / 16, LOADS = (X_LOADS + kWideCols / 8) * GROUPS / kSlices;
  const int loader = GROUPS == 2 ? w4 : wave;
  const char* from[LOADS];
  int size[LOADS];                                  // bytes of a term
#pragma unroll
  for (int j = 0; j < LOADS; ++j) {
    const int load = LOADS * loader + j;
    if (load < X_LOADS) {
      const int at = load * kWave + lane, r = at / 12, piece = at % 12;
      from[j] = (const char*)p.pieces + ((size_t)min(row0 + r, p.m - 1) * p.k + k0) * 6 + (piece ^ (r >> 1 & 3)) * 16;
      size[j] = 6;
    } else {
      const int r = (load - X_LOADS) * 8 + lane / 8;
      from[j] = (const char*)((const float*)p.w + (size_t)row_of_w(p, col0 + r) * p.k + k0 + (lane % 8 ^ (r >> 1 & 7)) * 4);
      size[j] = 4;
    }
  }
  char* mine = wide + group * 2 * kStageBytes;
  const auto fetch = [&](int buffer, int stage) {   // a group without steps of its own left reads its last stage again
    const int term = min(stage, max(count - 1, 0)) * kStep;
#pragma unroll
    for (int j = 0; j < LOADS; ++j)
      load_to_lds(from[j] + term * size[j], lds_address(mine + buffer * kStageBytes + (LOADS * loader + j) * 1024));
  };
  f32x4 acc[4][2], total[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = total[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  using Order = Products<3, 3>;
  struct Operands {
    bf16x8 a[4][3];
    Terms<float> b[2];
  };
  const auto read = [&](Operands& o, int stage) {
    const char* xs = mine + (stage & 1) * kStageBytes;
    const char* ws = xs + Wide<ROWS>::xs;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int r = 32 * w4 + 16 * j + side;
#pragma unroll
      for (int h = 0; h < 2; ++h)
        o.b[j].q[h] = *reinterpret_cast<const f32x4*>(ws + r * kStep * 4 + ((quad_at(quarter, h) / 4) ^ (r >> 1 & 7)) * 16);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = r0 + 16 * i + side;
#pragma unroll
      for (int t = 0; t < 3; ++t)
        o.a[i][t] = *reinterpret_cast<const bf16x8*>(xs + r * kStep * 6 + (4 * t + (quarter ^ (r >> 1 & 3))) * 16);
    }
  };
  int until = share, slice = 0;                     // steps until the slice ends
  // the first four slices' sums: those of the other half of the block, or the wave's own
  float* met = (float*)(wide + (GROUPS == 2 ? 0 : 2 * kStageBytes)) + (GROUPS == 2 ? w4 : wave) * 64 * 32;
  const auto place = [&](int i, int j, int t) { return place_of(i, j, t, quarter, side); };
  const bool second = GROUPS == 1 && steps > 4 * share;   // there are more slices than four
  const auto multiply = [&](const Operands& o, float factor, bool last) {
    bf16x8 bp[2][3];
    f32x4 part[2][4];
    o.b[0].pieces(bp[0]);
    __builtin_amdgcn_sched_barrier(0);
    // the first half's matrix instructions with the second half's splitting, the second half's with the first half's adding up
    // (in the order of the source, because the compiler splits in one go where registers are short)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int t = 0; t < Order::count; ++t) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          part[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(o.a[i][Order::x[t]], bp[j][Order::w[t]],
                                                               t ? part[j][i] : f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        if (t < 4) {
          if (j == 0) {
            const f32x4 q = o.b[1].q[t / 2];
            pieces_of_two(q[t % 2 * 2] * kUp, q[t % 2 * 2 + 1] * kUp, bp[1], 2 * t);
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[t][0][r] = fmaf(part[0][t][r], factor, acc[t][0][r]);
          }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (j == 0) __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
          else __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);
        }
        if (t == Order::count - 1) __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][1][r] = fmaf(part[1][i][r], factor, acc[i][1][r]);
    if (--until == 0 || last) {
      until = share;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
          for (int t = 0; t < 4; ++t) total[i][j][t] += acc[i][j][t];
          acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
      if (second && ++slice == kSlices / 2) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
#pragma unroll
            for (int t = 0; t < 4; ++t) met[place(i, j, t)] = total[i][j][t];
            total[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
      }
    }
  };
  // A stage's operands are read from LDS while the stage before is multiplied; its buffer then takes the stage after next.
  Operands even, odd;
  if (count > 0) fetch(0, 0);
  arrived();
  lds_barrier();
  if (count > 0) read(even, 0);
  if (count > 1) fetch(1, 1);
  const auto pass = [&](const Operands& now, Operands& next, int stage) {
    arrived();
    lds_barrier();                                  // the next stage is there, and all have read this one
    __builtin_amdgcn_s_waitcnt(0xc07f);             // (the barrier's wait for LDS once more, for the compiler's count)
    if (stage + 2 < count) fetch(stage & 1, stage + 2);
    if (stage + 1 < count) read(next, stage + 1);
    __builtin_amdgcn_sched_barrier(0);
    if (stage < count) multiply(now, factor_of<float, float>(k0 / kStep + stage), stage + 1 == count);
  };
  for (int stage = 0; stage < low; stage += 2) {
    pass(even, odd, stage);
    if (stage + 1 < low) pass(odd, even, stage + 1);
  }

  if constexpr (GROUPS == 2) {                      // the second group's half of the sum joins the first's
    __syncthreads();
    if (group) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int t = 0; t < 4; ++t) met[place(i, j, t)] = total[i][j][t];
    }
    __syncthreads();
    if (group) return;
  }
  bool any = false;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (GROUPS == 2 || second)
          total[i][j][t] = GROUPS == 2 ? total[i][j][t] + met[place(i, j, t)] : met[place(i, j, t)] + total[i][j][t];
        any = any || spoilt(total[i][j][t]);
      }
  if (__any(any)) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int t = 0; t < 4; ++t) met[place(i, j, t)] = total[i][j][t];
    sum_again_wide((const float*)p.x, (const float*)p.w, p.m, p.n, p.k, p.inter, met, row0 + r0, col0 + 32 * w4);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int t = 0; t < 4; ++t) total[i][j][t] = met[place(i, j, t)];
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int at = col0 + 32 * w4 + 16 * j + side;
      const int c = p.inter == 0 ? at : at / kSide * 8 + side % 8;     // the column of y
      if (c >= (p.inter == 0 ? p.n : p.inter)) continue;               // (gate and up lanes of a column go together)
      const float bias = p.bias != nullptr ? p.bias[c + (p.inter != 0 && side >= 8 ? p.inter : 0)] : 0.f;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int r = row0 + r0 + 16 * i + 4 * quarter + t;
        if (r >= p.m) continue;
        float sum = total[i][j][t];
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

// Rows of x that are split and multiplied at a time: what the pieces of as many take is all the scratch memory there is.
constexpr int kSplitRows = 2048;

template <int ROWS>
static int launch_gemm_f32_wide(GemmF32Params p, void* scratch, hipStream_t stream) {
  constexpr int bytes = Wide<ROWS>::bytes;
  static bool allowed = false;
  if (!allowed) {
    if (hipFuncSetAttribute((const void*)gemm_f32_wide_kernel<ROWS>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) !=
        hipSuccess)
      return ATOM_LAUNCH_FAILED;
    allowed = true;
  }
  const int m = p.m, out = p.inter ? p.inter : p.n;
  p.pieces = (const bf16_t*)scratch;
  for (int first = 0; first < m; first += kSplitRows) {
    p.m = min(kSplitRows, m - first);
    p.row_tiles = (p.m + ROWS - 1) / ROWS;
    const long tiles = (long)p.row_tiles * ((p.n + kWideCols - 1) / kWideCols);
    const size_t eights = (size_t)p.m * p.k / kLane;
    if (tiles > 0x3fffffL || eights / 256 > 0x3fffffL) return ATOM_TOO_LARGE;
    p.tiles = (int)tiles;
    hipLaunchKernelGGL(split_f32_kernel, dim3((unsigned)((eights + 255) / 256)), dim3(256), 0, stream, (const float*)p.x,
                       (bf16_t*)scratch, eights, p.k / kStep);
    hipLaunchKernelGGL((gemm_f32_wide_kernel<ROWS>), dim3((unsigned)(tiles + kXcds - 1) / kXcds * kXcds), dim3(kSlices * kWave),
                       bytes, stream, p);
    p.x = (const float*)p.x + (size_t)p.m * p.k;
    p.y = (char*)p.y + (size_t)p.m * out * (p.y_bf16 ? 2 : 4);
  }
  return launch_status();
}

template <typename TX, typename TW, int MT, int NT, int DEPTH>
static int launch_gemm_f32(GemmF32Params p, hipStream_t stream) {
  p.row_tiles = (p.m + MT * kSide - 1) / (MT * kSide);
  const long tiles = (long)p.row_tiles * ((p.n + NT * kSide - 1) / (NT * kSide));
  if (tiles > 0x3fffffL) return ATOM_TOO_LARGE;   // 2^31 threads
  p.tiles = (int)tiles;
  const dim3 grid((unsigned)(tiles + kXcds - 1) / kXcds * kXcds), block(kSlices * kWave);
  const bool whole = p.k % kStep == 0 && ((uintptr_t)p.x | (uintptr_t)p.w) % 16 == 0;
  if (whole)
    hipLaunchKernelGGL((gemm_f32_kernel<TX, TW, MT, NT, DEPTH, kWhole>), grid, block, 0, stream, p);
  else if (p.k >= 4)
    hipLaunchKernelGGL((gemm_f32_kernel<TX, TW, MT, NT, DEPTH, kAny>), grid, block, 0, stream, p);
  else if constexpr (MT * NT == 1)
    hipLaunchKernelGGL((gemm_f32_kernel<TX, TW, MT, NT, DEPTH, kTerms>), grid, block, 0, stream, p);
  return launch_status();
}

// The tiles that a product of more than 32 rows takes, those whose rounds over the CUs take least: 64 rows by 16, 32 or 64
// columns, or, through LDS, by 128, or 128 rows by 128 (kTall).  A round takes 38, 46, 71, 106 and 185 us at K 4,096 (465
// rows by 24,576: 48, 24, 12, 6 and 3 rounds of 1,800, 1,100, 843, 645 and 595 us in all; 180 rows: 5 rounds of 64 columns 378,
// three of 128 332, two of 128 rows 345).
constexpr int kTall = 256;
static int f32_columns(int m, int n, bool wide) {
  const long cus = device_cus();
  const auto cost = [&](int rows, int cols, int round) {
    return ((long)((m + rows - 1) / rows) * ((n + cols - 1) / cols) + cus - 1) / cus * round;
  };
  const long c1 = cost(64, 16, 38), c2 = cost(64, 32, 46), c4 = cost(64, 64, 71), c8 = cost(64, 128, 106), c16 = cost(128, 128, 185);
  if (wide && min(c8, c16) <= min(c1, min(c2, c4))) return c16 < c8 ? kTall : 128;
  return c1 <= c2 && c1 <= c4 ? 16 : c2 <= c4 ? 32 : 64;
}

static bool f32_wide(const void* x, int x_dtype, const void* w, int w_dtype, int m, int n, int k) {
  return x_dtype == ATOM_F32 && w_dtype == ATOM_F32 && m > 64 && k % kStep == 0 && ((uintptr_t)x | (uintptr_t)w) % 16 == 0 &&
         f32_columns(m, n, true) >= 128;
}

template <typename TX, typename TW>
static int choose_gemm_f32(const GemmF32Params& p, hipStream_t stream) {
  // Tiles two wide read x half as often, which pays from where there is one for most CUs on.
  if (p.k < 4) return launch_gemm_f32<TX, TW, 1, 1, 4>(p, stream);
  const long cus = device_cus();
  const bool wide_fills = p.n / 32 >= cus * 3 / 4;
  if (p.m <= 16) {
    if (p.m > 4 && wide_fills) return launch_gemm_f32<TX, TW, 1, 2, 3>(p, stream);
    return launch_gemm_f32<TX, TW, 1, 1, 4>(p, stream);
  }
  if (p.m <= 32) {
    // One step ahead, in 116 registers: two blocks a CU, where two steps ahead, in 148, leave room for one.  20 rows by 9,728 x
    // 96 4.4 and 5.9 us (4.5 with the float32 instructions), x 1,024 16.7 and 19.2 (17.3), by 24,576 x 4,096 86 and 92.
    if (wide_fills) return launch_gemm_f32<TX, TW, 2, 2, 1>(p, stream);
    return launch_gemm_f32<TX, TW, 2, 1, 3>(p, stream);
  }
  const int columns = f32_columns(p.m, p.n, false);
  if (columns == 16) return launch_gemm_f32<TX, TW, 4, 1, 2>(p, stream);
  if (columns == 32) return launch_gemm_f32<TX, TW, 4, 2, 2>(p, stream);
  return launch_gemm_f32<TX, TW, 4, 4, 1>(p, stream);
}

// Bytes of scratch memory that a product takes (its x as pieces); 0: none.
ATOM_EXPORT long atom_gemm_f32_scratch(const void* x, int x_dtype, const void* w, int w_dtype, int m, int n, int k) {
  if (m <= 0 || n <= 0 || k <= 0 || !f32_wide(x, x_dtype, w, w_dtype, m, n, k)) return 0;
  return 6L * min(m, kSplitRows) * k;
}

static int gemm_f32(GemmF32Params p, int x_dtype, int w_dtype, void* scratch, hipStream_t stream) {
  if (scratch != nullptr && f32_wide(p.x, x_dtype, p.w, w_dtype, p.m, p.n, p.k)) {
    if ((uintptr_t)scratch % 16) return ATOM_BAD_SHAPE;
    return f32_columns(p.m, p.n, true) == kTall ? launch_gemm_f32_wide<128>(p, scratch, stream)
                                                : launch_gemm_f32_wide<64>(p, scratch, stream);
  }
  switch (x_dtype * 2 + w_dtype) {
    case 0: return choose_gemm_f32<float, float>(p, stream);
    case 1: return choose_gemm_f32<float, bf16_t>(p, stream);
    case 2: return choose_gemm_f32<bf16_t, float>(p, stream);
    default: return choose_gemm_f32<bf16_t, bf16_t>(p, stream);
  }
}

// scratch: null, or atom_gemm_f32_scratch's bytes, aligned to 16 (without them the product takes the narrower tiles).
ATOM_EXPORT int atom_gemm_f32(const void* x, int x_dtype, const void* w, int w_dtype, const float* bias, void* y,
                              int y_dtype, int m, int n, int k, void* scratch, hipStream_t stream) {
  if (m < 0 || n <= 0 || k <= 0) return ATOM_BAD_SHAPE;
  if ((unsigned)x_dtype > 1u || (unsigned)w_dtype > 1u || (unsigned)y_dtype > 1u) return ATOM_BAD_DTYPE;
  if (m == 0) return ATOM_OK;
  return gemm_f32(GemmF32Params{x, w, bias, y, m, n, k, 0, 0, y_dtype == ATOM_BF16, nullptr, 0}, x_dtype, w_dtype, scratch, stream);
}

// y[M, inter] = silu(x wg^T + bg) * (x wu^T + bu), float32, for w of `inter` gate rows and then as many up rows: the sums of
// the plain product, gated where they are written instead of in a launch of their own that reads them back.
ATOM_EXPORT int atom_gemm_f32_gate(const void* x, int x_dtype, const void* w, int w_dtype, const float* bias, float* y, int m,
                                   int inter, int k, void* scratch, hipStream_t stream) {
  if (m < 0 || inter <= 0 || inter > 0x3fffffff || k <= 0) return ATOM_BAD_SHAPE;
  if ((unsigned)x_dtype > 1u || (unsigned)w_dtype > 1u) return ATOM_BAD_DTYPE;
  if (m == 0) return ATOM_OK;
  return gemm_f32(GemmF32Params{x, w, bias, y, m, 2 * inter, k, 0, 0, 0, nullptr, inter}, x_dtype, w_dtype, scratch, stream);
}
