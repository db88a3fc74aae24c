// y[M, N] = x[M, K] * w[N, K]^T (+ bias) of hundreds to thousands of rows, bfloat16 operands, float32 sums on the matrix
// cores (v_mfma_f32_16x16x32_bf16): the products of prompts.  With a gate w holds N gate rows and then N up rows and y is
// act(gate) * up; a plain product may end in an activation as well.
//
// A block of eight waves owns a tile of 128 to 256 rows of x by 128 to 256 rows of w and walks K in stages of 64 terms, a
// whole cache line of each row, which go straight from memory into LDS (lds_loads.h), two to four stages of them at a time (as many as fit).  A
// row's eight 16-byte pieces stand in LDS turned by the row's number, so that the sixteen rows a matrix operand reads lie in
// different banks.
//
// What bounds it: at 2,048 rows by 24,576 x 4,096 (314 to 323 us, 1.3 PFLOP/s) the matrix cores are busy for 70 % of the time, at
// the 1.8 GHz the chip holds then; the tile of 256 x 256 alone keeps them at 1.95 PFLOP/s without its loads and LDS reads, 1.6
// without its loads.  So:
//   - the operands of half a stage are read from LDS while the half before is multiplied, a few reads with every four matrix
//     instructions; the block meets once a stage, one such group after the last read of a stage, whose buffer is then free and
//     takes the stage that many buffers ahead (SX of x, SW of w), a load with every group (when the kernel was first built 318
//     -> 309 us at the size above);
//   - blocks go to the dies in turn; each die takes a run of tiles of its own, in bands of four row tiles.
// Tried then and not taken: stages of 32 terms, half lines, in four and five buffers (329; by tiles of 128 x 256 433, 367 with
// whole lines), four waves with 128 x 128 each, which read a third less from LDS (343).  Blocks that touch a quarter of their lines
// a stage further ahead, which the other blocks of their die read as well, take longer in every tile whose LDS has room for it
// (90 sizes: 128 x 128 1.05 times, 256 x 128 1.05, 256 x 192 1.02, 192 x 256 1.01).
//
// Where the tiles' last round would leave CUs idle, its tiles are cut along K (`slices`): their parts go to `scratch` in the
// order of the registers, and a second launch adds them, in slice order, and writes y.  A caller that adds slices itself may
// have them as [slices, M, N] where all of the product is cut (few tiles).
#include "common.h"
#include "lds_loads.h"

#include <type_traits>

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;

constexpr int kStageK = 64;               // terms of a stage
constexpr int kRowBytes = 2 * kStageK;    // of a row, a cache line
constexpr int kXcds = 8;                  // dies of the chip, each with an L2 of its own
constexpr int kBand = 4;                  // row tiles of a band
constexpr int kWaves = 8;
constexpr int kLdsBytes = 160 << 10;

// Activations, codes as in gemm_rows.hip: SiLU, ReLU or tanh-GELU of a gate, none, ReLU or its square of a plain product.
enum ManyAct : int { ACT_NONE = 0, ACT_SILU = 1, ACT_RELU = 2, ACT_GELU_TANH = 3, ACT_RELU_SQUARED = 4 };

struct ManyParams {
  const bf16_t* x;     // [m, k]
  const bf16_t* w;     // [n, k]; with a gate [2 n, k]
  const float* bias;   // [rows of w] or null
  void* y;             // [m, n] bfloat16 or float32
  float* parts;        // the cut tiles' sums; with as_slices [slices, m, n]
  int m, n, k, mtiles, ntiles;
  int whole;           // tiles that one block multiplies; those behind are cut into `slices`
  int slices, as_slices;
  int act, out_f32;
};

// SiLU, ReLU or tanh-GELU (0.5 v (1 + tanh(u)) is v times the logistic function of 2 u).
__device__ __forceinline__ float gate_of(float v, int act) {
  if (act == ACT_RELU) return fmaxf(v, 0.f);
  const float s = act == ACT_GELU_TANH ? 1.5957691216057308f * (v + 0.044715f * v * v * v) : v;
  return v / (1.f + expf(-s));
}

// Four neighbouring entries of y, from column c on, from their sums.
template <bool GATE>
__device__ __forceinline__ f32x4 finished(const ManyParams& p, f32x4 v, f32x4 up, int c) {
  if (p.bias != nullptr)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[i] += p.bias[c + i];
      if (GATE) up[i] += p.bias[p.n + c + i];
    }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (GATE) {
      v[i] = gate_of(v[i], p.act) * up[i];
    } else {
      if (p.act != ACT_NONE) v[i] = fmaxf(v[i], 0.f);
      if (p.act == ACT_RELU_SQUARED) v[i] *= v[i];
    }
  }
  return v;
}

// The tile of a number: bands of kBand row tiles, column by column.
__device__ __forceinline__ void place_of_tile(const ManyParams& p, int tile, int& mtile, int& ntile) {
  const int band = tile / (kBand * p.ntiles), in_band = tile - band * kBand * p.ntiles;
  const int height = min(kBand, p.mtiles - band * kBand);
  ntile = in_band / height;
  mtile = band * kBand + in_band % height;
}

// Number `at` of `count` things that are dealt out to the dies in turn, so that each die has a run of them.
__device__ __forceinline__ int in_runs(int at, int count) {
  const int xcd = at % kXcds;
  return xcd * (count / kXcds) + min(xcd, count % kXcds) + at / kXcds;
}

// A load of 16 bytes a lane from base + offset to LDS: lane l's land at `lds` + 16 l.
__device__ __forceinline__ void load_at_to_lds(const void* base, unsigned offset, unsigned lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(offset), "s"(base) : "memory");
}

// Waits until all but this wave's last LEFT loads have arrived and its LDS reads are done, then for the block.
template <int LEFT>
__device__ __forceinline__ void stage_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(LEFT) : "memory");
}

// Tiles of WM x WN waves, each with MF x NF squares of 16 rows of x by 16 rows of w; SX stages of x and SW of w in LDS.
template <int MF_, int NF_, int WM_, int WN_, int SX_, int SW_, bool GATE_>
struct Many {
  static constexpr int MF = MF_, NF = NF_, WM = WM_, WN = WN_, SX = SX_, SW = SW_;
  static constexpr bool GATE = GATE_;
  static constexpr int bm = 16 * MF * WM, bn = 16 * NF * WN, out = GATE ? bn / 2 : bn;
  static constexpr int xstage = bm * kRowBytes, wstage = bn * kRowBytes;       // LDS: the stages of w, those of x
  static constexpr int xloads = bm / 8 / kWaves, wloads = bn / 8 / kWaves;     // loads a wave
  static constexpr int xfrom = SW * wstage, lds = xfrom + SX * xstage;
  static constexpr int NO = GATE ? NF / 2 : NF;                                // fours of columns of y a lane holds of a row
  static_assert(WM * WN == kWaves && (!GATE || NF % 2 == 0), "as many gate as up rows a wave");
  static_assert(bm % 64 == 0 && bn % 64 == 0, "whole loads");
  static_assert(SW == SX || (SX == 2 && SW == 3), "the waits are counted for these");
  static_assert(lds <= kLdsBytes, "a CU's LDS");
};

template <typename G>
__global__ void __launch_bounds__(64 * kWaves, 2) gemm_many_kernel(ManyParams p) {
  constexpr int MF = G::MF, NF = G::NF, WN = G::WN, SX = G::SX, SW = G::SW, LX = G::xloads, LW = G::wloads, BM = G::bm, BN = G::bn;
  constexpr int NO = G::NO;
  extern __shared__ __align__(16) char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave % WN, wm = wave / WN;

  const int all = p.k / kStageK, cut = p.mtiles * p.ntiles - p.whole;
  int tile, unit = -1, begin = 0, stages = all;
  if ((int)blockIdx.x < p.whole) {
    tile = in_runs(blockIdx.x, p.whole);
  } else {
    unit = in_runs(blockIdx.x - p.whole, cut * p.slices);
    const int slice = unit / cut;
    tile = p.whole + unit % cut;
    begin = (int)((long)all * slice / p.slices);
    stages = (int)((long)all * (slice + 1) / p.slices) - begin;
  }
  int mtile, ntile;
  place_of_tile(p, tile, mtile, ntile);
  const int m0 = mtile * BM, n0 = ntile * G::out;

  // Load j of a wave brings eight rows, numbered over the tile's rows of w and then of x.  Sixteen rows of w, a matrix operand,
  // are four times four neighbouring columns, of which a lane ends up with one four an operand: `far` apart, operands `near`.
  // For bfloat16 results a lane's fours stand side by side (4 NO columns), for float32 ones those of the four lanes of a row, so
  // that either way a store writes 64 bytes or more of a row.  With a gate the first half of a wave's operands are gate rows, the
  // others the up rows of the same columns.  (Rows beyond the matrix: its last one again.)
  const bool in_floats = p.out_f32 || p.as_slices;
  const int far = in_floats ? 4 : 4 * NO, near = in_floats ? 16 : 4;
  const auto row_of = [&](int r) {
    if (r >= BN) return min(m0 + r - BN, p.m - 1);
    const int in = r % (16 * NF), operand = in / 16, i = in % 16;
    const int c = n0 + r / (16 * NF) * (16 * NO) + i / 4 * far + operand % NO * near + i % 4;
    return min(c, p.n - 1) + (operand < NO ? 0 : p.n);
  };
  const unsigned row_bytes = (unsigned)p.k * 2u;
  const char* const ws = (const char*)p.w + (size_t)begin * kRowBytes;
  const char* const xs = (const char*)p.x + (size_t)begin * kRowBytes;
  const unsigned lds0 = lds_address(smem);
  unsigned xfrom[LX], wfrom[LW];
  const unsigned turned = ((lane & 7) ^ (lane >> 3)) * 16;
#pragma unroll
  for (int j = 0; j < LX; ++j) xfrom[j] = (unsigned)row_of(BN + (j * kWaves + wave) * 8 + (lane >> 3)) * row_bytes + turned;
#pragma unroll
  for (int j = 0; j < LW; ++j) wfrom[j] = (unsigned)row_of((j * kWaves + wave) * 8 + (lane >> 3)) * row_bytes + turned;
  const auto load_x = [&](int j, int stage, int buf) {
    load_at_to_lds(xs + (size_t)stage * kRowBytes, xfrom[j], lds0 + G::xfrom + buf * G::xstage + (j * kWaves + wave) * 1024);
  };
  const auto load_w = [&](int j, int stage, int buf) {
    load_at_to_lds(ws + (size_t)stage * kRowBytes, wfrom[j], lds0 + buf * G::wstage + (j * kWaves + wave) * 1024);
  };
  f32x4 acc[MF][NF];
#pragma unroll
  for (int a = 0; a < MF; ++a)
#pragma unroll
    for (int b = 0; b < NF; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int at0 = (lane & 15) * kRowBytes + (((lane >> 4) ^ (lane & 7)) * 16);   // the first half of a stage
  const int at1 = at0 ^ 64;                                                      // the second
  const char* const wrow = smem + wn * 16 * NF * kRowBytes;
  const char* const xrow = smem + G::xfrom + wm * 16 * MF * kRowBytes;
  bf16x8 wf[2][NF], xf[2][MF];
  const auto read_w = [&](auto set, int i, int offset) {
    wf[set][i] = *reinterpret_cast<const bf16x8*>(wrow + offset + i * 16 * kRowBytes);
  };
  const auto read_x = [&](auto set, int i, int offset) {
    xf[set][i] = *reinterpret_cast<const bf16x8*>(xrow + offset + i * 16 * kRowBytes);
  };

  // Half a stage: the products of the operands in `set`, while the other set is read from woff and xoff on.  first and last:
  // what is to be done beside the groups of products.
  const auto half = [&](auto set, auto reads, auto meets, int woff, int xoff, auto beside) {
    constexpr int C = decltype(set)::value, FIRST = decltype(meets)::value >= 0 ? 1 : 0, GROUPS = MF - FIRST;
    using Other = std::integral_constant<int, C ^ 1>;
#pragma unroll
    for (int a = 0; a < MF; ++a) {
      const int g = a - FIRST;
      // the block meets behind the first group, which gives the last half's reads the time to arrive
      if constexpr (decltype(meets)::value >= 0)
        if (g == 0) stage_barrier<decltype(meets)::value>();
      if (decltype(reads)::value && g >= 0)
#pragma unroll
        for (int i = g * (MF + NF) / GROUPS; i < (g + 1) * (MF + NF) / GROUPS; ++i) {
          if (i < NF) read_w(Other{}, i, woff);
          else read_x(Other{}, i - NF, xoff);
        }
      if (g >= 0) beside(g, GROUPS);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < NF; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[C][b], xf[C][a], acc[a][b], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  using Yes = std::true_type;
  using No = std::false_type;
  using Set0 = std::integral_constant<int, 0>;
  using Set1 = std::integral_constant<int, 1>;
  using Apart = std::integral_constant<int, -1>;
  // A stage's loads go out as x, w; the next stage has arrived when no more than these of the newest are left: w where it is a
  // stage further ahead than x, else the stages behind the next.
  constexpr int LEFT = SW > SX ? LW : (SX - 2) * (LX + LW);
  using Meet = std::integral_constant<int, LEFT>;
  using MeetLast = std::integral_constant<int, 0>;
  const auto nothing = [](int, int) {};

#pragma unroll
  for (int s = 0; s < SW; ++s) {
    if (s < SX)
#pragma unroll
      for (int j = 0; j < LX; ++j) load_x(j, s, s);
#pragma unroll
    for (int j = 0; j < LW; ++j) load_w(j, s, s);
  }
  stage_barrier<(SX - 1) * LX + (SW - 1) * LW>();
#pragma unroll
  for (int i = 0; i < NF; ++i) read_w(Set0{}, i, at0);
#pragma unroll
  for (int i = 0; i < MF; ++i) read_x(Set0{}, i, at0);
  // (For the compiler's count of LDS reads, which is exact in the loop only if none are on their way into it: without this it
  // waits for all of them at the top of each stage.)
  __builtin_amdgcn_s_waitcnt(0xc07f);
  int wbuf = 0, xbuf = 0;
  const auto stage = [&](auto more_x, auto more_w, auto meet, auto more, int s) {
    const int wnext = wbuf + 1 == SW ? 0 : wbuf + 1, xnext = xbuf + 1 == SX ? 0 : xbuf + 1;
    half(Set0{}, Yes{}, Apart{}, wbuf * G::wstage + at1, xbuf * G::xstage + at1, nothing);
    if constexpr (decltype(more)::value)
      half(Set1{}, Yes{}, meet, wnext * G::wstage + at0, xnext * G::xstage + at0, [&](int g, int groups) {
        constexpr int N = (decltype(more_x)::value ? LX : 0) + (decltype(more_w)::value ? LW : 0);
#pragma unroll
        for (int j = g * N / groups; j < (g + 1) * N / groups; ++j) {
          if (j < LX) load_x(j, s + SX, xbuf);
          else load_w(j - LX, s + SW, wbuf);
        }
      });
    else
      half(Set1{}, No{}, Apart{}, 0, 0, nothing);
    wbuf = wnext, xbuf = xnext;
  };
  for (int s = 0; s < stages - SW; ++s) stage(Yes{}, Yes{}, Meet{}, Yes{}, s);
  if constexpr (SW > SX) stage(Yes{}, No{}, MeetLast{}, Yes{}, stages - SW);
#pragma unroll
  for (int s = SX; s > 1; --s) stage(No{}, No{}, MeetLast{}, Yes{}, stages - s);
  stage(No{}, No{}, Apart{}, No{}, stages - 1);

  // Lane (r, q) holds four columns an operand of row r of each sixteen rows, from `far` q and `near` b on.  (Through LDS, half a
  // tile's sums at a time, so that a wave wrote whole rows: 2,048 rows by twice 12,288 x 4,096 with SiLU 330 us, now 316.  Float32
  // results with a lane's columns side by side: 5,569 by 8,512 x 2,048 197 us, now 176.)
  if (unit >= 0 && !p.as_slices) {
    f32x4* dst = (f32x4*)p.parts + ((size_t)unit * kWaves + wave) * MF * NF * 64 + lane;
#pragma unroll
    for (int a = 0; a < MF; ++a)
#pragma unroll
      for (int b = 0; b < NF; ++b) dst[(a * NF + b) * 64] = acc[a][b];
    return;
  }
  const int row0 = m0 + wm * 16 * MF + (lane & 15), c0 = n0 + wn * 16 * NO + (lane >> 4) * far;
  if (in_floats) {
    float* const sums = unit >= 0 ? p.parts + (size_t)(unit / cut) * p.m * p.n : (float*)p.y;
#pragma unroll
    for (int b = 0; b < NO; ++b) {
      const int c = c0 + 16 * b;
      if (c >= p.n) continue;
#pragma unroll
      for (int a = 0; a < MF; ++a) {
        const int row = row0 + 16 * a;
        if (row >= p.m) continue;
        *reinterpret_cast<f32x4*>(sums + (size_t)row * p.n + c) =
            unit >= 0 ? acc[a][b] : finished<G::GATE>(p, acc[a][b], acc[a][NF - NO + b], c);
      }
    }
    return;
  }
  constexpr int PAIR = NO % 2 ? 1 : 2;
#pragma unroll
  for (int b = 0; b < NO; b += PAIR) {
    const int c = c0 + 4 * b;
    if (c >= p.n) continue;
#pragma unroll
    for (int a = 0; a < MF; ++a) {
      const int row = row0 + 16 * a;
      if (row >= p.m) continue;
      bf16_t* to = (bf16_t*)p.y + (size_t)row * p.n + c;
      f32x4 v[PAIR];
#pragma unroll
      for (int e = 0; e < PAIR; ++e) v[e] = finished<G::GATE>(p, acc[a][b + e], acc[a][NF - NO + b + e], c + 4 * e);
      if constexpr (PAIR == 2) {
        bf16x8 o;
#pragma unroll
        for (int i = 0; i < 8; ++i) o[i] = (bf16_t)v[i / 4][i % 4];
        *reinterpret_cast<bf16x8*>(to) = o;
      } else {
        *reinterpret_cast<bf16x4*>(to) = bf16x4{(bf16_t)v[0][0], (bf16_t)v[0][1], (bf16_t)v[0][2], (bf16_t)v[0][3]};
      }
    }
  }
}

// Adds the parts of the cut tiles: a block for every eighth of a tile's squares, what one wave of it holds.
template <typename G>
__global__ void __launch_bounds__(256) gemm_many_join_kernel(ManyParams p) {
  constexpr int MF = G::MF, NF = G::NF, NO = G::NO, SQUARES = MF * NF;
  const int cut = p.mtiles * p.ntiles - p.whole, at = blockIdx.x / kWaves, wave = blockIdx.x % kWaves, lane = threadIdx.x & 63;
  int mtile, ntile;
  place_of_tile(p, p.whole + at, mtile, ntile);
  const f32x4* src = (const f32x4*)p.parts + ((size_t)at * kWaves + wave) * SQUARES * 64 + lane;
  const size_t slice = (size_t)cut * kWaves * SQUARES * 64;
  const int row0 = mtile * G::bm + wave / G::WN * 16 * MF + (lane & 15);
  const int far = p.out_f32 ? 4 : 4 * NO, near = p.out_f32 ? 16 : 4;   // as in gemm_many_kernel
  const int col0 = ntile * G::out + wave % G::WN * 16 * NO + (lane >> 4) * far;
#pragma unroll 2
  for (int s = threadIdx.x / 64; s < MF * NO; s += 4) {
    const int row = row0 + s / NO * 16, c = col0 + s % NO * near;
    if (row >= p.m || c >= p.n) continue;
    const int square = s / NO * NF + s % NO;
    f32x4 v = src[square * 64], up = v;
    if (G::GATE) up = src[(square + NO) * 64];
    for (int i = 1; i < p.slices; ++i) {
      v += src[i * slice + square * 64];
      if (G::GATE) up += src[i * slice + (square + NO) * 64];
    }
    v = finished<G::GATE>(p, v, up, c);
    const size_t to = (size_t)row * p.n + c;
    if (p.out_f32) *reinterpret_cast<f32x4*>((float*)p.y + to) = v;
    else *reinterpret_cast<bf16x4*>((bf16_t*)p.y + to) = bf16x4{(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]};
  }
}

template <typename G>
static int launch_many(const ManyParams& p, hipStream_t stream) {
  const int cut = p.mtiles * p.ntiles - p.whole;
  static bool raised = false;
  if (!raised) {
    if (hipFuncSetAttribute((const void*)gemm_many_kernel<G>, hipFuncAttributeMaxDynamicSharedMemorySize, G::lds) != hipSuccess)
      return ATOM_LAUNCH_FAILED;
    raised = true;
  }
  hipLaunchKernelGGL(gemm_many_kernel<G>, dim3((unsigned)(p.whole + cut * p.slices)), dim3(64 * kWaves), G::lds, stream, p);
  if (cut > 0 && !p.as_slices)
    hipLaunchKernelGGL(gemm_many_join_kernel<G>, dim3((unsigned)(cut * kWaves)), dim3(256), 0, stream, p);
  return launch_status();
}

// The tiles: rows of x, rows of w, the most stages in LDS; what a stage takes on a chip that is nearly empty, what it takes more
// on a full one, and what a tile's start and end take (in 1/100 us).  Fitted to 10,700 measured products of 70 to 5,569 rows
// by 512 to 51,200 x 1,024 to 25,600, each by every tile and number of slices: they are met within 7.5 % (one standard
// deviation), and the plans so chosen take 2 % longer than each product's best.
struct ManyTile {
  int bm, bn, stages, stage, full, ends;
};
constexpr ManyTile kTiles[] = {
    {256, 256, 3, 91, 44, 707}, {192, 256, 3, 80, 30, 515}, {256, 192, 3, 79, 31, 491},
    {256, 128, 3, 59, 24, 289}, {128, 256, 3, 65, 21, 296}, {128, 128, 4, 34, 19, 133},
};
constexpr int kJoin = 600, kJoinMiB = 17;   // a second launch, and a MiB of parts written and read
constexpr long kMostParts = 128L << 20;     // bytes of parts at most

constexpr int kTileCount = sizeof(kTiles) / sizeof(kTiles[0]);

ATOM_EXPORT int atom_gemm_many_supports(int m, int n, int k, int gate) {
  // offsets into an operand are 32 bits
  return m >= 1 && n >= 8 && n % 8 == 0 && k >= 8 * kStageK && k % kStageK == 0 && (long)m * k <= 0x7fffffffL &&
         (long)n * k * (gate ? 2 : 1) <= 0x7fffffffL;
}

// The plan of a product: tile, tiles that stay whole, slices of the others, bytes of scratch memory.
ATOM_EXPORT int atom_gemm_many_plan(int m, int n, int k, int gate, int as_slices, int num_cus, int* plan) {
  if (!atom_gemm_many_supports(m, n, k, gate)) return ATOM_UNSUPPORTED;
  const int stages = k / kStageK;
  long best = -1;
  for (int t = 0; t < kTileCount; ++t) {
    const ManyTile& T = kTiles[t];
    const long mt = (m + T.bm - 1) / T.bm, out = gate ? T.bn / 2 : T.bn, nt = (n + out - 1) / out, tiles = mt * nt;
    if (tiles > 0x3fffffL) continue;
    const long full = tiles / num_cus * num_cus, rest = tiles - full;
    // `units` blocks of `count` stages each, in rounds over the CUs
    const auto time = [&](long units, long count) {
      const long last = units % num_cus;
      return units / num_cus * (count * (T.stage + T.full) + T.ends) + (last ? count * (T.stage + T.full * last / num_cus) + T.ends : 0);
    };
    for (int s = 1; s <= 8; ++s) {
      const long parts = rest * s * T.bm * T.bn * 4;
      if (s > 1 && (rest == 0 || stages / s < 8 || parts > kMostParts)) break;
      const bool apart = as_slices && full == 0;
      const long cost = s == 1 ? time(tiles, stages)
                               : time(full, stages) + time(rest * s, (stages + s - 1) / s) + parts * kJoinMiB / (1 << 20) + (apart ? 0 : kJoin);
      if (best < 0 || cost < best) {
        best = cost;
        plan[0] = t;
        plan[1] = s > 1 ? (int)full : (int)tiles;
        plan[2] = s;
        plan[3] = s > 1 && apart;
      }
    }
  }
  return best < 0 ? ATOM_TOO_LARGE : ATOM_OK;
}

// Bytes of scratch memory of a plan whose cut tiles are not handed out as slices.
ATOM_EXPORT long atom_gemm_many_scratch(int m, int n, int gate, int tile, int whole, int slices) {
  if (tile < 0 || tile >= kTileCount || slices <= 1) return 0;
  const ManyTile& T = kTiles[tile];
  const long out = gate ? T.bn / 2 : T.bn;
  const long cut = (long)((m + T.bm - 1) / T.bm) * ((n + out - 1) / out) - whole;
  return cut * slices * T.bm * T.bn * 4;
}

// The most memory that the parts of a product of `from` to `to` rows take by its plan, handed out as slices or not.  (A plan
// holds for all rows between two multiples of 64, which every tile's rows are.)
ATOM_EXPORT long atom_gemm_many_scratch_most(int from, int to, int n, int k, int gate, int num_cus) {
  long most = 0;
  for (long m = (from + 63L) / 64 * 64;; m += 64) {
    const int rows = (int)(m < to ? m : to);
    for (int as_slices = 0; rows >= from && as_slices <= (gate ? 0 : 1); ++as_slices) {
      int plan[4];
      if (atom_gemm_many_plan(rows, n, k, gate, as_slices, num_cus, plan) != ATOM_OK) continue;
      const long bytes = plan[3] ? 4L * plan[2] * rows * n : atom_gemm_many_scratch(rows, n, gate, plan[0], plan[1], plan[2]);
      if (bytes > most) most = bytes;
    }
    if (m >= to) return most;
  }
}

// plan: tile, tiles that stay whole, slices, whether the parts go to [slices, m, n] in `parts` (then all tiles are cut, and
// y, bias and act are not used).
ATOM_EXPORT int atom_gemm_many(const void* x, const void* w, const float* bias, void* y, float* parts, int m, int n, int k,
                               int gate, int act, int out_f32, int tile, int whole, int slices, int as_slices,
                               hipStream_t stream) {
  if (m < 0 || n <= 0 || k <= 0) return ATOM_BAD_SHAPE;
  if (m == 0) return ATOM_OK;
  if (!atom_gemm_many_supports(m, n, k, gate)) return ATOM_UNSUPPORTED;
  if (tile < 0 || tile >= kTileCount || slices < 1 || whole < 0 || act < 0 || act > ACT_RELU_SQUARED) return ATOM_BAD_SHAPE;
  if (gate ? act < ACT_SILU || act > ACT_GELU_TANH : act != ACT_NONE && act != ACT_RELU && act != ACT_RELU_SQUARED) return ATOM_UNSUPPORTED;
  const ManyTile& T = kTiles[tile];
  const long out = gate ? T.bn / 2 : T.bn, mt = (m + T.bm - 1) / T.bm, nt = (n + out - 1) / out;
  const long cut = mt * nt - whole;
  if (cut < 0 || (cut == 0) != (slices == 1) || (as_slices && (whole || slices == 1 || gate))) return ATOM_BAD_SHAPE;
  if (k / kStageK / slices < T.stages) return ATOM_BAD_SHAPE;
  if (mt * nt > 0x3fffffL || cut * slices > 0x3fffffL) return ATOM_TOO_LARGE;
  if (!x || !w || (!as_slices && !y) || (cut && !parts)) return ATOM_BAD_SHAPE;
  if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)y | (uintptr_t)parts) & 15) return ATOM_BAD_SHAPE;
  const ManyParams p{(const bf16_t*)x, (const bf16_t*)w, bias, y, parts, m, n, k, (int)mt, (int)nt, whole, slices, as_slices, act, out_f32};
  switch (tile) {
    case 0: return gate ? launch_many<Many<8, 4, 2, 4, 2, 3, true>>(p, stream) : launch_many<Many<8, 4, 2, 4, 2, 3, false>>(p, stream);
    case 1: return gate ? launch_many<Many<6, 4, 2, 4, 2, 3, true>>(p, stream) : launch_many<Many<6, 4, 2, 4, 2, 3, false>>(p, stream);
    case 2: return gate ? launch_many<Many<4, 6, 4, 2, 2, 3, true>>(p, stream) : launch_many<Many<4, 6, 4, 2, 2, 3, false>>(p, stream);
    case 3: return gate ? launch_many<Many<4, 4, 4, 2, 3, 3, true>>(p, stream) : launch_many<Many<4, 4, 4, 2, 3, 3, false>>(p, stream);
    case 4: return gate ? launch_many<Many<4, 4, 2, 4, 3, 3, true>>(p, stream) : launch_many<Many<4, 4, 2, 4, 3, 3, false>>(p, stream);
    default: return gate ? launch_many<Many<4, 2, 2, 4, 4, 4, true>>(p, stream) : launch_many<Many<4, 2, 2, 4, 4, 4, false>>(p, stream);
  }
}
