// Attention with a token's heads worked through together (attention_together.hip has the formulas) for few tokens whose keys are
// cut over several blocks, bfloat16, in two launches and one walk over the keys.
//
// Mixing the heads' finished weights commutes with the sum over the keys:
//
//   out_h = sum_j (sum_g talk[h, g] w_g(j)) v(j) = sum_g talk[h, g] (sum_j w_g(j) v(j)) / ...
//
// so a part needs no finished weights: it leaves, for every head g and every value head, the sum of its values weighed by
// exp(score_g - its own maximum), with its maximum and sum, and the second launch scales the parts, adds them in their order,
// divides by the whole sums and mixes the heads.  That is value heads times as many sums a key as mixing first, and in turn no
// pass for the maxima and sums before it.  Without mixing a part holds the heads of one value head.
//
// A part is a chain of waits for memory: the values are asked for before the scores are formed.  Scores come from the matrix
// cores (bfloat16 operands as stored, 16 keys a wave, 16 heads in the rows, of those only the ones that read these keys), whose
// loads take 64 bytes of a key row a time; a lane a key took most of the launch for them.  Weights and their sums are float32, on
// the matrix cores' float32 instructions, whose operand of values 16 entries of 16 keys are as they stand in a page.
// Heads of 128 with value heads of 128 in pages of 16, both launches in a replayed graph against the launches for maxima and sums,
// for values and for the parts' sum, us: 8 mixed heads, 2 value heads, 2 tokens behind 1,500 keys 11.7 and 22.3, one behind 8,000
// 15.8 and 32.3, 32 behind 1,500 29 and 66, 100 behind 1,000 51 and 108; 16 mixed heads, 4 value heads, 8 behind 2,048 19 and 36;
// 16 heads unmixed, 8 behind 2,048 24 and 49.  (Values summed by threads of one entry and several heads: 18.3 of the 22.3, most of
// it reading the weights from LDS.)
#include "common.h"

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;

constexpr int kFewThreads = 1024;
constexpr int kFewWaves = kFewThreads / kWave;
constexpr int kFewChunk = 64;          // keys a pass, counted from position 0
constexpr int kFewRow = kFewChunk + 4;
constexpr int kFewHeads = 16;          // heads of a block at most: a row of the matrix cores' tile each, a wave each
constexpr int kFewParts = 512;         // parts a token's keys are cut into at most
constexpr int kFewSteps = 8;           // steps of 32 entries over a head's size at most

struct TogetherFewArgs {
  const int* token_seq; const int* positions; const int* block_tables; int max_blocks;
  int H, G, D, DV, page_shift, window, parts;
  float scale;
  const float* head_scale; const float* sink; const float* talk;
  float* ws_ml;   // [tokens, H, parts, 2]: a part's maximum and sum
  float* ws_o;    // [tokens, parts, sets, heads of a set, value heads of a set, DV]
};

// grid (tokens, sets, parts): all heads where they are mixed, else a set is a value head's.  A wave owns TILES times 16 entries of
// value heads, with all heads.
template <int TILES>
__global__ void __launch_bounds__(kFewThreads)
together_few_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
                    TogetherFewArgs a) {
  __shared__ __align__(16) float s[kFewHeads * kFewRow];   // scores, then weights
  __shared__ __align__(16) float shrink[kFewHeads];                      // what a new maximum makes of the sums so far
  const int t = blockIdx.x, part = blockIdx.z, seq = a.token_seq[t];
  if (seq < 0) return;                                     // padding: the second launch knows it
  const bool mixes = a.talk != nullptr;
  const int group = a.H / a.G, HB = mixes ? a.H : group, VG = mixes ? a.G : 1;
  const int h0 = mixes ? 0 : blockIdx.y * HB, kv0 = mixes ? 0 : blockIdx.y;
  const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave), side = lane % 16, quarter = lane / 16;
  const int pos = a.positions[t];
  const int* table = a.block_tables + (size_t)seq * a.max_blocks;
  const int first = (a.window > 0 && pos - a.window + 1 > 0) ? pos - a.window + 1 : 0;
  const int start = first / kFewChunk * kFewChunk;
  const int chunks = (pos - start) / kFewChunk + 1, each = (chunks + a.parts - 1) / a.parts;
  const int c0 = part * each, c1 = min(c0 + each, chunks);
  const size_t page_keys = (size_t)1 << a.page_shift;
  const int in_page = (1 << a.page_shift) - 1;

  const int entries = VG * a.DV;
  int entry[TILES];                                        // this lane's of each tile; tiles behind the last are read as the last
  const bf16_t* column[TILES];
#pragma unroll
  for (int x = 0; x < TILES; ++x) {
    entry[x] = (wave + x * kFewWaves) * 16 + side;
    const int e = min(entry[x], entries - 16 + side);
    column[x] = v_cache + ((size_t)(kv0 + e / a.DV) * a.DV + e % a.DV) * page_keys;
  }
  const size_t v_page = (size_t)a.G * a.DV * page_keys;
  float top = -INFINITY, sum = 0.f;                        // of head `wave`
  f32x4 acc[TILES];
#pragma unroll
  for (int x = 0; x < TILES; ++x) acc[x] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int c = c0; c < c1; ++c) {
    const int base = start + c * kFewChunk;
    const int lo = max(base, first), hi = min(base + kFewChunk - 1, pos);
    // keys 16 u + 4 quarter .. of the chunk; fours wholly outside lo .. hi read one inside
    bf16x4 v[TILES][4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int key = min(max(base + 16 * u + 4 * quarter, lo & ~3), hi & ~3);
      const size_t at = (size_t)table[key >> a.page_shift] * v_page + (key & in_page);
#pragma unroll
      for (int x = 0; x < TILES; ++x) v[x][u] = *reinterpret_cast<const bf16x4*>(column[x] + at);
    }
    for (int job = wave; job < kFewChunk / 16 * VG; job += kFewWaves) {
      const int kv = job / (kFewChunk / 16), col = job % (kFewChunk / 16) * 16 + side;
      const int key = min(max(base + col, lo), hi);
      const bf16_t* kr = k_cache + (((size_t)table[key >> a.page_shift] * a.G + kv0 + kv) * page_keys + (key & in_page)) * a.D + 8 * quarter;
      const bool reads = side < HB && (!mixes || side / group == kv);
      const bf16_t* qr = q + ((size_t)t * a.H + h0 + min(side, HB - 1)) * a.D + 8 * quarter;
      float by[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) by[r] = a.scale * (a.head_scale != nullptr ? a.head_scale[h0 + min(4 * quarter + r, HB - 1)] : 1.f);
      f32x4 d = {0.f, 0.f, 0.f, 0.f};
      const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
      for (int u = 0; u < kFewSteps; ++u) {
        if (32 * u >= a.D) break;
        const bf16x8 x = *reinterpret_cast<const bf16x8*>(qr + 32 * u);
        d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(reads ? x : zero, *reinterpret_cast<const bf16x8*>(kr + 32 * u), d, 0, 0, 0);
      }
      const bool seen = base + col >= lo && base + col <= hi;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int h = 4 * quarter + r;
        if (h < HB && (!mixes || h / group == kv)) s[h * kFewRow + col] = seen ? d[r] * by[r] : -INFINITY;
      }
    }
    __syncthreads();
    if (wave < HB) {
      const float x = s[wave * kFewRow + lane];
      const float now = fmaxf(top, wave_max(x));           // finite: a chunk holds at least one visible key
      const float w = expf(x - now), was = top == -INFINITY ? 0.f : expf(top - now);
      s[wave * kFewRow + lane] = w;
      sum = sum * was + wave_sum(w);
      top = now;
      if (lane == 0) shrink[wave] = was;
    }
    __syncthreads();
    const f32x4 was = *reinterpret_cast<const f32x4*>(shrink + 4 * quarter);
    float vf[TILES][16];
#pragma unroll
    for (int x = 0; x < TILES; ++x) {
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[x][r] *= was[r];
#pragma unroll
      for (int i = 0; i < 16; ++i) vf[x][i] = to_f32(v[x][i / 4][i % 4]);
    }
    if (lo > base || hi < base + kFewChunk - 1) {          // (a key outside adds nothing, whatever its place in the page holds)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int key = base + i / 4 * 16 + 4 * quarter + i % 4;
#pragma unroll
        for (int x = 0; x < TILES; ++x) vf[x][i] = key >= lo && key <= hi ? vf[x][i] : 0.f;
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const f32x4 w = *reinterpret_cast<const f32x4*>(s + side * kFewRow + 16 * u + 4 * quarter);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int x = 0; x < TILES; ++x) acc[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[e], vf[x][4 * u + e], acc[x], 0, 0, 0);
    }
    __syncthreads();                                       // the weights have been read
  }
  if (wave < HB && lane == 0) {
    float* ml = a.ws_ml + (((size_t)t * a.H + h0 + wave) * a.parts + part) * 2;
    ml[0] = top, ml[1] = sum;
  }
  if (c0 >= c1) return;
  float* to = a.ws_o + (((size_t)t * a.parts + part) * gridDim.y + blockIdx.y) * HB * entries;
#pragma unroll
  for (int x = 0; x < TILES; ++x)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (entry[x] < entries && 4 * quarter + r < HB) to[(size_t)(4 * quarter + r) * entries + entry[x]] = acc[x][r];
}

constexpr int kMixThreads = 1024;
constexpr int kMixCols = 32;
constexpr int kMixAhead = 8;
constexpr int kMixSplits = 4;   // threads that share a head's parts: every fourth part each, so that a part's wait is shared by many

// grid (tokens, value heads, blocks of 32 entries): the parts scaled and added in a fixed order, the heads mixed.
__global__ void __launch_bounds__(kMixThreads) together_mix_kernel(bf16_t* __restrict__ out, TogetherFewArgs a) {
  extern __shared__ float lds[];
  __shared__ float value[kMixSplits][kFewHeads][kMixCols + 1];
  const int t = blockIdx.x, kv = blockIdx.y, col = blockIdx.z * kMixCols + threadIdx.x % kMixCols;
  const bool mixes = a.talk != nullptr;
  const int group = a.H / a.G, HB = mixes ? a.H : group, VG = mixes ? a.G : 1, h0 = mixes ? 0 : kv * group, sets = mixes ? 1 : a.G;
  float* weight = lds;                                     // [HB][parts]
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  constexpr int kSlots = kMixThreads / kMixCols / kMixSplits, kHeadsOfSlot = kFewHeads / kSlots;
  const int slot = threadIdx.x / kMixCols % kSlots, split = threadIdx.x / kMixCols / kSlots;
  const bool has = col < a.DV;
  bf16_t* to = out + ((size_t)t * a.H + kv * group) * a.DV + col;
  if (a.token_seq[t] < 0) {                                // padding row
    if (has && split == 0)
      for (int j = slot; j < group; j += kSlots) to[(size_t)j * a.DV] = from_f32<bf16_t>(0.f);
    return;
  }
  const size_t of_part = (size_t)sets * HB * VG * a.DV;
  const float* from = a.ws_o + (size_t)t * a.parts * of_part + (size_t)(mixes ? 0 : kv) * HB * a.DV + (size_t)(mixes ? kv : 0) * a.DV + (has ? col : 0);
  float o[kHeadsOfSlot][kMixAhead];
  const auto fetch = [&](int i0) {                         // the split's parts i0 .. of its own
#pragma unroll
    for (int x = 0; x < kHeadsOfSlot; ++x)
#pragma unroll
      for (int p = 0; p < kMixAhead; ++p)
        o[x][p] = from[(size_t)min((i0 + p) * kMixSplits + split, a.parts - 1) * of_part + (size_t)min(slot + x * kSlots, HB - 1) * VG * a.DV];
  };
  fetch(0);
  for (int h = wave; h < HB; h += kMixThreads / kWave) {
    const float* ml = a.ws_ml + ((size_t)t * a.H + h0 + h) * a.parts * 2;
    float m = -INFINITY;
    for (int p = lane; p < a.parts; p += kWave) m = fmaxf(m, ml[2 * p]);
    m = wave_max(m);
    const float sink = a.sink != nullptr ? a.sink[h0 + h] : -INFINITY;
    m = fmaxf(m, sink);
    float l = 0.f;
    for (int p = lane; p < a.parts; p += kWave) {
      const float mp = ml[2 * p], w = mp == -INFINITY ? 0.f : expf(mp - m);
      weight[h * a.parts + p] = w;
      l += w == 0.f ? 0.f : ml[2 * p + 1] * w;
    }
    l = wave_sum(l);
    if (a.sink != nullptr) l += expf(sink - m);
    const float inv = 1.f / l;
    for (int p = lane; p < a.parts; p += kWave) weight[h * a.parts + p] *= inv;
  }
  __syncthreads();
  float sum[kHeadsOfSlot];
#pragma unroll
  for (int x = 0; x < kHeadsOfSlot; ++x) sum[x] = 0.f;
  for (int i0 = 0; i0 * kMixSplits < a.parts; i0 += kMixAhead) {
    if (i0) fetch(i0);
#pragma unroll
    for (int x = 0; x < kHeadsOfSlot; ++x)
#pragma unroll
      for (int p = 0; p < kMixAhead; ++p) {
        const int part = (i0 + p) * kMixSplits + split;
        const float w = part < a.parts ? weight[min(slot + x * kSlots, HB - 1) * a.parts + part] : 0.f;
        sum[x] += w == 0.f ? 0.f : w * o[x][p];            // (an empty part has left nothing to read)
      }
  }
#pragma unroll
  for (int x = 0; x < kHeadsOfSlot; ++x)
    if (slot + x * kSlots < HB) value[split][slot + x * kSlots][threadIdx.x % kMixCols] = sum[x];
  __syncthreads();
  const int at = threadIdx.x % kMixCols;
  const auto whole = [&](int h) { return (value[0][h][at] + value[1][h][at]) + (value[2][h][at] + value[3][h][at]); };
  static_assert(kMixSplits == 4);
  if (!has) return;
  for (int j = threadIdx.x / kMixCols; j < group; j += kSlots * kMixSplits) {
    float y = 0.f;
    if (mixes) {
      const float* row = a.talk + (size_t)(kv * group + j) * a.H;
      for (int g = 0; g < a.H; ++g) y += row[g] * whole(g);
    } else {
      y = whole(j);
    }
    to[(size_t)j * a.DV] = from_f32<bf16_t>(y);
  }
}

// How many tiles of 16 entries a wave owns, or 0 where the sizes do not fit: up to 16 heads a block, of whole steps of 32 entries,
// value heads of whole tiles, up to 64 of them, pages of a power of two of 4 keys or more.
static int few_tiles(int H, int G, int D, int DV, int page_size, int mixes) {
  if (H <= 0 || G <= 0 || H % G || D <= 0 || DV <= 0 || page_size < 4 || (page_size & (page_size - 1))) return 0;
  const long HB = mixes ? H : H / G, tiles = (long)(mixes ? G : 1) * DV / 16;
  if (HB > kFewHeads || D % 32 || D > 32 * kFewSteps || DV % 16 || tiles > 4 * kFewWaves) return 0;
  return (int)((tiles + kFewWaves - 1) / kFewWaves);
}

ATOM_EXPORT int atom_attention_together_few_supports(int H, int G, int D, int DV, int page_size, int mixes, int parts) {
  return few_tiles(H, G, D, DV, page_size, mixes) > 0 && parts > 1 && parts <= kFewParts;
}

// bfloat16 q [tokens, H, D], pages and out as atom_attention_together's; ws_ml [tokens, H, parts, 2], ws_o [tokens, parts, H, DV],
// G times that with `talk`.
ATOM_EXPORT int atom_attention_together_few(const void* q, const void* k_cache, const void* v_cache, void* out, const int* token_seq,
                                            const int* positions, const int* block_tables, int max_blocks, int tokens, int H, int G,
                                            int D, int DV, int page_size, float scale, const float* head_scale, const float* sink,
                                            const float* talk, int window, int parts, float* ws_ml, float* ws_o, hipStream_t stream) {
  if (tokens < 0 || max_blocks <= 0 || window < 0) return ATOM_BAD_SHAPE;
  if (!atom_attention_together_few_supports(H, G, D, DV, page_size, talk != nullptr, parts)) return ATOM_UNSUPPORTED;
  if (q == nullptr || k_cache == nullptr || v_cache == nullptr || out == nullptr || ws_ml == nullptr || ws_o == nullptr) return ATOM_BAD_SHAPE;
  if (token_seq == nullptr || positions == nullptr || block_tables == nullptr) return ATOM_BAD_SHAPE;
  if (((uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache) & 15) return ATOM_BAD_SHAPE;
  if (tokens == 0) return ATOM_OK;
  int shift = 0;
  while ((1 << shift) < page_size) ++shift;
  const TogetherFewArgs a{token_seq, positions, block_tables, max_blocks, H, G, D, DV, shift, window, parts, scale, head_scale, sink, talk, ws_ml, ws_o};
  const dim3 grid(tokens, talk != nullptr ? 1 : G, parts);
#define GO_FEW(TILES) \
  hipLaunchKernelGGL(together_few_kernel<TILES>, grid, dim3(kFewThreads), 0, stream, (const bf16_t*)q, (const bf16_t*)k_cache, (const bf16_t*)v_cache, a)
  switch (few_tiles(H, G, D, DV, page_size, talk != nullptr)) {
    case 1: GO_FEW(1); break;
    case 2: GO_FEW(2); break;
    case 3: GO_FEW(3); break;
    default: GO_FEW(4); break;
  }
#undef GO_FEW
  const int HB = talk != nullptr ? H : H / G;
  hipLaunchKernelGGL(together_mix_kernel, dim3(tokens, G, (DV + kMixCols - 1) / kMixCols), dim3(kMixThreads),
                     (size_t)HB * parts * sizeof(float), stream, (bf16_t*)out, a);
  return launch_status();
}
