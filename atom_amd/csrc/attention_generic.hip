// Paged attention, general form: any head size, any page size, float32 or bfloat16,
// every query token of a mixed batch (prompt portions and single decoded tokens alike).
//
// One block per (query token, query head), or, for many tokens, per token and two or four heads that share keys.  The
// token's request and absolute position are given per token; the keys it sees are positions max(0, p - window + 1) .. p of that
// request, found through the request's block table; with `chunk` only those from the start of the run of `chunk`
// positions (counted from position 0) that p lies in.  With `softcap` a score s becomes softcap * tanh(s / softcap); with
// `slopes` head h's score of key j then loses slopes[h] * (p - j); exp(sink[h]) joins head h's denominator with no key and
// no value; the output, of which the first `od` entries of a head are written, is multiplied by sigmoid(gate[t, h]).  Keys are walked in fixed chunks
// counted from position 0 with a running maximum and sum (all float32), so the result
// for a token depends only on its own keys: not on the batch, not on how the prompt
// was cut into steps, not on which pages hold the keys.
//
// Pages: keys [num_pages, Hkv, page_size, D]; values [num_pages, Hkv, D, page_size].
#include "common.h"

constexpr int kAttnItems = 512;   // (entry, run of keys) pairs a block has
constexpr int kAttnFew = 1024;    // blocks up to which the chip holds them all at once with 512 threads each
constexpr int kAttnFours = 600;  // blocks of four heads from which on a launch has enough of them
constexpr int kAttnChunk = 512;  // keys per pass
constexpr int kAttnStretch = 16; // keys a thread adds in one go

// Over a block, for all its threads and each of HEADS heads: the maximum of a value a thread, or the sum of kAttnItems values, PER
// a thread: over each 64 of them, then group by group; the same order whether a block's waves hold one group each or several.
template <int HEADS, int PER>
__device__ __forceinline__ void block_maxima(float (&v)[HEADS], float* scratch) {
  const int wave = threadIdx.x / kWave;
  constexpr int WAVES = kAttnItems / kWave / PER;
  __syncthreads();   // what was there before has been read
#pragma unroll
  for (int h = 0; h < HEADS; ++h) {
    const float m = wave_max(v[h]);
    if (threadIdx.x % kWave == 0) scratch[h * WAVES + wave] = m;
  }
  __syncthreads();
#pragma unroll
  for (int h = 0; h < HEADS; ++h) {
    v[h] = scratch[h * WAVES];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) v[h] = fmaxf(v[h], scratch[h * WAVES + w]);
  }
}

template <int HEADS, int PER>
__device__ __forceinline__ void groups_sums(const float (&v)[HEADS][PER], float (&sums)[HEADS], float* scratch) {
  constexpr int WAVES = kAttnItems / kWave / PER, GROUPS = kAttnItems / kWave;
  const int wave = threadIdx.x / kWave;
  __syncthreads();   // what was there before has been read
#pragma unroll
  for (int h = 0; h < HEADS; ++h)
#pragma unroll
    for (int r = 0; r < PER; ++r) {
      const float s = wave_sum(v[h][r]);
      if (threadIdx.x % kWave == 0) scratch[h * GROUPS + r * WAVES + wave] = s;
    }
  __syncthreads();
#pragma unroll
  for (int h = 0; h < HEADS; ++h) {
    sums[h] = 0.f;
#pragma unroll
    for (int g = 0; g < GROUPS; ++g) sums[h] += scratch[h * GROUPS + g];
  }
}

// A block's items are (output entry, every `runs`-th stretch of kAttnStretch keys counted from position 0): as many runs side
// by side as the head leaves items for.  One thread that walks all keys of an entry is a chain of waits, so few blocks take a
// thread an item (PER 1); where there are blocks enough to fill the chip, 128 threads with four items each (PER 4) leave fewer
// of them idle at a short row's end.  Float32, 32 heads of 128: one or two tokens behind some 300 keys 26 us with one run, 15.7
// with PER 1; a prompt of 461 tokens 250 us with PER 1, 198 with PER 4.  The items and the order of every sum are the same in both.
// What then bounds a prompt is what its blocks read of the keys and values, 32 times over for 32 heads: HEADS query heads of a
// block, which have one head of keys, use what is read for all of them (that prompt, four heads a head of keys: 214 -> 85 us).
template <typename T, int PER, int HEADS>
__global__ void __launch_bounds__(kAttnItems / PER)
paged_attention_generic_kernel(const T* __restrict__ q, const T* __restrict__ k_cache,
                               const T* __restrict__ v_cache, T* __restrict__ out,
                               const int* __restrict__ token_seq, const int* __restrict__ positions,
                               const int* __restrict__ block_tables, int max_blocks, int hq, int hkv,
                               int d, int page_size, float scale, int window, int chunk, float softcap,
                               const float* __restrict__ sink, const float* __restrict__ slopes,
                               const float* __restrict__ gate, long gate_ld, int od, int key_fours, int value_fours) {
  extern __shared__ __align__(16) float smem[];
  const int dq = (d + 3) / 4 * 4;
  float* qs = smem;                                // HEADS x dq
  float* probs = qs + HEADS * dq;                  // HEADS x kAttnChunk
  float* scratch = probs + HEADS * kAttnChunk;     // HEADS x 16
  float* shares = scratch + HEADS * 16;            // HEADS x kAttnItems
  constexpr int kAttnThreads = kAttnItems / PER;
  const int t = blockIdx.x;
  const int h0 = blockIdx.y * HEADS;
  const int kvh = h0 / (hq / hkv);
  const int tid = threadIdx.x;
  const int seq = token_seq[t];
  const int pos = positions[t];
  T* dst = out + ((size_t)t * hq + h0) * od;
  if (seq < 0) {  // padding row
    for (int i = tid; i < HEADS * od; i += kAttnThreads) dst[i] = from_f32<T>(0.f);
    return;
  }
  const int* table = block_tables + (size_t)seq * max_blocks;
  const T* qr = q + ((size_t)t * hq + h0) * d;
  for (int i = tid; i < d; i += kAttnThreads)
#pragma unroll
    for (int h = 0; h < HEADS; ++h) qs[h * dq + i] = to_f32(qr[h * d + i]) * scale;
  __syncthreads();

  int first = (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;
  if (chunk > 0 && pos / chunk * chunk > first) first = pos / chunk * chunk;
  const int last = pos;  // inclusive
  const int wide = min(kAttnItems, (d + kWave - 1) / kWave * kWave), runs = kAttnItems / wide;
  float acc[HEADS][PER], run_max[HEADS], run_sum[HEADS], slope[HEADS];
#pragma unroll
  for (int h = 0; h < HEADS; ++h) {
#pragma unroll
    for (int r = 0; r < PER; ++r) acc[h][r] = 0.f;
    // a sink: as if a key with that score and a value of zeros had been seen already
    run_max[h] = sink != nullptr ? sink[h0 + h] : -INFINITY;
    run_sum[h] = sink != nullptr ? 1.f : 0.f;
    slope[h] = slopes != nullptr ? slopes[h0 + h] : 0.f;
  }

  // chunks are aligned to multiples of kAttnChunk from position 0, so the grouping of
  // keys does not move with the window start
  for (int base = (first / kAttnChunk) * kAttnChunk; base <= last; base += kAttnChunk) {
    const int lo = base > first ? base : first;
    const int hi = (base + kAttnChunk - 1 < last) ? base + kAttnChunk - 1 : last;
    const int n = hi - lo + 1;
    float new_max[HEADS];
#pragma unroll
    for (int h = 0; h < HEADS; ++h) new_max[h] = -INFINITY;
    for (int j = tid; j < n; j += kAttnThreads) {
      const int key = lo + j;
      const int page = table[key / page_size];
      const int off = key % page_size;
      const T* kr = k_cache + (((size_t)page * hkv + kvh) * page_size + off) * (size_t)d;
      float s[HEADS];
#pragma unroll
      for (int h = 0; h < HEADS; ++h) s[h] = 0.f;
      if (key_fours) {   // rows of four-element pieces: a piece a load
#pragma unroll 8
        for (int i = 0; i < d; i += 4) {
          const Four<T> four = *reinterpret_cast<const Four<T>*>(kr + i);
#pragma unroll
          for (int h = 0; h < HEADS; ++h) {
            const float4 qi = *reinterpret_cast<const float4*>(qs + h * dq + i);
            s[h] += qi.x * to_f32(four.at[0]);
            s[h] += qi.y * to_f32(four.at[1]);
            s[h] += qi.z * to_f32(four.at[2]);
            s[h] += qi.w * to_f32(four.at[3]);
          }
        }
      } else {
        for (int i = 0; i < d; ++i)
#pragma unroll
          for (int h = 0; h < HEADS; ++h) s[h] += qs[h * dq + i] * to_f32(kr[i]);
      }
#pragma unroll
      for (int h = 0; h < HEADS; ++h) {
        if (softcap > 0.f) s[h] = softcap * tanhf(s[h] / softcap);
        s[h] = fmaf(slope[h], (float)(key - pos), s[h]);
        probs[h * kAttnChunk + j] = s[h];
        new_max[h] = fmaxf(new_max[h], s[h]);
      }
    }
    block_maxima<HEADS, PER>(new_max, scratch);
    float rescale[HEADS], p[HEADS][PER], chunk_sum[HEADS];
    static_assert(kAttnChunk == kAttnItems, "a key of a chunk an item");
#pragma unroll
    for (int h = 0; h < HEADS; ++h) {
      new_max[h] = fmaxf(run_max[h], new_max[h]);
      rescale[h] = (run_max[h] == -INFINITY) ? 0.f : expf(run_max[h] - new_max[h]);
#pragma unroll
      for (int r = 0; r < PER; ++r) {
        const int j = tid + r * kAttnThreads;
        p[h][r] = j < n ? expf(probs[h * kAttnChunk + j] - new_max[h]) : 0.f;
        if (j < n) probs[h * kAttnChunk + j] = p[h][r];
      }
    }
    groups_sums<HEADS, PER>(p, chunk_sum, scratch);  // also orders the probs[] writes
#pragma unroll
    for (int h = 0; h < HEADS; ++h) {
      run_sum[h] = run_sum[h] * rescale[h] + chunk_sum[h];
      run_max[h] = new_max[h];
    }
#pragma unroll
    for (int r = 0; r < PER; ++r) {
      const int item = tid + r * kAttnThreads, entry = item % wide, run = item / wide;
      if (entry >= d || run >= runs) continue;
      float a[HEADS];
#pragma unroll
      for (int h = 0; h < HEADS; ++h) a[h] = acc[h][r] * rescale[h];
      for (int from = base + run * kAttnStretch; from <= hi; from += runs * kAttnStretch) {
        const int stop = min(from + kAttnStretch, hi + 1);
        // page by page: a page's values of one entry lie side by side
        for (int key = max(from, lo); key < stop;) {
          const int off = key % page_size;
          const int here = min(page_size - off, stop - key);
          const T* vr = v_cache + (((size_t)table[key / page_size] * hkv + kvh) * d + entry) * (size_t)page_size + off;
          const float* pr = probs + (key - lo);
          int j = 0;
          if (value_fours && off % 4 == 0) {
            for (; j + 4 <= here; j += 4) {
              const Four<T> four = *reinterpret_cast<const Four<T>*>(vr + j);
#pragma unroll
              for (int h = 0; h < HEADS; ++h)
#pragma unroll
                for (int e = 0; e < 4; ++e) a[h] += pr[h * kAttnChunk + j + e] * to_f32(four.at[e]);
            }
          }
          for (; j < here; ++j)
#pragma unroll
            for (int h = 0; h < HEADS; ++h) a[h] += pr[h * kAttnChunk + j] * to_f32(vr[j]);
          key += here;
        }
      }
#pragma unroll
      for (int h = 0; h < HEADS; ++h) acc[h][r] = a[h];
    }
    __syncthreads();  // probs[] is rewritten by the next chunk
  }
#pragma unroll
  for (int h = 0; h < HEADS; ++h) {
    run_sum[h] = 1.f / run_sum[h];
    if (gate != nullptr) run_sum[h] /= 1.f + expf(-gate[(size_t)t * gate_ld + h0 + h]);
#pragma unroll
    for (int r = 0; r < PER; ++r) shares[h * kAttnItems + tid + r * kAttnThreads] = acc[h][r];
  }
  __syncthreads();
#pragma unroll
  for (int h = 0; h < HEADS; ++h)
    for (int entry = tid; entry < od; entry += kAttnThreads) {   // the runs' shares
      float sum = 0.f;
      for (int r = 0; r < runs; ++r) sum += shares[h * kAttnItems + r * wide + entry];
      dst[h * od + entry] = from_f32<T>(sum * run_sum[h]);
    }
}

// Heads that a block of 128 threads takes; 0: a block of 512 threads each.  Four where that leaves two blocks or more a CU: 484 sizes
// (seven layouts of 6 to 64 heads, prompts of 20 to 1,000 tokens, portions behind 2,000 keys, decoded tokens behind 300 and 2,000; both
// types) take 0.9 % longer than each's best of one, two and four; with four always 2.5 % (32 heads over 8, 33 tokens 10.7 us, with
// two 8.5, with one 8.8; 461 tokens 121, 188 and 332).
ATOM_EXPORT int atom_paged_attention_generic_heads(int tokens, int hq, int hkv) {
  const long rows = (long)tokens * hq;
  const int group = hq / hkv;
  if (rows <= kAttnFew) return 0;
  if (group % 4 == 0 && rows / 4 >= kAttnFours) return 4;
  return group % 2 == 0 ? 2 : 1;
}

ATOM_EXPORT int atom_paged_attention_generic(const void* q, const void* k_cache, const void* v_cache, void* out,
                                             const int* token_seq, const int* positions,
                                             const int* block_tables, int max_blocks, int dtype, int tokens,
                                             int hq, int hkv, int d, int page_size, float scale, int window,
                                             int chunk, float softcap, const float* sink, const float* slopes,
                                             const float* gate, long gate_ld, int od, hipStream_t stream) {
  if (tokens < 0 || hq <= 0 || hkv <= 0 || d <= 0 || page_size <= 0 || max_blocks <= 0) return ATOM_BAD_SHAPE;
  if (hq % hkv || window < 0 || chunk < 0 || softcap < 0.f) return ATOM_BAD_SHAPE;
  if (od <= 0 || od > d || (gate != nullptr && gate_ld < hq)) return ATOM_BAD_SHAPE;
  if (d > kAttnItems) return ATOM_TOO_LARGE;
  if (hq > 65535) return ATOM_TOO_LARGE;
  if (tokens == 0) return ATOM_OK;
  // four keys' entries, or an entry of four keys, a load where they begin at multiples of their size in memory
  const size_t four = dtype == ATOM_F32 ? 16 : 8;
  const int key_fours = d % 4 == 0 && (uintptr_t)k_cache % four == 0;
  const int value_fours = page_size % 4 == 0 && (uintptr_t)v_cache % four == 0;
#define LAUNCH(PER, HEADS)                                                                                           \
  ATOM_DISPATCH_DTYPE(dtype, hipLaunchKernelGGL((paged_attention_generic_kernel<T, PER, HEADS>), dim3(tokens, hq / (HEADS)), \
                                                 dim3(kAttnItems / PER),                                             \
                                                 (HEADS) * ((d + 3) / 4 * 4 + kAttnChunk + 16 + kAttnItems) * sizeof(float), \
                                                 stream, (const T*)q, (const T*)k_cache, (const T*)v_cache, (T*)out,  \
                                                 token_seq, positions, block_tables, max_blocks, hq, hkv, d, page_size, \
                                                 scale, window, chunk, softcap, sink, slopes, gate, gate_ld, od, key_fours, \
                                                 value_fours))
  const int heads = atom_paged_attention_generic_heads(tokens, hq, hkv);
  if (heads == 0) LAUNCH(1, 1);
  else if (heads == 4) LAUNCH(4, 4);
  else if (heads == 2) LAUNCH(4, 2);
  else LAUNCH(4, 1);
#undef LAUNCH
  return launch_status();
}
