// Kernels around a float32 residual stream that is normed after every sum, and the step between a packed q | k | v
// product and attention over pages whose value heads have a size of their own.
//
//   sum_norm        stream <- rms_norm(alpha * stream + sum_i scale_i * y_i) * w   (w null: the sum alone; alpha 0:
//                   the stream is not read), up to four summands of float32 or bfloat16, all in float32; the new
//                   rows optionally also in another type for the products that read them next
//   shift_rows      out[t] = x[t] + (x[t - 1] - x[t]) * mu; the row before a request's first token of the step is what
//                   its state slot holds (float32), and the request's last row of the step is left there
//   qkv_rot_write   per token: RMS norm of every q and k head with a weight per entry (no weight: no norm), rotation
//                   of the pairs (i, i + rot_dims / 2) of every head by position * freq[i] (float64 angle, reduced,
//                   float32 sine and cosine), values optionally kept as they are (float32) and optionally blended
//                   with another layer's, v <- (1 - l) v + l v_source; q goes to q_out [T, H, D], k to the key pages
//                   [pages, G, page, D], v to the value pages [pages, G, DV, page]
#include "common.h"

struct SumTerms {
  const void* y[4];
  int dtype[4];
  float scale[4];
  int n;
};

__device__ __forceinline__ float term_at(const void* y, int dtype, size_t at) {
  return dtype == ATOM_F32 ? static_cast<const float*>(y)[at] : to_f32(static_cast<const bf16_t*>(y)[at]);
}

template <typename T>
__global__ void __launch_bounds__(256)
sum_norm_kernel(float* __restrict__ stream, float alpha, SumTerms terms, const float* __restrict__ weight, float eps,
                T* __restrict__ out, int width) {
  extern __shared__ float row[];
  __shared__ float scratch[16];
  const size_t base = (size_t)blockIdx.x * width;
  float ss = 0.f;
#pragma unroll 4
  for (int i = threadIdx.x; i < width; i += blockDim.x) {
    float v = alpha != 0.f ? alpha * stream[base + i] : 0.f;
    // the terms by constant index, so that the argument's arrays stay in scalar registers
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (k < terms.n) v += terms.scale[k] * term_at(terms.y[k], terms.dtype[k], base + i);
    row[i] = v;
    ss += v * v;
  }
  float inv = 1.f;
  if (weight != nullptr) inv = 1.f / sqrtf(block_sum(ss, scratch) / (float)width + eps);
#pragma unroll 4
  for (int i = threadIdx.x; i < width; i += blockDim.x) {   // a thread reads back what it wrote itself
    const float v = weight != nullptr ? row[i] * inv * weight[i] : row[i];
    stream[base + i] = v;
    if (out != nullptr) out[base + i] = from_f32<T>(v);
  }
}

// The same with a row in registers, four entries a thread and access, every load of the row asked for before any is
// waited for: width % 4 = 0 and at most 1,024 V entries.
typedef __attribute__((ext_vector_type(4))) float sn_f32x4;
typedef __attribute__((ext_vector_type(4))) __bf16 sn_bf16x4;

// SHIFT: every request brings one token, and `out` receives the new rows as shift_rows blends them, out = x + (x' - x) * mu
// with x' what the request's slot holds, where the new row is left.  (Two rows of 2,048: 3.6 us behind a sum_norm of 4.0 in a
// launch of its own; three of them in a step of 1 / 4 / 8 / 64 requests, width 2,048: 4.5 / 5.4 / 7.8 / 7.8 us less.)
struct ShiftOne {
  const float* mu;
  float* state;
  long slot_stride, state_off;
  const int* slot_of_seq;
  const int* token_seq;
};

template <typename T, int V, bool SHIFT>
__global__ void __launch_bounds__(256)
sum_norm_vec_kernel(float* __restrict__ stream, float alpha, SumTerms terms, const float* __restrict__ weight, float eps,
                    T* __restrict__ out, int width, ShiftOne shift) {
  __shared__ float scratch[16];
  const size_t base = (size_t)blockIdx.x * width;
  sn_f32x4 v[V], w[V];
  float* kept = nullptr;
  if constexpr (SHIFT) {
    const int seq = shift.token_seq[blockIdx.x], slot = seq >= 0 ? shift.slot_of_seq[seq] : -1;
    if (slot >= 0) kept = shift.state + (size_t)slot * shift.slot_stride + shift.state_off;
  }
#pragma unroll
  for (int j = 0; j < V; ++j) {
    const int i = (threadIdx.x + 256 * j) * 4;
    v[j] = w[j] = sn_f32x4{0.f, 0.f, 0.f, 0.f};
    if (i < width) {
      if (alpha != 0.f) v[j] = *reinterpret_cast<const sn_f32x4*>(stream + base + i);
      if (weight != nullptr) w[j] = *reinterpret_cast<const sn_f32x4*>(weight + i);
    }
  }
#pragma unroll
  for (int j = 0; j < V; ++j) v[j] *= alpha;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (k >= terms.n) break;
    sn_f32x4 y[V];
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const int i = (threadIdx.x + 256 * j) * 4;
      y[j] = sn_f32x4{0.f, 0.f, 0.f, 0.f};
      if (i < width) {
        if (terms.dtype[k] == ATOM_F32) {
          y[j] = *reinterpret_cast<const sn_f32x4*>(static_cast<const float*>(terms.y[k]) + base + i);
        } else {
          const sn_bf16x4 b = *reinterpret_cast<const sn_bf16x4*>(static_cast<const bf16_t*>(terms.y[k]) + base + i);
#pragma unroll
          for (int q = 0; q < 4; ++q) y[j][q] = static_cast<float>(b[q]);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < V; ++j) v[j] += terms.scale[k] * y[j];
  }
  sn_f32x4 prev[SHIFT ? V : 1], mu[SHIFT ? V : 1];
  if constexpr (SHIFT) {
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const int i = (threadIdx.x + 256 * j) * 4;
      prev[j] = mu[j] = sn_f32x4{0.f, 0.f, 0.f, 0.f};
      if (i < width) {
        if (kept != nullptr) prev[j] = *reinterpret_cast<const sn_f32x4*>(kept + i);
        mu[j] = *reinterpret_cast<const sn_f32x4*>(shift.mu + i);
      }
    }
  }
  float inv = 1.f;
  if (weight != nullptr) {
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < V; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) ss += v[j][q] * v[j][q];
    inv = 1.f / sqrtf(block_sum(ss, scratch) / (float)width + eps);
  }
#pragma unroll
  for (int j = 0; j < V; ++j) {
    const int i = (threadIdx.x + 256 * j) * 4;
    if (i >= width) break;
    sn_f32x4 o = weight != nullptr ? v[j] * inv * w[j] : v[j];
    *reinterpret_cast<sn_f32x4*>(stream + base + i) = o;
    if constexpr (SHIFT) {
      if (kept != nullptr) *reinterpret_cast<sn_f32x4*>(kept + i) = o;
      o = o + (prev[j] - o) * mu[j];
    }
    if (out != nullptr) {
      if constexpr (sizeof(T) == 2) {
        sn_bf16x4 b;
#pragma unroll
        for (int q = 0; q < 4; ++q) b[q] = static_cast<__bf16>(o[q]);
        *reinterpret_cast<sn_bf16x4*>(out + base + i) = b;
      } else {
        *reinterpret_cast<sn_f32x4*>(out + base + i) = o;
      }
    }
  }
}

ATOM_EXPORT int atom_sum_norm(float* stream, float alpha, const void* y0, int d0, float s0, const void* y1, int d1,
                              float s1, const void* y2, int d2, float s2, const void* y3, int d3, float s3, int n,
                              const float* weight, float eps, void* out, int out_dtype, int rows, int width,
                              hipStream_t stream_id) {
  if (rows < 0 || width <= 0 || n < 0 || n > 4 || stream == nullptr) return ATOM_BAD_SHAPE;
  if (width > 15360) return ATOM_TOO_LARGE;
  SumTerms terms{{y0, y1, y2, y3}, {d0, d1, d2, d3}, {s0, s1, s2, s3}, n};
  for (int i = 0; i < n; ++i) {
    if (terms.y[i] == nullptr) return ATOM_BAD_SHAPE;
    if (terms.dtype[i] != ATOM_F32 && terms.dtype[i] != ATOM_BF16) return ATOM_BAD_DTYPE;
  }
  if (rows == 0) return ATOM_OK;
  const size_t smem = (size_t)width * sizeof(float);
  if (out == nullptr) out_dtype = ATOM_F32;
  bool vec = width % 4 == 0 && width <= 8192 && (size_t)stream % 16 == 0 && (size_t)weight % 16 == 0 && (size_t)out % 16 == 0;
  for (int i = 0; i < n; ++i) vec = vec && (size_t)terms.y[i] % 16 == 0;
  if (vec) {
#define ATOM_SUM_NORM_VEC(V)                                                                                        \
  ATOM_DISPATCH_DTYPE(out_dtype, hipLaunchKernelGGL((sum_norm_vec_kernel<T, V, false>), dim3(rows), dim3(256), 0, stream_id, \
                                                     stream, alpha, terms, weight, eps, (T*)out, width, ShiftOne{}))
    if (width <= 1024) ATOM_SUM_NORM_VEC(1);
    else if (width <= 2048) ATOM_SUM_NORM_VEC(2);
    else if (width <= 4096) ATOM_SUM_NORM_VEC(4);
    else ATOM_SUM_NORM_VEC(8);
#undef ATOM_SUM_NORM_VEC
    return launch_status();
  }
  ATOM_DISPATCH_DTYPE(out_dtype, hipLaunchKernelGGL((sum_norm_kernel<T>), dim3(rows), dim3(256), smem, stream_id, stream,
                                                     alpha, terms, weight, eps, (T*)out, width));
  return launch_status();
}

// The same with the rows blended with their predecessors on the way out; every request brings one token.  ATOM_UNSUPPORTED where
// the rows cannot be read four entries at a time.
ATOM_EXPORT int atom_sum_norm_shift(float* stream, float alpha, const void* y0, int d0, float s0, const void* y1, int d1,
                                    float s1, const void* y2, int d2, float s2, const void* y3, int d3, float s3, int n,
                                    const float* weight, float eps, void* out, int out_dtype, int rows, int width,
                                    const float* mu, float* state, long slot_stride, long state_off, const int* slot_of_seq,
                                    const int* token_seq, hipStream_t stream_id) {
  if (rows < 0 || width <= 0 || n < 0 || n > 4 || !stream || !out || !weight) return ATOM_BAD_SHAPE;
  if (!mu || !state || !slot_of_seq || !token_seq || state_off < 0 || slot_stride < state_off + width) return ATOM_BAD_SHAPE;
  SumTerms terms{{y0, y1, y2, y3}, {d0, d1, d2, d3}, {s0, s1, s2, s3}, n};
  uintptr_t ends = (uintptr_t)stream | (uintptr_t)weight | (uintptr_t)out | (uintptr_t)mu | (uintptr_t)state;
  for (int i = 0; i < n; ++i) {
    if (terms.y[i] == nullptr) return ATOM_BAD_SHAPE;
    if (terms.dtype[i] != ATOM_F32 && terms.dtype[i] != ATOM_BF16) return ATOM_BAD_DTYPE;
    ends |= (uintptr_t)terms.y[i];
  }
  if (width % 4 || width > 8192 || ends % 16 || slot_stride % 4 || state_off % 4) return ATOM_UNSUPPORTED;
  if (rows == 0) return ATOM_OK;
  const ShiftOne shift{mu, state, slot_stride, state_off, slot_of_seq, token_seq};
#define ATOM_SUM_NORM_SHIFT(V)                                                                                              \
  ATOM_DISPATCH_DTYPE(out_dtype, hipLaunchKernelGGL((sum_norm_vec_kernel<T, V, true>), dim3(rows), dim3(256), 0, stream_id, \
                                                     stream, alpha, terms, weight, eps, (T*)out, width, shift))
  if (width <= 1024) ATOM_SUM_NORM_SHIFT(1);
  else if (width <= 2048) ATOM_SUM_NORM_SHIFT(2);
  else if (width <= 4096) ATOM_SUM_NORM_SHIFT(4);
  else ATOM_SUM_NORM_SHIFT(8);
#undef ATOM_SUM_NORM_SHIFT
  return launch_status();
}

// Entries of a row a block takes.  Few tokens: two a thread, so that they are more than a few blocks.  From four tokens a CU on
// a whole row (bfloat16, 4,096 rows of 8,192 in pieces and whole: 64 and 48 us, of 2,048 19.5 and 16.4).
constexpr int kShiftSpan = 512;

template <typename TI, typename TO>
__global__ void __launch_bounds__(256)
shift_rows_kernel(const TI* __restrict__ x, const float* __restrict__ mu, TO* __restrict__ out, float* __restrict__ state,
                  long slot_stride, long state_off, const int* __restrict__ cu_seqlens, const int* __restrict__ slot_of_seq,
                  const int* __restrict__ token_seq, int width, int span) {
  const int t = blockIdx.x;
  const int seq = token_seq[t];
  const bool padding = seq < 0;
  const int first = padding ? t : cu_seqlens[seq];
  const int slot = padding ? -1 : slot_of_seq[seq];
  const bool heads = t == first;             // the request's first token of this step
  const int last = padding ? t : cu_seqlens[seq + 1] - 1;
  float* kept = slot >= 0 ? state + (size_t)slot * slot_stride + state_off : nullptr;
  const TI* row = x + (size_t)t * width;
#pragma unroll 4
  for (int i = blockIdx.y * span + threadIdx.x; i < min(width, (int)(blockIdx.y + 1) * span); i += 256) {
    const float cur = to_f32(row[i]);
    float prev;
    if (heads) {
      // only this thread touches the entry of the slot's row in this launch: it reads the old one and leaves the step's last
      prev = kept != nullptr ? kept[i] : 0.f;
      if (kept != nullptr) kept[i] = to_f32(x[(size_t)last * width + i]);
    } else {
      prev = to_f32(x[(size_t)(t - 1) * width + i]);
    }
    out[(size_t)t * width + i] = from_f32<TO>(cur + (prev - cur) * mu[i]);
  }
}

ATOM_EXPORT int atom_shift_rows(const void* x, int x_dtype, const float* mu, void* out, int out_dtype, float* state,
                                long slot_stride, long state_off, const int* cu_seqlens, const int* slot_of_seq,
                                const int* token_seq, int tokens, int width, hipStream_t stream) {
  if (tokens < 0 || width <= 0 || state_off < 0 || slot_stride < state_off + width) return ATOM_BAD_SHAPE;
  if (x == nullptr || mu == nullptr || out == nullptr || state == nullptr) return ATOM_BAD_SHAPE;
  if (cu_seqlens == nullptr || slot_of_seq == nullptr || token_seq == nullptr) return ATOM_BAD_SHAPE;
  if (tokens == 0) return ATOM_OK;
  const int span = tokens < 4 * device_cus() && width <= 65535 * kShiftSpan ? kShiftSpan : width;
  const dim3 grid(tokens, (width - 1) / span + 1);
#define ATOM_SHIFT(TI, TO)                                                                                          \
  hipLaunchKernelGGL((shift_rows_kernel<TI, TO>), grid, dim3(256), 0, stream, (const TI*)x, mu, (TO*)out,           \
                     state, slot_stride, state_off, cu_seqlens, slot_of_seq, token_seq, width, span)
  if (x_dtype == ATOM_F32 && out_dtype == ATOM_F32) ATOM_SHIFT(float, float);
  else if (x_dtype == ATOM_F32 && out_dtype == ATOM_BF16) ATOM_SHIFT(float, bf16_t);
  else if (x_dtype == ATOM_BF16 && out_dtype == ATOM_BF16) ATOM_SHIFT(bf16_t, bf16_t);
  else if (x_dtype == ATOM_BF16 && out_dtype == ATOM_F32) ATOM_SHIFT(bf16_t, float);
  else return ATOM_BAD_DTYPE;
#undef ATOM_SHIFT
  return launch_status();
}

__device__ __forceinline__ void half_turn_angle(int position, double freq, float* c, float* s) {
  double a = (double)position * freq;
  const double two_pi = 6.283185307179586476925286766559;
  a -= two_pi * floor(a / two_pi);
  sincosf((float)a, s, c);
}

// A wave a (token, head), value heads among them.  A lane owns rotated pairs (i, i + half) and entries behind the rotated
// ones, the first of each kept in registers from the norm on, and forms its pairs' angles itself while the row is on its
// way; nothing goes through LDS.  A block that took all of a token's heads in turn was one long chain of waits in a decode
// step (2 tokens of 16 + 2 x 4 heads: 4.0 us, 10.4 so; 2,305 tokens 21 us, 26.8 so, over two layers of 24 and 12 heads).
template <typename T>
__global__ void __launch_bounds__(256)
qkv_rot_write_kernel(const float* __restrict__ qkv, int ld, T* __restrict__ q_out, T* __restrict__ k_cache,
                     T* __restrict__ v_cache, const float* __restrict__ qw, const float* __restrict__ kw,
                     const double* __restrict__ freq, int rot_dims, const int* __restrict__ positions,
                     const int* __restrict__ slots, int H, int G, int D, int DV, int page_size, float eps,
                     const float* __restrict__ v_source, const float* __restrict__ v_blend, float* __restrict__ v_keep) {
  const size_t t = blockIdx.x;
  const int lane = threadIdx.x & (kWave - 1);
  const int unit = blockIdx.y * (256 / kWave) + threadIdx.x / kWave;
  if (unit >= H + 2 * G) return;
  const float* row = qkv + t * ld;
  const int slot = slots != nullptr ? slots[t] : -1;
  const int page = slot >= 0 ? slot / page_size : 0, off = slot >= 0 ? slot % page_size : 0;
  if (unit >= H + G) {
    const int g = unit - H - G;
    const size_t at = t * G * DV + (size_t)g * DV;     // this head's values among the token's
    const float lam = v_source != nullptr ? v_blend[0] : 0.f;
    const float* src = row + (size_t)(H + G) * D + (size_t)g * DV;
    for (int i = lane; i < DV; i += kWave) {
      float v = src[i];
      if (v_keep != nullptr) v_keep[at + i] = v;
      if (v_source != nullptr) v = (1.f - lam) * v + lam * v_source[at + i];
      if (slot >= 0) v_cache[(((size_t)page * G + g) * DV + i) * page_size + off] = from_f32<T>(v);
    }
    return;
  }
  const bool is_k = unit >= H;
  const float* src = row + (size_t)unit * D;
  const float* w = is_k ? kw : qw;
  const int half = rot_dims / 2;
  constexpr int R = 2;                     // entries behind the rotated ones that a lane keeps
  float lo = 0.f, hi = 0.f, wlo = 1.f, whi = 1.f, c = 1.f, s = 0.f, rest[R], wrest[R];
  const int pos = rot_dims > 0 ? positions[t] : 0;
  if (lane < half) {
    lo = src[lane];
    hi = src[lane + half];
    if (w != nullptr) wlo = w[lane], whi = w[lane + half];
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = rot_dims + lane + r * kWave;
    rest[r] = i < D ? src[i] : 0.f;
    wrest[r] = w != nullptr && i < D ? w[i] : 1.f;
  }
  if (lane < half) half_turn_angle(pos, freq[lane], &c, &s);
  float inv = 1.f;
  if (w != nullptr) {
    float ss = lo * lo + hi * hi;
#pragma unroll
    for (int r = 0; r < R; ++r) ss += rest[r] * rest[r];
    for (int i = lane + kWave; i < half; i += kWave) ss += src[i] * src[i] + src[i + half] * src[i + half];
    for (int i = rot_dims + lane + R * kWave; i < D; i += kWave) ss += src[i] * src[i];
    inv = 1.f / sqrtf(wave_sum(ss) / (float)D + eps);
  }
  if (is_k && slot < 0) return;
  T* dst = is_k ? k_cache + (((size_t)page * G + (unit - H)) * page_size + off) * (size_t)D : q_out + (t * H + unit) * (size_t)D;
  const auto pair = [&](int i, float a, float b, float wa, float wb, float cs, float sn) {
    if (w != nullptr) a *= inv * wa, b *= inv * wb;
    dst[i] = from_f32<T>(a * cs - b * sn);
    dst[i + half] = from_f32<T>(b * cs + a * sn);
  };
  if (lane < half) pair(lane, lo, hi, wlo, whi, c, s);
  for (int i = lane + kWave; i < half; i += kWave) {
    half_turn_angle(pos, freq[i], &c, &s);
    pair(i, src[i], src[i + half], w != nullptr ? w[i] : 1.f, w != nullptr ? w[i + half] : 1.f, c, s);
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = rot_dims + lane + r * kWave;
    if (i < D) dst[i] = from_f32<T>(w != nullptr ? rest[r] * (inv * wrest[r]) : rest[r]);
  }
  for (int i = rot_dims + lane + R * kWave; i < D; i += kWave)
    dst[i] = from_f32<T>(w != nullptr ? src[i] * (inv * w[i]) : src[i]);
}

ATOM_EXPORT int atom_qkv_rot_write(const float* qkv, int ld, void* q_out, void* k_cache, void* v_cache, int dtype,
                                   const float* qw, const float* kw, const double* freq, int rot_dims,
                                   const int* positions, const int* slots, int tokens, int H, int G, int D, int DV,
                                   int page_size, float eps, const float* v_source, const float* v_blend, float* v_keep,
                                   hipStream_t stream) {
  if (tokens < 0 || H <= 0 || G <= 0 || D <= 0 || DV <= 0 || page_size <= 0 || ld < (H + G) * D + G * DV) return ATOM_BAD_SHAPE;
  if (rot_dims < 0 || rot_dims > D || (rot_dims & 1)) return ATOM_BAD_SHAPE;
  if (rot_dims > 0 && (freq == nullptr || positions == nullptr)) return ATOM_BAD_SHAPE;
  if (qkv == nullptr || q_out == nullptr) return ATOM_BAD_SHAPE;
  if (slots != nullptr && (k_cache == nullptr || v_cache == nullptr)) return ATOM_BAD_SHAPE;
  if (v_source != nullptr && v_blend == nullptr) return ATOM_BAD_SHAPE;
  if (tokens == 0) return ATOM_OK;
  if (H + 2L * G > 4L * 65535) return ATOM_TOO_LARGE;
  const dim3 grid(tokens, (H + 2 * G + 3) / 4);
  ATOM_DISPATCH_DTYPE(dtype, hipLaunchKernelGGL((qkv_rot_write_kernel<T>), grid, dim3(256), 0, stream, qkv, ld,
                                                 (T*)q_out, (T*)k_cache, (T*)v_cache, qw, kw, freq, rot_dims, positions,
                                                 slots, H, G, D, DV, page_size, eps, v_source, v_blend, v_keep));
  return launch_status();
}
