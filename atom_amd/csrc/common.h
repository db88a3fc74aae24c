// Shared device helpers for the gfx950 kernels: element types, wave and block
// reductions.  A wavefront has 64 lanes on CDNA; every reduction below assumes it.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#define ATOM_EXPORT extern "C" __attribute__((visibility("default")))

// Element type codes of the C interface.
enum AtomDtype : int { ATOM_F32 = 0, ATOM_BF16 = 1 };

// Return codes of the C interface (0 = launched).
enum AtomStatus : int {
  ATOM_OK = 0,
  ATOM_BAD_DTYPE = 1,
  ATOM_BAD_SHAPE = 2,
  ATOM_UNSUPPORTED = 3,
  ATOM_LAUNCH_FAILED = 4,
  ATOM_TOO_LARGE = 5,
};

typedef __bf16 bf16_t;

constexpr int kWave = 64;

__device__ __forceinline__ float to_f32(float v) { return v; }
__device__ __forceinline__ float to_f32(bf16_t v) { return static_cast<float>(v); }

template <typename T>
__device__ __forceinline__ T from_f32(float v);
template <>
__device__ __forceinline__ float from_f32<float>(float v) { return v; }
template <>
__device__ __forceinline__ bf16_t from_f32<bf16_t>(float v) { return static_cast<bf16_t>(v); }

// Blocks of 256 threads that share one row of `entries` where a row is only copied or looked up: four entries a thread, which
// are in flight together.  With one block a row and its loads one after the other: 6.4 us for four rows of 2,048 bfloat16
// entries, 8.1 for two of 4,096 float32; so 3.2 and 4.7.
static inline unsigned blocks_of_row(int entries) {
  const int blocks = entries / 1024 + (entries % 1024 != 0);
  return blocks < 1024 ? blocks : 1024;
}

// Token ids that are still on the device: token t's id is sampled[source[t]] where that names one of the `count` sampled rows (what
// the last step's sampler left there), else ids[t].  A kernel that looks tokens up takes them so and leaves them in ids for the
// kernels behind it (a launch of its own before an embedding of few tokens is 4 us of a decode step).
struct FedTokens {
  const int* source;   // null: ids as they are
  const int* sampled;
  int count;
};

__device__ __forceinline__ int fed_id(int* ids, int t, const FedTokens& fed, bool leaves) {
  const int src = fed.source != nullptr ? fed.source[t] : -1;
  if (src < 0 || src >= fed.count) return ids[t];
  const int id = fed.sampled[src];
  if (leaves) ids[t] = id;   // (nobody reads the old one: whoever looks this token up goes by its source)
  return id;
}

// Four neighbouring elements of either type as float32.
template <typename T>
struct alignas(4 * sizeof(T)) Four {
  T at[4];
  __device__ __forceinline__ void to(float* v) const {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = to_f32(at[e]);
  }
  __device__ __forceinline__ void from(const float* v) {
#pragma unroll
    for (int e = 0; e < 4; ++e) at[e] = from_f32<T>(v[e]);
  }
};

// v of the lane N places further on in the lane's row of 16, around its end.
template <int N>
__device__ __forceinline__ float row_turned(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + N, 0xf, 0xf, false));
}

// Sum (maximum) over a wavefront whose lanes are all active, in every lane.  Halves, rows of 16 lanes, then lanes 8, 4,
// 2 and 1 apart: the halves and rows change places in registers, and inside a row a turn by N lanes meets the lane at
// distance N, because the values repeat every 2 N lanes by then.  No step goes through LDS, whose six round trips were
// about a microsecond of every kernel of a small step that sums over a block twice.
__device__ __forceinline__ float wave_sum(float v) {
  const unsigned bits = __float_as_uint(v);
  const auto a = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
  const unsigned half = __float_as_uint(__uint_as_float(a[0]) + __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane16_swap(half, half, false, false);
  v = __uint_as_float(b[0]) + __uint_as_float(b[1]);
  v += row_turned<8>(v);
  v += row_turned<4>(v);
  v += row_turned<2>(v);
  v += row_turned<1>(v);
  return v;
}

__device__ __forceinline__ float wave_max(float v) {
  const unsigned bits = __float_as_uint(v);
  const auto a = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
  const unsigned half = __float_as_uint(fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1])));
  const auto b = __builtin_amdgcn_permlane16_swap(half, half, false, false);
  v = fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
  v = fmaxf(v, row_turned<8>(v));
  v = fmaxf(v, row_turned<4>(v));
  v = fmaxf(v, row_turned<2>(v));
  v = fmaxf(v, row_turned<1>(v));
  return v;
}

// The maximum (the sum) of v over the four lanes r, r + 16, r + 32 and r + 48, in each of them.  The rows of 16
// lanes change places through the row-swap instructions of gfx950, without a trip through LDS: the first leaves
// rows (0, 0, 2, 2) of v in one register and rows (1, 1, 3, 3) in the other, the second the lower half of its
// operand twice in one and the upper half twice in the other.
__device__ __forceinline__ float rows_max(float v) {
  const unsigned bits = __float_as_uint(v);
  const auto a = __builtin_amdgcn_permlane16_swap(bits, bits, false, false);
  const unsigned pair = __float_as_uint(fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1])));
  const auto b = __builtin_amdgcn_permlane32_swap(pair, pair, false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

__device__ __forceinline__ float rows_sum(float v) {
  const unsigned bits = __float_as_uint(v);
  const auto a = __builtin_amdgcn_permlane16_swap(bits, bits, false, false);
  const unsigned pair = __float_as_uint(__uint_as_float(a[0]) + __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(pair, pair, false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Sum over a block of up to 1024 threads; `scratch` holds one float per wave
// (16 at most).  Every thread receives the total.  The order of the partial sums
// is fixed, so the result does not depend on what else runs.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int waves = (blockDim.x + kWave - 1) / kWave;
  v = wave_sum(v);
  __syncthreads();  // scratch may still be read from a previous call
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float total = 0.f;
  for (int w = 0; w < waves; ++w) total += scratch[w];
  return total;
}

__device__ __forceinline__ float block_max(float v, float* scratch) {
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int waves = (blockDim.x + kWave - 1) / kWave;
  v = wave_max(v);
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float total = scratch[0];
  for (int w = 1; w < waves; ++w) total = fmaxf(total, scratch[w]);
  return total;
}

// The CUs of the current device, asked for once per device: what the launch plans count blocks against (256 on
// the MI355X that their other figures were measured on; also the answer where no device can be asked).
static inline int device_cus() {
  static int known[16] = {0};
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 16) return 256;
  if (!known[device]) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus <= 0) cus = 256;
    known[device] = cus;
  }
  return known[device];
}

static inline int launch_status() {
  return hipGetLastError() == hipSuccess ? ATOM_OK : ATOM_LAUNCH_FAILED;
}

// Calls `fn.template operator()<T>()` with the element type that `dtype` names.
#define ATOM_DISPATCH_DTYPE(dtype, ...)                 \
  do {                                                  \
    if ((dtype) == ATOM_F32) {                          \
      using T = float;                                  \
      __VA_ARGS__;                                      \
    } else if ((dtype) == ATOM_BF16) {                  \
      using T = bf16_t;                                 \
      __VA_ARGS__;                                      \
    } else {                                            \
      return ATOM_BAD_DTYPE;                            \
    }                                                   \
  } while (0)
