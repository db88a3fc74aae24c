// What the kernels for linear recurrences share: their arguments, and how requests are cut into runs.
#pragma once
#include "common.h"

constexpr int kScanStage = 16;   // tokens staged at a time
constexpr int kScanRunTimes = 256;   // floats of scratch memory a run and head takes for its decays, where runs are matrix products

struct ScanArgs {
  const float* r; long ldr; int r_div;       // head h reads r-head h / r_div, K entries each
  const float* k; long ldk; int k_div;
  const float* v; long ldv;                  // [T, H * V] at v
  const float* w; long ldw; int w_per_channel;   // [T, H * K] or [T, H]
  const float* w_bias; int w_mode;           // 0: w is the decay; 1: decay = exp(-exp(w + w_bias[h * K + i]));
                                             // 2 (one decay per head): step = softplus(w + w_bias[h]) multiplies v,
  const float* a_log;                        //    decay = exp(-exp(a_log[h]) step)
  const float* v_scale; long ldvs;           // [T, H] or null
  const float* bonus;                        // [H, K]: read_before; null: read_after
  const float* skip;                         // [H] or null
  float* out; long ldo;                      // [T, H * V]
  float* state; long slot_stride; long state_off;
  const int* cu_seqlens; const int* slot_of_seq;
  int num_seqs, H, K, V, lpc, waves;
  int most;                                  // the walk leaves out requests of more tokens (0: none)
  int run_len;                               // R, a multiple of kScanStage; 0: a request is one run whatever its length
  float* run_state;                          // [places, H, K, V]: B of a run after pass 1, the state before it after pass 2
  float* run_decay;                          // [places, H, K]: the product of a run's decays; [places, H, kScanRunTimes] where
                                             // runs are matrix products
};

// Which request and which of its runs the block with index b works on: the last s with cu[s] / R + s <= b.
__device__ __forceinline__ bool scan_place(const ScanArgs& a, int b, int& seq, int& run, int& runs) {
  if (a.run_len == 0) {
    seq = b; run = 0; runs = 1;
    return true;
  }
  int lo = 0, hi = a.num_seqs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (a.cu_seqlens[mid] / a.run_len + mid <= b) lo = mid; else hi = mid - 1;
  }
  seq = lo;
  const int t0 = a.cu_seqlens[seq], len = a.cu_seqlens[seq + 1] - t0;
  runs = max(1, (len + a.run_len - 1) / a.run_len);
  run = b - (t0 / a.run_len + seq);
  return run >= 0 && run < runs;
}

// Whether the runs of this scan are worked as matrix products (linear_scan_runs.hip), and their launches, which leave out
// requests of one run; `need` is the number of scratch places.
bool scan_runs_takes(const ScanArgs& a);
int scan_runs_launch(const ScanArgs& a, long need, int tokens, hipStream_t stream);
