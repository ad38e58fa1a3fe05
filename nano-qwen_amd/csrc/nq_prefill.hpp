// Parameters shared by the prefill kernels (bf16 MFMA and fp32 MFMA forms).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace nq {

struct PrefillParams {
  const void* q;
  const void* k;
  const void* v;
  void* o;
  float* lse;
  int64_t qsb, qsh, qss;
  int64_t ksb, ksh, kss;
  int64_t vsb, vsh, vss;
  int64_t osb, osh, oss;
  const float* qw;  // bf16 when q16
  int q16;
  float eps;
  const float* cos_tab;
  const float* sin_tab;
  int max_pos;
  const int32_t* q_pos;
  const int32_t* q_pos_base;
  int q_pos0;
  int B, Hq, Hkv, G, S, T, BM, nqb;
  float scale_log2;  // sm_scale * log2(e)
  // Per-sequence key counts (key padding, ragged or paged caches): sequence
  // b holds keys [0, kv_lens[b] + kv_extra), or none if kv_lens[b] lies
  // outside [0, kv_max - kv_extra] (its rows then come out NaN; a sequence
  // with no keys gives zeros); NULL = every sequence holds T.  With kv_lens
  // and neither q_pos nor q_pos0 >= 0 (decode), a query sits at position
  // keys - 1.
  const int32_t* kv_lens;
  int kv_extra, kv_max;
  // paged K/V (NULL bt = dense): key t of sequence b is row t % page of page
  // bt[b * bts + t / page], strides (ksb, ksh, kss) = (page, head, row)
  const int32_t* bt;
  int64_t bts;
  int page;
  // additive attention bias (SDPA's attn_mask: a bool mask as 0 / -inf, or a
  // float mask), in the kernel's element type: bias[b, h, i, j] at
  // b * bsb + h * bsh + i * bss + j (0 strides broadcast), each row's keys
  // contiguous and readable up to T rounded up to a multiple of 8
  const void* bias;
  int64_t bsb, bsh, bss;
  // keys split over nsplit workgroups per query block (bf16 form; 1 = none),
  // whose partials go to ws
  int nsplit;
  float* ws;
  int run;  // fp32 form: tiles per workgroup of a split launch
};

// How the fp32 kernels that own query rows (the prefill, the backward's dQ)
// deal a query block's 32-key tiles to workgroups: runs of `len` tiles, `n` for
// the longest block, n = 1 for none.  A launch of fewer workgroups than two per
// CU leaves the device to its heaviest blocks (B2 S1000 8/2 heads D64: 128
// workgroups of 1 to 32 tiles, 90 us whole and 54 in runs): runs of the length that
// gives two workgroups per CU the same work, at least F32_MIN_RUN tiles, at most
// F32_MAX_RUNS of them, whose partials the merge adds one after another.
//
// They are taken where this estimate says that they pay.  Unit: the time for a tile
// of a workgroup that has its CU to itself, tile_us; dQ takes twice the prefill's.  The
// prefill's workspace is sized without knowing the mask, so that counts on a causal
// one; a full launch then leaves it unused where its own estimate says so.  Whole, a launch lasts as long as its longest block or an
// even share of all tiles.  Split, it lasts
//   - one run where every run has a CU to itself;
//   - up to `fit` runs per CU (by registers): two runs, as they take turns, or the share;
//   - beyond that the share, and on average half of a run that ends last;
//   - with a multiple of 4 runs per causal block, where they have no CU each and fit <= 2:
//     the first runs of all blocks come to lie on the same CUs, and the launch lasts as
//     if every block had them all;
// and 5 us for the merge launch, and the partials' way out and back at 4 TB/s.
// Of 200 prefills drawn at random, 1 to 511 workgroups, none is 2% slower than whole
// (22 of 110 were without this) and they take 0.56 of the time.  Left out are, whole /
// split: B16 1/1 heads S3863 D128 703 / 1002 us, B1 16/2 S2461 D128 392 / 537, B16 8/1
// S239 D128 50 / 63, B3 64/16 S277 D32 22 / 29; the backward by dQ's, B16 32/4 S53 T172
// D128 241 / 262, B4 8/1 S1239 D64 1779 / 1825.  Below ~12 us of tiles a call lasts as
// long as the host takes to launch it, and a second launch adds to that.
constexpr int F32_MIN_RUN = 4, F32_MAX_RUNS = 32;
struct KeyRuns { int n, len; };
inline KeyRuns f32_key_runs(int B, int Hq, int Hkv, int S, int T, int D, bool dq = false, bool causal = true) {
  if (128 % (Hq / Hkv)) return {1, 1};
  const int BM = 128 / (Hq / Hkv);
  const int64_t wgs = (int64_t)B * Hkv * ((S + BM - 1) / BM);
  const int64_t most = ((int64_t)T + 31) / 32;
  if (wgs >= 512) return {1, 1};
  const int64_t half = wgs * ((int64_t)T - (S < T ? S : T) / 2) / 32;  // a causal row's keys on average
  int64_t len = (half + 511) / 512;
  const int least = most <= 6 ? 3 : F32_MIN_RUN;
  if (len < least) len = least;
  if (len * F32_MAX_RUNS < most) len = (most + F32_MAX_RUNS - 1) / F32_MAX_RUNS;
  const int64_t n = (most + len - 1) / len;
  const int fit = D == 32 ? 4 : D == 64 ? 2 : 1;
  const double tile_us = (D == 32 ? 1.62 : D == 64 ? 2.78 : 5.05) * (dq ? 2 : 1);
  const double tiles = causal ? half : wgs * (T / 32.0), share = tiles / 256;
  const double mean = tiles / wgs / len + (dq ? 0.5 : 1);  // runs of a block
  const double runs = wgs * (mean < n ? mean : n);
  double whole = most > share ? most : share;
  if (!causal && fit == 1) whole = (double)((wgs + 255) / 256 * most);  // all blocks alike
  double split = len;
  if (runs > 256 * fit) split = share + 0.5 * len / fit;
  else if (runs > 256) split = 2 * len > share ? 2 * len : share;
  if (causal && fit <= 2 && n % 4 == 0 && runs > 256 && wgs * n * len > 256 * split) split = wgs * n * len / 256.0;
  if (whole * tile_us < 12.4 || split * tile_us + 5.0 + runs * 1024 * D / 4e6 >= whole * tile_us) return {1, 1};
  return {(int)n, (int)len};
}
// Floats of one workgroup's partial accumulators, 4 waves of 32 rows.
constexpr int64_t f32_part(int D) { return 128 * (int64_t)D; }

// Keys of sequence b (-1: a length out of range).
__device__ __forceinline__ int pf_keys(const PrefillParams& p, int b) {
  if (!p.kv_lens) return p.T;
  const int l = ld_uniform(p.kv_lens, b);
  return (l < 0 || l > p.kv_max - p.kv_extra) ? -1 : l + p.kv_extra;
}

// The fp32 prefill (q, k, v, o all fp32; products on v_mfma_f32_32x32x2_f32).
// p.BM must be 128 / G (4 waves of 32 query rows).
hipError_t launch_prefill_f32(const PrefillParams& p, int D, bool causal, bool fuse, hipStream_t st);

// Plain bf16 attention at head_dim 256 (no fusion, key lengths, bias or
// pages); p.nqb counts 64-row query blocks.
hipError_t launch_prefill_wide(const PrefillParams& p, bool causal, hipStream_t st);

}  // namespace nq
