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
// They are taken where this estimate says that they pay, from the prefill's tile
// time tile_us (a workgroup alone on its CU; those that share one take turns).
// Whole, a launch lasts as long as its longest block or an even share of the
// tiles.  Split, it lasts one run if the runs have a CU each, else the even share,
// the run that ends last, and a tile for each run's start; then 5 us for the merge
// and the partials' way to memory and back at 3 TB/s.  Over 110 launches of 1 to 496
// workgroups no split it takes was slower than the whole launch; without it 22 were:
// B16 1/1 heads S3863 D128 (496 workgroups) 703 us whole and 1002 split, B1 16/8 S2000
// D128 320 and 348, B3 64/16 S277 D32 22 and 29.  Below ~12 us of tiles a call is as
// long as the host takes to launch it, and a second launch only adds to that.
constexpr int F32_MIN_RUN = 3, F32_MAX_RUNS = 32;
struct KeyRuns { int n, len; };
inline KeyRuns f32_key_runs(int B, int Hq, int Hkv, int S, int T, int D) {
  if (128 % (Hq / Hkv)) return {1, 1};
  const int BM = 128 / (Hq / Hkv);
  const int64_t wgs = (int64_t)B * Hkv * ((S + BM - 1) / BM);
  const int64_t most = ((int64_t)T + 31) / 32;
  if (wgs >= 512) return {1, 1};
  const int64_t tiles = wgs * ((int64_t)T - (S < T ? S : T) / 2) / 32;  // a causal row's keys on average
  int64_t len = (tiles + 511) / 512;
  if (len < F32_MIN_RUN) len = F32_MIN_RUN;
  if (len * F32_MAX_RUNS < most) len = (most + F32_MAX_RUNS - 1) / F32_MAX_RUNS;
  const double tile_us = D == 32 ? 1.62 : D == 64 ? 2.78 : 5.05;
  const double share = tiles / 256.0, each = (double)((most + len - 1) / len);
  const double mean = (double)tiles / wgs / len + 0.5;
  const double runs = wgs * (mean < each ? mean : each);
  const double whole = (most > share ? most : share) * tile_us;
  const double split = (runs <= 256 ? len : share + len + runs / 256) * tile_us + 5.0 + runs * 1024 * D / 3e6;
  if (whole < 12.4 || split >= whole) return {1, 1};
  return {(int)each, (int)len};
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
