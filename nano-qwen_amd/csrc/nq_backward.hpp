// Parameters shared by the attention backward kernels (bf16 MFMA and fp32
// MFMA forms).
#pragma once

#include "nq_common.hpp"

namespace nq {

struct BwdParams {
  const void* q;
  const void* k;
  const void* v;
  const void* o;
  const void* dout;
  const float* lse;  // (B, Hq, S) natural log
  // scratch written by bwd_dq_kernel: per (batch, head) and 32-row query
  // tile, 64 floats = [32 x LSE * log2(e) | 32 x Delta], rows past S zero
  float* ws;
  int nst;           // 32-row tiles per (batch, head)
  void* dq;
  void* dk;
  void* dv;
  int64_t qsb, qsh, qss, ksb, ksh, kss, vsb, vsh, vss;
  int64_t osb, osh, oss, dosb, dosh, doss;
  int64_t dqsb, dqsh, dqss, dksb, dksh, dkss, dvsb, dvsh, dvss;
  int B, Hq, Hkv, G, S, T, BM, nqb, coff;
  float scale, scale_log2;
  // key padding: sequence b attends keys [0, kv_lens[b]) (clamped to
  // [0, T]; the rest get zero gradients); NULL = all T keys
  const int32_t* kv_lens;
  // additive attention bias as in the forward (bias[b, h, i, j], keys
  // contiguous, rows readable up to T rounded up to 8), and its transpose
  // bias_t[b, h, j, i] (queries contiguous, rows readable up to S rounded up
  // to 8) for the dK/dV kernel, whose lanes hold keys; NULL = no bias
  const void* bias;
  int64_t bsb, bsh, bss;
  const void* bias_t;
  int64_t btsb, btsh, btss;
  // dK/dV: a key block's steps split over nsplit workgroups of `run` steps
  // each (1 = none), whose partial sums go to part
  int nsplit, run;
  float* part;
  int kblk_turn;  // bf16 dK/dV, causal: the rank from which key blocks go lightest first
  // fp32 dQ: a query block's key tiles split likewise (f32_key_runs), whose
  // partials use the same memory before it
  int qsplit, qrun;
};

// Keys sequence b attends.
__device__ __forceinline__ int bw_keys(const BwdParams& p, int b) {
  if (!p.kv_lens) return p.T;
  const int l = p.kv_lens[b];
  return l < 0 ? 0 : (l > p.T ? p.T : l);
}

// Scratch slot of query row s of (batch b, head h): LSE * log2(e) at the
// returned index, Delta 32 floats later.
__device__ __forceinline__ int64_t bw_ws_index(const BwdParams& p, int b, int h, int s) {
  return (((int64_t)b * p.Hq + h) * p.nst + s / 32) * 64 + (s & 31);
}

// ---- split dK/dV.  A key block's work is a list of steps (32-row query tiles of
// each of its G heads).  Run s of a block takes steps [s * run, (s + 1) * run); a
// block with one run writes its rows itself, the others leave their
// accumulators in p.part, in lane order (per block and run: 4 waves x dK, dV x
// D/32 x 4 x 64 lanes float4), for bwd_dkdv_merge_kernel.
constexpr int BW_SPLIT_KEYS = 128;  // keys per block, 32 per wave
__device__ __forceinline__ int bw_first_query(const BwdParams& p, bool causal, int k0, int tile) {
  return causal ? max(0, k0 - p.coff) / tile * tile : 0;
}
// Steps of the block at key k0 (0: no query sees it, or it is all padding).
__device__ __forceinline__ int bw_steps(const BwdParams& p, bool causal, int b, int k0) {
  const int q = bw_first_query(p, causal, k0, 32);
  return q < p.S && k0 < bw_keys(p, b) ? p.G * ((p.S - q + 31) / 32) : 0;
}
__device__ __forceinline__ int bw_runs(const BwdParams& p, int steps) {
  return steps > p.run ? (steps + p.run - 1) / p.run : 1;
}
template <int D>
__device__ __forceinline__ floatx4* bw_part(const BwdParams& p, int blk, int pair, int run, int wave) {
  const int64_t slot = (((int64_t)blk * p.B * p.Hkv + pair) * p.nsplit + run) * 4 + wave;
  return reinterpret_cast<floatx4*>(p.part) + slot * (2 * (D / 32) * 4 * 64);
}
// This wave's accumulators into its run's partials.
template <int D>
__device__ __forceinline__ void bw_store_part(const BwdParams& p, int blk, int pair, int run, int wave, int lane,
                                              const floatx16* dk, const floatx16* dv) {
  floatx4* o = bw_part<D>(p, blk, pair, run, wave) + lane;
#pragma unroll
  for (int dd = 0; dd < D / 32; ++dd)
#pragma unroll
    for (int gq = 0; gq < 4; ++gq) {
      o[(dd * 4 + gq) * 64] = floatx4{dk[dd][gq * 4], dk[dd][gq * 4 + 1], dk[dd][gq * 4 + 2], dk[dd][gq * 4 + 3]};
      o[(D / 8 + dd * 4 + gq) * 64] =
          floatx4{dv[dd][gq * 4], dv[dd][gq * 4 + 1], dv[dd][gq * 4 + 2], dv[dd][gq * 4 + 3]};
    }
}

// Sums the partials of the blocks with several runs, in run order: a workgroup
// takes the 32 keys of one wave, its wave (dK or dV, dd) their dims 32dd ..
// 32dd + 31 in the accumulators' lane order.  HBM- or L2-bound.
template <int D, typename T, bool CAUSAL>
__global__ void __launch_bounds__(4 * D) bwd_dkdv_merge_kernel(BwdParams p) {
  constexpr int NDO = D / 32;
  const int lane = threadIdx.x & 63, part = threadIdx.x >> 6;
  const int npairs = p.B * p.Hkv;
  const int wave = blockIdx.x & 3, pair = (blockIdx.x >> 2) % npairs, blk = (blockIdx.x >> 2) / npairs;
  const int b = pair / p.Hkv, kvh = pair % p.Hkv;
  const int runs = bw_runs(p, bw_steps(p, CAUSAL, b, blk * BW_SPLIT_KEYS));
  if (runs == 1) return;
  const int isv = part / NDO, dd = part % NDO;
  floatx4 a[4] = {floatx4{}, floatx4{}, floatx4{}, floatx4{}};
  const floatx4* src = bw_part<D>(p, blk, pair, 0, wave) + part * 256 + lane;
  for (int s = 0; s < runs; ++s, src += 4 * (2 * NDO * 4 * 64)) {
#pragma unroll
    for (int gq = 0; gq < 4; ++gq) a[gq] += src[gq * 64];
  }
  const int key = blk * BW_SPLIT_KEYS + wave * 32 + (lane & 31);
  if (key >= p.T) return;
  T* out = isv ? reinterpret_cast<T*>(p.dv) + b * p.dvsb + kvh * p.dvsh + (int64_t)key * p.dvss
               : reinterpret_cast<T*>(p.dk) + b * p.dksb + kvh * p.dksh + (int64_t)key * p.dkss;
  const float f = isv ? 1.0f : p.scale;
#pragma unroll
  for (int gq = 0; gq < 4; ++gq) store4<T>(out + dd * 32 + gq * 8 + (lane >> 5) * 4, a[gq] * f);
}

template <int D, typename T>
inline hipError_t launch_dkdv_merge(const BwdParams& p, bool causal, hipStream_t st) {
  const dim3 grid((unsigned)(((p.T + BW_SPLIT_KEYS - 1) / BW_SPLIT_KEYS) * p.B * p.Hkv * 4)), block(4 * D);
  if (causal) hipLaunchKernelGGL((bwd_dkdv_merge_kernel<D, T, true>), grid, block, 0, st, p);
  else hipLaunchKernelGGL((bwd_dkdv_merge_kernel<D, T, false>), grid, block, 0, st, p);
  return hipGetLastError();
}

// The fp32 backward (every tensor fp32; products on v_mfma_f32_32x32x2_f32).
hipError_t launch_bwd_f32(const BwdParams& p, int D, bool causal, hipStream_t st);

// The head_dim 256 backward (bf16, no key lengths or bias): dQ with Delta,
// then dK/dV; p.nqb counts 64-row query blocks.
hipError_t launch_bwd_wide(const BwdParams& p, bool causal, hipStream_t st);

}  // namespace nq
