// The elementwise and row work of a transformer block around its attention and
// GEMMs (model/norm.py:17-22, model/ffn.py:17-28): the layer RMSNorm's backward
// and SwiGLU's product, forward and backward.  Each is one pass over its
// operands in place of the 3 to 15 that the same formulas take as separate
// tensor operations, with the same roundings between the steps.

#include "nq_common.hpp"
#include "nq_internal.hpp"

namespace nq {

template <typename T>
__device__ __forceinline__ float as_stored(float v) {
  return (float)(T)v;
}

// 8 elements as they are stored
template <typename T> struct Raw8;
template <> struct Raw8<bf16> { typedef bf16x8 type; };
template <> struct Raw8<float> { typedef floatx8 type; };

// ---------------------------------------------------------------------------
// RMSNorm backward: y = n.to(x.dtype) * w, n = x r, r = rsqrt(mean(x^2) + eps).
//   g  = (dy w).to(x.dtype),  dx = r (g - n mean(g n)),
//   dw = sum over rows of dy n.to(x.dtype), in fp32.
// Bound by HBM: x and dy in, dx out.  One wave per row (lane l holds the
// 8-element chunks l, l + 64, ..., NC of them, so x and dy are read once and no
// barrier stands between rows); the next row's loads go out before this row's
// sums.  dw stays in registers over a wave's rows, the workgroup's four waves
// add theirs in LDS, in wave order, and the second kernel adds the workgroups'
// partials.  4096 x 2048 bf16, 50 MB: 15.3 + 4.6 us (3.3 TB/s without the second).
struct RmsBwdParams {
  const void* x;
  const void* dy;
  const void* w;
  int w16;  // the weight is bf16, else fp32
  void* dx;
  float* ws;  // (gridDim.x, width) partial sums of dw
  int64_t rows;
  int width;
  float eps;
};

template <typename TX, typename TDY, int NC>
__global__ __launch_bounds__(256) void rmsnorm_bwd_kernel(RmsBwdParams p) {
  __shared__ float red[NC * 512];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nch = p.width / 8;
  const int64_t step = (int64_t)gridDim.x * 4;
  floatx8 dw[NC];
  typename Raw8<TX>::type x[NC];
  typename Raw8<TDY>::type d[NC];
#pragma unroll
  for (int i = 0; i < NC; ++i) dw[i] = floatx8{};
  auto fetch = [&](int64_t row) {
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = lane + 64 * i;
      if (c < nch) {
        x[i] = *reinterpret_cast<const typename Raw8<TX>::type*>(reinterpret_cast<const TX*>(p.x) + row * p.width + c * 8);
        d[i] = *reinterpret_cast<const typename Raw8<TDY>::type*>(reinterpret_cast<const TDY*>(p.dy) + row * p.width + c * 8);
      }
    }
  };
  int64_t row = (int64_t)blockIdx.x * 4 + wave;
  if (row < p.rows) fetch(row);
  for (; row < p.rows; row += step) {
    floatx8 xv[NC], dv[NC], g[NC];
    float ss = 0.f, gx = 0.f;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = lane + 64 * i;
      xv[i] = dv[i] = g[i] = floatx8{};
      if (c < nch) {
        Weight8 wl;
        wl.load(p.w, p.w16, c * 8);
        const floatx8 w = wl.value(p.w16);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          xv[i][e] = (float)x[i][e];
          dv[i][e] = (float)d[i][e];
          g[i][e] = as_stored<TX>(dv[i][e] * w[e]);
          ss = __builtin_fmaf(xv[i][e], xv[i][e], ss);
          gx = __builtin_fmaf(g[i][e], xv[i][e], gx);
        }
      }
    }
    if (row + step < p.rows) fetch(row + step);
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) {
      ss += __shfl_xor(ss, m, 64);
      gx += __shfl_xor(gx, m, 64);
    }
    const float r = rsqrtf(ss / (float)p.width + p.eps);
    const float mean = gx * r / (float)p.width;
    TX* out = reinterpret_cast<TX*>(p.dx) + row * p.width;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = lane + 64 * i;
      if (c < nch) {
        floatx8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float n = xv[i][e] * r;
          o[e] = r * (g[i][e] - n * mean);
          dw[i][e] = __builtin_fmaf(dv[i][e], as_stored<TX>(n), dw[i][e]);
        }
        store8<TX>(out + c * 8, o);
      }
    }
  }
  for (int v = 0; v < 4; ++v) {
    if (wave == v) {
#pragma unroll
      for (int i = 0; i < NC; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          float* s = red + i * 512 + e * 64 + lane;
          *s = v ? *s + dw[i][e] : dw[i][e];
        }
    }
    __syncthreads();
  }
  for (int k = threadIdx.x; k < p.width; k += 256)
    p.ws[(int64_t)blockIdx.x * p.width + k] = red[(k >> 9) * 512 + (k & 7) * 64 + ((k >> 3) & 63)];
}

// dw[k] = sum of the nblk partials of column k, in a fixed order: workgroup of
// 32 columns x 32 row slots, each slot's loads independent, then over the slots.
template <typename TW>
__global__ __launch_bounds__(1024) void rmsnorm_dw_kernel(const float* ws, int nblk, int width, TW* dw) {
  __shared__ float part[32][33];
  const int c = threadIdx.x & 31, slot = threadIdx.x >> 5;
  const int k = blockIdx.x * 32 + c;
  float t = 0.f;
  if (k < width) {
#pragma unroll 8
    for (int i = slot; i < nblk; i += 32) t += ws[(int64_t)i * width + k];
  }
  part[slot][c] = t;
  __syncthreads();
  if (slot == 0 && k < width) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 32; ++i) s += part[i][c];
    dw[k] = (TW)s;
  }
}

// A workgroup per 4 rows up to two per CU: from there on more partials cost as
// much as the further waves in flight gain.
constexpr int RMS_BWD_BLOCKS = 512;
constexpr int RMS_BWD_WIDTH = 4096;  // 8 chunks a lane; beyond, a wave's rows leave the registers
static int rms_bwd_blocks(int64_t rows) {
  const int64_t b = (rows + 3) / 4;
  return (int)(b < RMS_BWD_BLOCKS ? b : RMS_BWD_BLOCKS);
}

template <typename TX, typename TDY>
static void launch_rms_bwd(const RmsBwdParams& p, int nblk, hipStream_t st) {
  const int nch = (p.width / 8 + 63) / 64;
  if (nch == 1) hipLaunchKernelGGL((rmsnorm_bwd_kernel<TX, TDY, 1>), dim3(nblk), dim3(256), 0, st, p);
  else if (nch == 2) hipLaunchKernelGGL((rmsnorm_bwd_kernel<TX, TDY, 2>), dim3(nblk), dim3(256), 0, st, p);
  else if (nch <= 4) hipLaunchKernelGGL((rmsnorm_bwd_kernel<TX, TDY, 4>), dim3(nblk), dim3(256), 0, st, p);
  else hipLaunchKernelGGL((rmsnorm_bwd_kernel<TX, TDY, 8>), dim3(nblk), dim3(256), 0, st, p);
}

// ---------------------------------------------------------------------------
// SwiGLU's product y = silu(gate) * up, silu rounded to T as a tensor of its
// own would be.  Bound by HBM; 8 elements (16 bytes of bf16) per thread.  25M bf16
// elements: 26 us forward, 151 MB, and 41 us backward, 252 MB (5.8 and 6.1 TB/s).
__device__ __forceinline__ float sigmoid(float v) { return 1.f / (1.f + expf(-v)); }

template <typename T>
__global__ __launch_bounds__(256) void swiglu_kernel(const T* gate, const T* up, T* y, int64_t n8) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n8) return;
  const floatx8 g = Vec8<T>::load_f32(gate + i * 8), u = Vec8<T>::load_f32(up + i * 8);
  floatx8 o;
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = as_stored<T>(g[e] / (1.f + expf(-g[e]))) * u[e];
  store8<T>(y + i * 8, o);
}

// d_up = dy silu(gate); d_gate = (dy up) s (1 + gate (1 - s)), s = sigmoid(gate),
// with silu(gate) and dy up rounded to T.
template <typename T>
__global__ __launch_bounds__(256) void swiglu_bwd_kernel(const T* gate, const T* up, const T* dy, T* dgate, T* dup,
                                                         int64_t n8) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n8) return;
  const floatx8 g = Vec8<T>::load_f32(gate + i * 8), u = Vec8<T>::load_f32(up + i * 8);
  const floatx8 d = Vec8<T>::load_f32(dy + i * 8);
  floatx8 dg, du;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float s = sigmoid(g[e]);
    du[e] = d[e] * as_stored<T>(g[e] / (1.f + expf(-g[e])));
    dg[e] = as_stored<T>(d[e] * u[e]) * s * (1.f + g[e] * (1.f - s));
  }
  store8<T>(dgate + i * 8, dg);
  store8<T>(dup + i * 8, du);
}

// ---------------------------------------------------------------------------
// A bool keep-mask as the additive bias the attention kernels read: 0 where the
// mask holds, -inf where not, in rows of T keys padded with zeros to a multiple of
// 8.  Bound by HBM; a thread writes 8 keys, which it reads as one word where the
// mask's keys are adjacent and 8-byte aligned.  As tensor operations (fill, not,
// masked fill, fill, copy) 22 us for (4, 1, 1024, 1024) in bf16, 5.6 so (2.3 TB/s).
struct MaskParams {
  const unsigned char* mask;
  int64_t sb, sh, ss, st;  // strides (bytes)
  void* bias;
  int H, S, T, nch;
  int64_t n;  // chunks of 8 keys
};

template <typename T>
__global__ __launch_bounds__(256) void mask_bias_kernel(MaskParams p) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= p.n) return;
  const int64_t row = i / p.nch;
  const int k0 = (int)(i - row * p.nch) * 8;
  const int64_t bh = row / p.S, b = bh / p.H;
  const unsigned char* m = p.mask + b * p.sb + (bh - b * p.H) * p.sh + (row - bh * p.S) * p.ss + k0 * p.st;
  floatx8 o;
  if (p.st == 1 && k0 + 8 <= p.T && (reinterpret_cast<uintptr_t>(m) & 7u) == 0) {
    const uint64_t w = *reinterpret_cast<const uint64_t*>(m);
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = (w >> (8 * e)) & 0xff ? 0.f : -INFINITY;
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = k0 + e >= p.T || m[e * p.st] ? 0.f : -INFINITY;
  }
  store8<T>(reinterpret_cast<T*>(p.bias) + i * 8, o);
}

}  // namespace nq

using namespace nq;

extern "C" int nq_mask_bias(const void* mask, const int64_t* mask_strides, void* bias, int B, int H, int S, int T,
                            int dtype, void* stream) {
  nq_clear_error();
  if (!nq_dtype_ok(dtype)) return nq_fail(NQ_ERR_UNSUPPORTED, "dtype must be NQ_DTYPE_BF16 or NQ_DTYPE_F32");
  if (B <= 0 || H <= 0 || S <= 0 || T <= 0)
    return nq_fail(NQ_ERR_INVALID, "sizes must be positive (B=%d H=%d S=%d T=%d)", B, H, S, T);
  if (!mask || !mask_strides || !bias) return nq_fail(NQ_ERR_INVALID, "mask, its strides and bias are required");
  if (!nq_aligned16(bias)) return nq_fail(NQ_ERR_INVALID, "the bias must be 16-byte aligned");
  const int nch = (int)(((int64_t)T + 7) / 8);
  MaskParams p{reinterpret_cast<const unsigned char*>(mask), mask_strides[0], mask_strides[1], mask_strides[2],
               mask_strides[3], bias, H, S, T, nch, (int64_t)B * H * S * nch};
  if ((p.n + 255) / 256 > INT32_MAX) return nq_fail(NQ_ERR_UNSUPPORTED, "too many elements for one launch");
  const dim3 grid((unsigned)((p.n + 255) / 256));
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (dtype == NQ_DTYPE_BF16) hipLaunchKernelGGL((mask_bias_kernel<bf16>), grid, dim3(256), 0, st, p);
  else hipLaunchKernelGGL((mask_bias_kernel<float>), grid, dim3(256), 0, st, p);
  return nq_check_launch(hipGetLastError());
}

extern "C" int64_t nq_rmsnorm_bwd_workspace_bytes(int64_t rows, int width) {
  if (rows <= 0 || width <= 0 || width % 8 || width > RMS_BWD_WIDTH) return 0;
  return (int64_t)rms_bwd_blocks(rows) * width * (int64_t)sizeof(float);
}

extern "C" int nq_rmsnorm_bwd(const void* x, const void* dy, const void* weight, void* dx, void* dweight,
                              void* workspace, int64_t workspace_bytes, int64_t rows, int width, int dtype_x,
                              int dtype_w, float eps, void* stream) {
  nq_clear_error();
  if (!nq_dtype_ok(dtype_x) || !nq_dtype_ok(dtype_w))
    return nq_fail(NQ_ERR_UNSUPPORTED, "dtype codes must be NQ_DTYPE_BF16 or NQ_DTYPE_F32");
  if (rows <= 0 || width <= 0 || width % 8 || width > RMS_BWD_WIDTH)
    return nq_fail(NQ_ERR_UNSUPPORTED, "rows must be positive and width a multiple of 8 up to %d, got %lld and %d",
                   RMS_BWD_WIDTH, (long long)rows, width);
  if (!x || !dy || !weight || !dx || !dweight || !workspace)
    return nq_fail(NQ_ERR_INVALID, "x, dy, weight, dx, dweight and workspace are required");
  if (!nq_aligned16(x) || !nq_aligned16(dy) || !nq_aligned16(weight) || !nq_aligned16(dx) || !nq_aligned16(workspace))
    return nq_fail(NQ_ERR_INVALID, "base pointers must be 16-byte aligned");
  if (workspace_bytes < nq_rmsnorm_bwd_workspace_bytes(rows, width))
    return nq_fail(NQ_ERR_WORKSPACE, "workspace too small: %lld bytes, need %lld", (long long)workspace_bytes,
                   (long long)nq_rmsnorm_bwd_workspace_bytes(rows, width));
  const bool w16 = dtype_w == NQ_DTYPE_BF16;
  RmsBwdParams p{x, dy, weight, w16, dx, reinterpret_cast<float*>(workspace), rows, width, eps};
  const int nblk = rms_bwd_blocks(rows);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  // dy has the promoted dtype of x and weight
  if (dtype_x == NQ_DTYPE_F32) launch_rms_bwd<float, float>(p, nblk, st);
  else if (w16) launch_rms_bwd<bf16, bf16>(p, nblk, st);
  else launch_rms_bwd<bf16, float>(p, nblk, st);
  const dim3 grid((unsigned)((width + 31) / 32));
  if (w16) hipLaunchKernelGGL((rmsnorm_dw_kernel<bf16>), grid, dim3(1024), 0, st, p.ws, nblk, width, (bf16*)dweight);
  else hipLaunchKernelGGL((rmsnorm_dw_kernel<float>), grid, dim3(1024), 0, st, p.ws, nblk, width, (float*)dweight);
  return nq_check_launch(hipGetLastError());
}

static int swiglu_check(int64_t n, int dtype, const void* a, const void* b, const void* c) {
  nq_clear_error();
  if (!nq_dtype_ok(dtype)) return nq_fail(NQ_ERR_UNSUPPORTED, "dtype must be NQ_DTYPE_BF16 or NQ_DTYPE_F32");
  if (n <= 0 || n % 8 || n / 8 > (int64_t)INT32_MAX * 256)
    return nq_fail(NQ_ERR_UNSUPPORTED, "n must be a positive multiple of 8, got %lld", (long long)n);
  if (!a || !b || !c) return nq_fail(NQ_ERR_INVALID, "every operand is required");
  if (!nq_aligned16(a) || !nq_aligned16(b) || !nq_aligned16(c))
    return nq_fail(NQ_ERR_INVALID, "base pointers must be 16-byte aligned");
  return NQ_OK;
}

extern "C" int nq_swiglu(const void* gate, const void* up, void* y, int64_t n, int dtype, void* stream) {
  if (int rc = swiglu_check(n, dtype, gate, up, y)) return rc;
  const dim3 grid((unsigned)((n / 8 + 255) / 256));
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (dtype == NQ_DTYPE_BF16)
    hipLaunchKernelGGL((swiglu_kernel<bf16>), grid, dim3(256), 0, st, (const bf16*)gate, (const bf16*)up, (bf16*)y, n / 8);
  else
    hipLaunchKernelGGL((swiglu_kernel<float>), grid, dim3(256), 0, st, (const float*)gate, (const float*)up, (float*)y, n / 8);
  return nq_check_launch(hipGetLastError());
}

extern "C" int nq_swiglu_bwd(const void* gate, const void* up, const void* dy, void* dgate, void* dup, int64_t n,
                             int dtype, void* stream) {
  if (int rc = swiglu_check(n, dtype, gate, up, dy)) return rc;
  if (int rc = swiglu_check(n, dtype, dgate, dup, dy)) return rc;
  const dim3 grid((unsigned)((n / 8 + 255) / 256));
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (dtype == NQ_DTYPE_BF16)
    hipLaunchKernelGGL((swiglu_bwd_kernel<bf16>), grid, dim3(256), 0, st, (const bf16*)gate, (const bf16*)up,
                       (const bf16*)dy, (bf16*)dgate, (bf16*)dup, n / 8);
  else
    hipLaunchKernelGGL((swiglu_bwd_kernel<float>), grid, dim3(256), 0, st, (const float*)gate, (const float*)up,
                       (const float*)dy, (float*)dgate, (float*)dup, n / 8);
  return nq_check_launch(hipGetLastError());
}
