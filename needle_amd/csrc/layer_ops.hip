// The decoder layer's elementwise work around the attention, for gfx950.
//
// Reference: needle/model/qwen2.py:52-65 (Qwen2DecoderLayer.forward: residual adds around
// the attention and the MLP, an RMSNorm before each), needle/layers/norm.py:14-17 (RMSNorm),
// needle/model/llama.py:36-37 (LlamaMLP: silu(gate) * up).
//
// The reference runs these as torch ops, one kernel each: the residual add, the RMSNorm's
// fp32 statistic, reciprocal square root, products and casts, the weight product, the SiLU
// and the product with up.  Here the residual add, the RMSNorm and its weight product are one
// kernel, and SiLU(gate) * up another, each keeping the reference's roundings:
//   h   = round(x + residual)                                  (qwen2.py:58, :63)
//   var = (sum_i float(h_i)^2) * (1 / hidden)                   (norm.py:15, torch's mean)
//   y   = round(float(h) * rsqrt(var + eps))                    (norm.py:16, cast to the dtype)
//   out = round(float(weight) * float(y))                       (norm.py:17)
//   act = round(round(silu(g)) * u), silu(g) = g / (1 + exp(-g)) (llama.py:37, torch's silu)
// round() is the model dtype's round-to-nearest-even (identity for float32).  Only the order
// of the sum of squares differs from torch's reduction, which can move the statistic by an
// ulp and an element of the output by an ulp of its format now and then.
//
// Both kernels are latency-bound at decode sizes (tens of rows) and
// HBM-bound at prefill sizes: every element is read and written once.
#include "ndl_common.hpp"

namespace ndl {
namespace {

constexpr int kThreads = 256;           // four waves
constexpr int kMaxHidden = 8192;        // four chunks of 8 elements per lane of four waves

// Eight consecutive elements of a row as fp32 (16 bytes of a 16-bit format, 32 of float32).
template <int FMT>
__device__ __forceinline__ void load8(const void* p, float (&v)[8]) {
  if constexpr (FMT == kFmtF32) {
    const u32x4 a = ld16(p), b = ld16(static_cast<const char*>(p) + 16);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[i] = __uint_as_float(a[i]);
      v[4 + i] = __uint_as_float(b[i]);
    }
  } else {
    using T = Elt<FMT == kFmtF16>;
    const u32x4 w = ld16(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = T::lo(w[i]);
      v[2 * i + 1] = T::hi(w[i]);
    }
  }
}

// v, already representable in the format, stored as eight elements.
template <int FMT>
__device__ __forceinline__ void store8(void* p, const float (&v)[8]) {
  if constexpr (FMT == kFmtF32) {
    st16(p, u32x4{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]),
                  __float_as_uint(v[3])});
    st16(static_cast<char*>(p) + 16, u32x4{__float_as_uint(v[4]), __float_as_uint(v[5]),
                                            __float_as_uint(v[6]), __float_as_uint(v[7])});
  } else {
    using T = Elt<FMT == kFmtF16>;
    st16(p, u32x4{T::pack(v[0], v[1]), T::pack(v[2], v[3]), T::pack(v[4], v[5]),
                  T::pack(v[6], v[7])});
  }
}

// x rounded to the format (round to nearest even), as fp32.
template <int FMT>
__device__ __forceinline__ float round_to(float x) {
  if constexpr (FMT == kFmtF32) {
    return x;
  } else {
    using T = Elt<FMT == kFmtF16>;
    return T::lo(T::pack(x, 0.f));
  }
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) v += xor_shfl(v, m);
  return v;
}

struct NormArgs {
  void* out;                // [rows][hidden]
  void* residual_out;       // [rows][hidden]: x + residual (may be residual itself)
  const void* x;            // [rows] rows of hidden elements, row stride x_stride
  const void* residual;     // [rows][hidden], or null
  const void* weight;       // [hidden]
  int64_t rows, x_stride;   // x_stride in elements
  int hidden;
  float eps, inv_hidden;
};

// Eight elements as loaded.
template <int FMT>
struct Raw8 {
  u32x4 v[FMT == kFmtF32 ? 2 : 1];
};
template <int FMT>
__device__ __forceinline__ Raw8<FMT> raw8(const void* p) {
  Raw8<FMT> r;
  r.v[0] = ld16(p);
  if constexpr (FMT == kFmtF32) r.v[1] = ld16(static_cast<const char*>(p) + 16);
  return r;
}
template <int FMT>
__device__ __forceinline__ void unpack8(const Raw8<FMT>& r, float (&v)[8]) {
  if constexpr (FMT == kFmtF32) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[i] = __uint_as_float(r.v[0][i]);
      v[4 + i] = __uint_as_float(r.v[1][i]);
    }
  } else {
    using T = Elt<FMT == kFmtF16>;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = T::lo(r.v[0][i]);
      v[2 * i + 1] = T::hi(r.v[0][i]);
    }
  }
}

// WPR waves per row; lane l of wave w holds chunks 64 w + l, + 64 WPR, .. (8 elements each) of
// the row, and the same chunks of the weight, in registers between the statistic and the
// products.  Every load goes out before any store (the compiler cannot move a load over the
// store of the residual sum, which may be the residual's own memory), and lanes past the row
// load its last chunk again instead of branching, so a row costs one memory round trip:
// interleaved with the stores it cost one per chunk.
template <int FMT, int NC, bool RES, int WPR>
__global__ __launch_bounds__(kThreads) void rms_norm_kernel(NormArgs a) {
  constexpr int EB = FMT == kFmtF32 ? 4 : 2;
  constexpr int RPG = kThreads / 64 / WPR;   // rows per workgroup
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int64_t row = (int64_t)blockIdx.x * RPG + wv / WPR;
  if (row >= a.rows) return;   // whole workgroups where waves share a row (RPG = 1)
  const int chunks = a.hidden / 8;
  const int ch0 = 64 * (wv % WPR) + lane;
  const char* x = static_cast<const char*>(a.x) + row * a.x_stride * EB;
  const int64_t row_off = row * a.hidden * EB;
  Raw8<FMT> xr[NC], rr[RES ? NC : 1], wr[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int ch = ch0 + 64 * WPR * c < chunks ? ch0 + 64 * WPR * c : chunks - 1;
    xr[c] = raw8<FMT>(x + ch * 8 * EB);
    if constexpr (RES) rr[c] = raw8<FMT>(static_cast<const char*>(a.residual) + row_off + ch * 8 * EB);
  }
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int ch = ch0 + 64 * WPR * c < chunks ? ch0 + 64 * WPR * c : chunks - 1;
    wr[c] = raw8<FMT>(static_cast<const char*>(a.weight) + ch * 8 * EB);
  }
  float h[NC][8];
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const bool live = ch0 + 64 * WPR * c < chunks;
    unpack8<FMT>(xr[c], h[c]);
    if constexpr (RES) {
      float r[8];
      unpack8<FMT>(rr[c], r);
#pragma unroll
      for (int e = 0; e < 8; ++e) h[c][e] = round_to<FMT>(__fadd_rn(h[c][e], r[e]));
    }
    if (live) {
#pragma unroll
      for (int e = 0; e < 8; ++e) ss = __fadd_rn(ss, __fmul_rn(h[c][e], h[c][e]));
    }
  }
  ss = wave_sum(ss);
  if constexpr (WPR > 1) {
    __shared__ float part[WPR];
    if (lane == 0) part[wv] = ss;
    __syncthreads();
    ss = part[0];
#pragma unroll
    for (int w = 1; w < WPR; ++w) ss = __fadd_rn(ss, part[w]);
  }
  const float var = __fmul_rn(ss, a.inv_hidden);
  const float rstd = rsqrtf(__fadd_rn(var, a.eps));
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int ch = ch0 + 64 * WPR * c;
    if (ch >= chunks) continue;
    if constexpr (RES)
      store8<FMT>(static_cast<char*>(a.residual_out) + row_off + ch * 8 * EB, h[c]);
    float w[8], o[8];
    unpack8<FMT>(wr[c], w);
#pragma unroll
    for (int e = 0; e < 8; ++e)
      o[e] = round_to<FMT>(__fmul_rn(w[e], round_to<FMT>(__fmul_rn(h[c][e], rstd))));
    store8<FMT>(static_cast<char*>(a.out) + row_off + ch * 8 * EB, o);
  }
}

struct SiluArgs {
  void* out;                          // [rows][inter]
  const void* gate;                   // row stride gate_stride (elements)
  const void* up;                     // row stride up_stride
  int64_t rows, gate_stride, up_stride;
  int inter;
};

// One thread per 8 elements of a row.
template <int FMT>
__global__ __launch_bounds__(kThreads) void silu_mul_kernel(SiluArgs a) {
  constexpr int EB = FMT == kFmtF32 ? 4 : 2;
  const int cpr = a.inter / 8;
  const int64_t idx = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  const int64_t row = idx / cpr;
  if (row >= a.rows) return;
  const int ch = (int)(idx - row * cpr);
  float g[8], u[8], o[8];
  load8<FMT>(static_cast<const char*>(a.gate) + (row * a.gate_stride + ch * 8) * EB, g);
  load8<FMT>(static_cast<const char*>(a.up) + (row * a.up_stride + ch * 8) * EB, u);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float s = round_to<FMT>(g[e] / __fadd_rn(1.f, expf(-g[e])));
    o[e] = round_to<FMT>(__fmul_rn(s, u[e]));
  }
  store8<FMT>(static_cast<char*>(a.out) + (row * a.inter + ch * 8) * EB, o);
}

// Four waves share a row where a wave alone would hold more than four chunks per lane, and up to
// kNormSharedRows rows (a decode step's).  us, residual form, bf16, out of cache, four waves /
// one wave per row / loads between the stores: 9 x 896 2.8 / 2.9 / 3.6, 300 x 896 3.2 / 3.4 /
// 4.2, 2,736 x 896 6.9 / 6.5 / 6.8, 16 x 3,584 3.3 / 4.6 / 7.0, 700 x 3,584 6.8 / 7.6 / 10.0,
// 4,096 x 4,096 26.0 (5.2 TB/s) / 30.0 / 30.5.
constexpr int64_t kNormSharedRows = 256;
constexpr int kNormSharedHidden = 4 * 64 * 8;   // past it, four chunks per lane of one wave

template <int FMT, bool RES, int WPR>
int launch_norm_wpr(const NormArgs& a, hipStream_t stream) {
  const int nc = (a.hidden / 8 + 64 * WPR - 1) / (64 * WPR);
  constexpr int RPG = kThreads / 64 / WPR;
  const dim3 grid((unsigned)((a.rows + RPG - 1) / RPG));
  if (nc <= 1)
    hipLaunchKernelGGL((rms_norm_kernel<FMT, 1, RES, WPR>), grid, dim3(kThreads), 0, stream, a);
  else if (nc <= 2)
    hipLaunchKernelGGL((rms_norm_kernel<FMT, 2, RES, WPR>), grid, dim3(kThreads), 0, stream, a);
  else
    hipLaunchKernelGGL((rms_norm_kernel<FMT, 4, RES, WPR>), grid, dim3(kThreads), 0, stream, a);
  return check_launch();
}

template <int FMT, bool RES>
int launch_norm(const NormArgs& a, hipStream_t stream) {
  static_assert(kMaxHidden <= 8 * 64 * 4 * 4, "four chunks per lane of four waves");
  return a.rows <= kNormSharedRows || a.hidden > kNormSharedHidden
             ? launch_norm_wpr<FMT, RES, 4>(a, stream)
             : launch_norm_wpr<FMT, RES, 1>(a, stream);
}

template <int FMT>
int launch_norm_fmt(const NormArgs& a, hipStream_t stream) {
  return a.residual != nullptr ? launch_norm<FMT, true>(a, stream)
                               : launch_norm<FMT, false>(a, stream);
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

}  // namespace
}  // namespace ndl

extern "C" int ndl_rms_norm(void* out, void* residual_out, const void* x, int64_t x_row_stride,
                            const void* residual, const void* weight, int64_t rows, int hidden,
                            float eps, int dtype, ndl_stream_t stream) {
  using namespace ndl;
  if (!dtype_known(dtype)) return NDL_ERR_UNSUPPORTED;
  if (rows < 0 || hidden <= 0) return NDL_ERR_INVALID_ARG;
  if (hidden % 8 != 0 || hidden > kMaxHidden) return NDL_ERR_UNSUPPORTED;
  if (rows == 0) return NDL_OK;
  if (!out || !x || !weight || (residual && !residual_out)) return NDL_ERR_INVALID_ARG;
  if (x_row_stride < hidden || x_row_stride % 8 != 0) return NDL_ERR_INVALID_ARG;
  if (!aligned16(out) || !aligned16(x) || !aligned16(weight) ||
      (residual && (!aligned16(residual) || !aligned16(residual_out))))
    return NDL_ERR_INVALID_ARG;
  if ((rows + 3) / 4 > 0x7fffffff) return NDL_ERR_UNSUPPORTED;
  NormArgs a;
  a.out = out;
  a.residual_out = residual ? residual_out : nullptr;
  a.x = x;
  a.residual = residual;
  a.weight = weight;
  a.rows = rows;
  a.x_stride = x_row_stride;
  a.hidden = hidden;
  a.eps = eps;
  a.inv_hidden = 1.f / (float)hidden;
  const hipStream_t s = (hipStream_t)stream;
  if (dtype_is_f32(dtype)) return launch_norm_fmt<kFmtF32>(a, s);
  if (dtype_is_f16(dtype)) return launch_norm_fmt<kFmtF16>(a, s);
  return launch_norm_fmt<kFmtBF16>(a, s);
}

extern "C" int ndl_silu_mul(void* out, const void* gate, int64_t gate_row_stride,
                            const void* up, int64_t up_row_stride, int64_t rows,
                            int intermediate, int dtype, ndl_stream_t stream) {
  using namespace ndl;
  if (!dtype_known(dtype)) return NDL_ERR_UNSUPPORTED;
  if (rows < 0 || intermediate <= 0) return NDL_ERR_INVALID_ARG;
  if (intermediate % 8 != 0) return NDL_ERR_UNSUPPORTED;
  if (rows == 0) return NDL_OK;
  if (!out || !gate || !up) return NDL_ERR_INVALID_ARG;
  if (gate_row_stride < intermediate || up_row_stride < intermediate ||
      gate_row_stride % 8 != 0 || up_row_stride % 8 != 0)
    return NDL_ERR_INVALID_ARG;
  if (!aligned16(out) || !aligned16(gate) || !aligned16(up)) return NDL_ERR_INVALID_ARG;
  const int64_t items = rows * (intermediate / 8);
  const int64_t blocks = (items + kThreads - 1) / kThreads;
  if (blocks > 0x7fffffff) return NDL_ERR_UNSUPPORTED;
  SiluArgs a;
  a.out = out;
  a.gate = gate;
  a.up = up;
  a.rows = rows;
  a.gate_stride = gate_row_stride;
  a.up_stride = up_row_stride;
  a.inter = intermediate;
  const hipStream_t s = (hipStream_t)stream;
  const dim3 grid((unsigned)blocks);
  if (dtype_is_f32(dtype))
    hipLaunchKernelGGL((silu_mul_kernel<kFmtF32>), grid, dim3(kThreads), 0, s, a);
  else if (dtype_is_f16(dtype))
    hipLaunchKernelGGL((silu_mul_kernel<kFmtF16>), grid, dim3(kThreads), 0, s, a);
  else
    hipLaunchKernelGGL((silu_mul_kernel<kFmtBF16>), grid, dim3(kThreads), 0, s, a);
  return check_launch();
}
