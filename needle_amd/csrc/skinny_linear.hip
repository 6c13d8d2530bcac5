// Linear layers on few rows (the projections of a decode step), for gfx950:
//   out[m][n] = round(sum_k x[m][k] * w[n][k] + bias[n]),  1 <= m <= 64,
// bf16 or fp16 operands, fp32 products and sums on the matrix cores, one rounding at the end
// (as torch's F.linear); and the SwiGLU form over a fused gate/up weight,
//   out[m][n] = round(round(silu(g)) * u),  g = round(x . w[n]),  u = round(x . w[inter + n]),
// with the roundings of the projection followed by ndl_silu_mul (llama.py:37).
//
// Reference: the projections of needle/layers/attention.py:84-96 and
// needle/model/llama.py:36-37, which are torch linears.
//
// Bound: the weights, each read once.  A library GEMM tiled for many rows leaves a decode
// step's weights at 0.5 to 4.9 TB/s; what limits a kernel that loads the matrix-core operand
// layout itself is the vector memory path (an instruction then reads 64 bytes of each of 16
// rows: 73 us at Qwen2-7B's gate/up projection, 9 rows, however many loads are in flight).
// So:
//   * Weights and activations go through LDS by direct loads of 8 whole 128-byte lines of 8
//     rows per instruction (1 KiB), with an XOR swizzle of the 16-byte chunks inside a row so
//     that the operand reads (16 rows at one chunk) are conflict-free.
//   * Every wave has a ring of its own in LDS and takes every NW-th 64-wide chunk of k
//     for all 16 RT weight rows of its workgroup: no barrier until the waves' sums are
//     combined (in wave order: deterministic), and a workgroup reads 128 NW contiguous bytes
//     of each row at a time.
//   * The loads are waited for by count (they complete in order), DEPTH chunks in flight
//     per wave; a chunk's slot is refilled as soon as its operands are in registers.
//   * Weights are read nontemporally: 10% at the large projections (51.2 -> 45.6 us at the
//     gate/up above, 5.3 -> 6.0 TB/s).
// Measured against torch's linear (a replayed graph, weights out of cache, 9 rows, us):
// Qwen2-0.5B qkv 5.4 -> 3.0, o 5.4 -> 2.9, gate/up 8.5 -> 5.5, down 17.1 -> 6.5, lm_head
// 57 -> 44.7; Qwen2-7B qkv 12.5 -> 8.5, o 12.0 -> 6.3, gate/up 59.5 -> 45.6, down 49.7 -> 26.8;
// at 48 rows 7.4 -> 4.3, 7.4 -> 4.3, 11.8 -> 7.4, 16.6 -> 11.9, 75 -> 69, 19.3 -> 12.6,
// 12.4 -> 10.5, 62.5 -> 60.1, 114 -> 44.3.  An empty kernel takes 1.9 us in such a graph.
#include "ndl_common.hpp"

namespace ndl {
namespace {

constexpr int kLinMaxRows = 64;
constexpr int kLinK = 64;           // k per chunk: one 128-byte line of a row

struct LinearArgs {
  u16* out;            // [m][cols], contiguous
  const u16* x;        // [m] rows of x_stride elements
  const u16* w;        // [n][k], contiguous
  const u16* bias;     // [n], or null
  int64_t x_stride;
  int m, k;
  int cols;            // columns of the output (SILU: w holds 2 * cols rows, gate then up)
};

// Waits until at most n (0 .. MAX) groups of I loads are in flight.
template <int I, int MAX>
__device__ __forceinline__ void vm_wait_groups(int n) {
  if constexpr (MAX == 0) {
    vm_wait<0>();
  } else {
    if (n >= MAX)
      vm_wait<MAX * I>();
    else
      vm_wait_groups<I, MAX - 1>(n);
  }
}

// MT: 16-row tiles of x; RT: 16-row tiles of w per workgroup (SILU: the first half gate rows,
// the second half the up rows of the same columns); NW waves split k.
template <bool F16, int MT, int RT, int NW, int DEPTH, bool SILU>
__global__ __launch_bounds__(64 * NW) void skinny_linear_kernel(LinearArgs a) {
  using T = Elt<F16>;
  using X8 = typename T::x8;
  constexpr int RO = SILU ? RT / 2 : RT;              // output tiles per workgroup
  constexpr int kTile = 16 * kLinK * 2;               // bytes of a staged 16-row tile
  constexpr int kStage = (RT + MT) * kTile;           // w tiles, then x tiles
  constexpr int I = 2 * (RT + MT);                    // loads per stage
  static_assert(DEPTH * I < 64, "vmcnt range");
  static_assert(DEPTH * kStage >= RT * MT * 1024, "a wave's sums fit its ring");
  constexpr int kRing = DEPTH * kStage;
  __shared__ __attribute__((aligned(16))) unsigned char smem[NW * kRing];
  const int lane = threadIdx.x & 63, j = lane >> 4, c = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * 16 * RO;
  unsigned char* const ring = smem + wv * kRing;
  const uint32_t ring_lds = lds_addr(ring);

  // A load covers 8 rows of a tile: lane L lands in slot L % 8 of row L / 8 and reads chunk
  // (L % 8) ^ (L / 8) of that row.
  const int lr = lane >> 3, lc = (lane & 7) ^ lr;
  const uint32_t w_off = (uint32_t)(lr * a.k * 2 + lc * 16);
  const char* wb[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    // tiles past the last one (cols is a multiple of 16) read the last again
    int row = n0 + 16 * (t % RO);
    if (row > a.cols - 16) row = a.cols - 16;
    if (t >= RO) row += a.cols;
    wb[t] = (const char*)(a.w + (int64_t)row * a.k);
  }
  const int64_t w8 = (int64_t)8 * a.k * 2;
  uint32_t x_off[2 * MT];
#pragma unroll
  for (int e = 0; e < 2 * MT; ++e) {
    // rows past the last one read it again; their sums are not stored
    const int m = 8 * e + lr < a.m ? 8 * e + lr : a.m - 1;
    x_off[e] = (uint32_t)(m * a.x_stride * 2 + lc * 16);
  }
  const int chunks = a.k / kLinK;
  const int cnt = wv < chunks ? (chunks - wv + NW - 1) / NW : 0;   // wv, wv + NW, ..
  auto issue = [&](int i, int slot) {
    const int64_t kb = (int64_t)(wv + i * NW) * (kLinK * 2);
    const uint32_t l = ring_lds + slot * kStage;
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      lds_dma16_nt(wb[t] + kb, w_off, l + t * kTile);
      lds_dma16_nt(wb[t] + w8 + kb, w_off, l + t * kTile + 1024);
    }
#pragma unroll
    for (int e = 0; e < 2 * MT; ++e)
      lds_dma16((const char*)a.x + kb, x_off[e], l + RT * kTile + e * 1024);
  };
  f32x4 acc[RT][MT];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[t][i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int d = 0; d < DEPTH; ++d)
    if (d < cnt) issue(d, d);
  // Operand of k-step s (32 k): lane (j, c) reads chunk 4 s + j of row c.
  const int foff[2] = {c * 128 + ((j ^ (c & 7)) << 4), c * 128 + (((j + 4) ^ (c & 7)) << 4)};
  int slot = 0;
  for (int i = 0; i < cnt; ++i) {
    const int later = cnt - 1 - i < DEPTH - 1 ? cnt - 1 - i : DEPTH - 1;   // issued after i
    vm_wait_groups<I, DEPTH - 1>(later);
    asm volatile("" ::: "memory");   // no LDS read above the wait
    const unsigned char* st = ring + slot * kStage;
    u32x4 wf[2][RT], xf[2][MT];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int t = 0; t < RT; ++t)
        wf[s][t] = *reinterpret_cast<const u32x4*>(st + t * kTile + foff[s]);
#pragma unroll
      for (int q = 0; q < MT; ++q)
        xf[s][q] = *reinterpret_cast<const u32x4*>(st + (RT + q) * kTile + foff[s]);
    }
    if (i + DEPTH < cnt) {
      // the slot's operands are in registers before its next loads go out
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      issue(i + DEPTH, slot);
    }
    slot = slot + 1 == DEPTH ? 0 : slot + 1;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int q = 0; q < MT; ++q)
          acc[t][q] = T::mfma16x16x32(__builtin_bit_cast(X8, wf[s][t]),
                                      __builtin_bit_cast(X8, xf[s][q]), acc[t][q]);
  }
  // Each wave's sums into its own ring (its loads have landed and its reads are done), one
  // barrier, then wave w finishes tiles w, w + NW, ...  Lane (j, c) of tile (t, q) holds
  // out[16 q + c][n0 + 16 t + 4 j ..].
  auto sums = [&](int w, int p) {
    return reinterpret_cast<f32x4*>(smem + w * kRing + p * 1024) + lane;
  };
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int q = 0; q < MT; ++q) *sums(wv, t * MT + q) = acc[t][q];
  __syncthreads();
  auto total = [&](int p) {
    f32x4 v = *sums(0, p);
#pragma unroll
    for (int w = 1; w < NW; ++w) v += *sums(w, p);
    return v;
  };
  for (int p = wv; p < RO * MT; p += NW) {
    const int t = p / MT, q = p - t * MT;
    const int n = n0 + 16 * t + 4 * j, m = 16 * q + c;
    const f32x4 v = total(p);
    float o[4];
    if constexpr (SILU) {
      const f32x4 up = total(p + RO * MT);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float g = T::lo(T::one(v[e])), u = T::lo(T::one(up[e]));
        const float s = T::lo(T::one(g / __fadd_rn(1.f, expf(-g))));
        o[e] = __fmul_rn(s, u);
      }
    }
    if (m >= a.m || n >= a.cols) continue;
    if constexpr (!SILU) {
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = v[e];
      if (a.bias != nullptr) {
        const u32x2 b = ld8(a.bias + n);
        o[0] += T::lo(b[0]);
        o[1] += T::hi(b[0]);
        o[2] += T::lo(b[1]);
        o[3] += T::hi(b[1]);
      }
    }
    *reinterpret_cast<u32x2*>(a.out + (int64_t)m * a.cols + n) =
        u32x2{T::pack(o[0], o[1]), T::pack(o[2], o[3])};
  }
}

template <bool F16, int MT, int RT, int NW, int DEPTH, bool SILU>
int launch_linear(const LinearArgs& a, hipStream_t s) {
  constexpr int RO = SILU ? RT / 2 : RT;
  hipLaunchKernelGGL((skinny_linear_kernel<F16, MT, RT, NW, DEPTH, SILU>),
                     dim3((unsigned)((a.cols + 16 * RO - 1) / (16 * RO))), dim3(64 * NW), 0, s, a);
  return check_launch();
}

// Weight tiles per workgroup: the fewest (1, 2 or 4) for which every workgroup has a CU of
// its own; where no choice does (more than 1024 tiles) 2, and 4 from 33 rows on, where the
// activations each workgroup reads outweigh its weights.  Measured, us at RT = 1 / 2 / 4:
// 224 tiles (Qwen2-7B o, 9 rows) 6.3 / 9.2 / 12.4; 288 (its qkv) 8.9 / 8.5 / 12.7; 608
// (Qwen2-0.5B gate/up) - / 5.7 / 5.4; 2368 (7B gate/up) - / 45.6 / 49.3, at 48 rows
// - / 62.9 / 60.1.  A workgroup of one tile takes eight waves when k is long enough to keep
// them busy (Qwen2-7B down, k 18,944, 16 rows: 31.2 us with four, 28.6 with eight; k 3,584:
// 7.0 and 7.1).
constexpr int kLinCUs = 256;
constexpr int kLinLongK = 8192;

template <bool F16, int MT, bool SILU>
int pick_linear(const LinearArgs& a, hipStream_t s) {
  const int tiles = (a.cols / 16) * (SILU ? 2 : 1);
  constexpr int kDeep = MT == 1 || MT == 4 ? 3 : 2;
  if constexpr (!SILU) {
    if (tiles <= kLinCUs) {
      if (a.k >= kLinLongK)
        return launch_linear<F16, MT, 1, 8, MT == 1 ? 4 : MT == 2 ? 3 : 2, false>(a, s);
      return launch_linear<F16, MT, 1, 4, MT == 1 ? 4 : 3, false>(a, s);
    }
  }
  const bool two = tiles <= 2 * kLinCUs || (tiles > 4 * kLinCUs && MT <= 2);
  if (two) return launch_linear<F16, MT, 2, 4, kDeep, SILU>(a, s);
  return launch_linear<F16, MT, 4, 4, 2, SILU>(a, s);
}

template <bool F16, bool SILU>
int pick_linear_rows(const LinearArgs& a, hipStream_t s) {
  if (a.m <= 16) return pick_linear<F16, 1, SILU>(a, s);
  if (a.m <= 32) return pick_linear<F16, 2, SILU>(a, s);
  if (a.m <= 48) return pick_linear<F16, 3, SILU>(a, s);
  return pick_linear<F16, 4, SILU>(a, s);
}

template <bool SILU>
int skinny_linear(void* out, const void* x, int64_t x_row_stride, const void* w,
                  const void* bias, int rows, int cols, int k, int dtype, hipStream_t stream) {
  if (!dtype_supported(dtype)) return NDL_ERR_UNSUPPORTED;
  if (rows < 0 || cols <= 0 || k <= 0) return NDL_ERR_INVALID_ARG;
  // Offsets inside a row group are 32-bit in the kernel: 8 rows of w, 64 rows of x.
  if (rows > kLinMaxRows || cols % 16 != 0 || cols > (1 << 28) || k % kLinK != 0 ||
      k > (1 << 24) || x_row_stride > (1 << 24))
    return NDL_ERR_UNSUPPORTED;
  if (rows == 0) return NDL_OK;
  if (!out || !x || !w || x_row_stride < k || x_row_stride % 8 != 0) return NDL_ERR_INVALID_ARG;
  if (((uintptr_t)out | (uintptr_t)x | (uintptr_t)w | (uintptr_t)bias) & 15u)
    return NDL_ERR_INVALID_ARG;
  LinearArgs a;
  a.out = (u16*)out;
  a.x = (const u16*)x;
  a.w = (const u16*)w;
  a.bias = (const u16*)bias;
  a.x_stride = x_row_stride;
  a.m = rows;
  a.k = k;
  a.cols = cols;
  return dtype_is_f16(dtype) ? pick_linear_rows<true, SILU>(a, stream)
                             : pick_linear_rows<false, SILU>(a, stream);
}

}  // namespace
}  // namespace ndl

extern "C" int ndl_skinny_linear(void* out, const void* x, int64_t x_row_stride,
                                 const void* weight, const void* bias, int rows, int cols, int k,
                                 int dtype, ndl_stream_t stream) {
  return ndl::skinny_linear<false>(out, x, x_row_stride, weight, bias, rows, cols, k, dtype,
                                   (hipStream_t)stream);
}

extern "C" int ndl_skinny_linear_silu(void* out, const void* x, int64_t x_row_stride,
                                      const void* weight, int rows, int intermediate, int k,
                                      int dtype, ndl_stream_t stream) {
  return ndl::skinny_linear<true>(out, x, x_row_stride, weight, nullptr, rows, intermediate, k,
                                  dtype, (hipStream_t)stream);
}
