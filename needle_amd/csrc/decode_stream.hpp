// The stream split of the paged decode kernels and the merge of its partials, shared by the
// 16-bit kernel (paged_decode.hip) and the float32 one (paged_decode_f32.hip).
#pragma once

#include "ndl_common.hpp"

namespace ndl {

struct DecodeArgs {
  u16* out;
  const u16* q;
  int64_t q_tok_stride;
  const u16* kplane;
  const u16* vplane;
  int64_t num_blocks;
  int num_kv_heads;
  const int32_t* block_table;
  int64_t bt_row_stride;
  int max_blocks;
  // log2(block_size / 16): a block (table column) holds 1 << tile_shift tiles of 16 tokens;
  // tile t of a sequence is rows 16 (t mod 2^shift) .. + 16 of its column t >> shift.
  int tile_shift;
  const int32_t* context_lens;
  int num_heads;
  int group;
  float scale_log2;
  int num_seqs;
  // The stream split (a taker is a wave of the 16-bit kernels, a workgroup of the float32
  // one).
  int chunk;      // C: stream slots per taker; 0: ceil(T / waves) from the stream length T,
  int min_chunk;  // at least min_chunk
  int waves;      // takers per kv head
  int nseg;       // segment slots per kv head: takers per kv head + num_seqs
  float* ws_ml;   // [kv head][segment][group head][2] = (m, l)
  float* ws_acc;  // [kv head][segment][group head][D]
  // Fused append (null: none): the step's new k/v rows, [seq][kv head][D] with these token
  // strides, written into the cache and attended in the same pass.
  const u16* k_new;
  const u16* v_new;
  int64_t k_new_stride, v_new_stride;
  // Rotary embedding of the step (null: q and k_new are already rotated): cos/sin rows of
  // each sequence's new token, [seq][D] with row stride rope_stride.
  const u16* rope_cos;
  const u16* rope_sin;
  int64_t rope_stride;
};

__device__ __forceinline__ int64_t attended_len(const DecodeArgs& a, int seq) {
  int64_t L = (int64_t)a.context_lens[seq] + 1;  // attention.py:299
  // a table row holds at most W blocks of 16 << tile_shift tokens
  const int64_t cap = (int64_t)a.max_blocks << (4 + a.tile_shift);
  return L < cap ? L : cap;
}

__device__ __forceinline__ int seq_tiles(const DecodeArgs& a, int q) {
  const int64_t L = attended_len(a, q);
  return L <= 0 ? 0 : (int)((L + 15) >> 4);
}

// Stream slots of a sequence with n tiles: PAD empty slots, then its tiles (none for
// a sequence with nothing to attend).  The empty slots stand for what a wave spends on
// starting a sequence (its q rows, its table window and its first block load before any
// tile computes), so that the waves that cross a sequence boundary take fewer tiles and
// finish with the others.
template <int PAD>
__device__ __forceinline__ int stream_slots(int n) { return n > 0 ? n + PAD : 0; }

// Inclusive prefix sum over the 64 lanes of a wave.
__device__ __forceinline__ int wave_incl_scan(int v, int lane) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(v, d, 64);
    if (lane >= d) v += o;
  }
  return v;
}

// Stream position of sequence `target`'s first slot, or of the first sequence whose slots
// reach past stream slot `tile` (target < 0).  Sequences are scanned 64 at a time; the scan
// stops at the chunk that holds the answer.  Returns the sequence in *seq (num_seqs if none) and
// its first slot in *first.
template <int PAD>
__device__ __forceinline__ void stream_locate(const DecodeArgs& a, int lane, int target,
                                              int64_t tile, int* seq, int64_t* first) {
  int64_t carry = 0;
  for (int base = 0; base < a.num_seqs; base += 64) {
    const int q = base + lane;
    const int n = q < a.num_seqs ? seq_tiles(a, q) : 0;
    const int v = stream_slots<PAD>(n);
    const int incl = wave_incl_scan(v, lane);
    const int64_t excl = carry + incl - v;
    const uint64_t hit = target >= 0
        ? __builtin_amdgcn_ballot_w64(q == target)
        : __builtin_amdgcn_ballot_w64(q < a.num_seqs && n > 0 && excl + v > tile);
    if (hit) {
      const int l = __builtin_ctzll(hit);
      *seq = base + l;
      *first = __builtin_amdgcn_readlane((int)(excl - carry), l) + carry;
      return;
    }
    carry += __builtin_amdgcn_readlane(incl, 63);
  }
  *seq = a.num_seqs;
  *first = carry;
}

// Slots per taker: the fixed chunk, or the stream length (slots of all sequences of one
// kv head) over the takers of a kv head, at least min_chunk.
// The chunk for a stream of `total` slots.
__device__ __forceinline__ int64_t stream_chunk_of(const DecodeArgs& a, int64_t total) {
  if (a.chunk > 0) return a.chunk;
  const int64_t c = (total + a.waves - 1) / a.waves;
  return c < a.min_chunk ? a.min_chunk : c;
}
template <int PAD>
__device__ __forceinline__ int64_t stream_chunk(const DecodeArgs& a, int lane) {
  if (a.chunk > 0) return a.chunk;
  int64_t total = 0;
  for (int base = 0; base < a.num_seqs; base += 64) {
    const int q = base + lane;
    const int n = q < a.num_seqs ? seq_tiles(a, q) : 0;
    total += __builtin_amdgcn_readlane(wave_incl_scan(stream_slots<PAD>(n), lane), 63);
  }
  return stream_chunk_of(a, total);
}

// What one pass over the context lengths gives (longest: per lane, of the sequences it saw).
struct StreamSizes {
  int64_t slots;   // of the stream
  int seqs;        // sequences with something to attend
  int longest;     // tiles
};
__device__ __forceinline__ void add_sizes(StreamSizes& z, int n) {
  z.seqs += __builtin_popcountll(__builtin_amdgcn_ballot_w64(n > 0));
  z.longest = n > z.longest ? n : z.longest;
}

// Whether the float32 stream's workgroups take whole sequences instead of equal shares (its
// attention kernel and its merge both ask).  Equal shares end the wait for the longest sequence
// and cost a second start per workgroup, the partials and the merge; only the lengths tell, and
// only the device knows those (the table may be much wider).  Whole sequences where the longest
// has at most f32_short_tiles, or, while each (kv head, sequence) has a workgroup of its own, at
// most a third more than an equal share (and, at head_dim 64, f32_spare_tiles, what the second
// start and the merge take there).  us per launch pair, equal shares / whole / one launch per
// sequence (a 16-tile table): tables of 256 columns, 14/2 heads of 64, 8 sequences of 100 tokens
// 13.9 / 9.4 / 7.5, 400 14.1 / 12.6, 500 13.8 / 13.4; 28/4 of 128, 100 17.7 / 13.5 / 11.8, 300
// 18.4 / 18.1 / 16.1, 400 18.8 / 21.8.  Even batches: 32/8 heads, 32 of 1,000 60.9 / 58.7; 32/32,
// 8 of 1,000 58.9 / 57.2; 28/4, 48 of 1,000 53.9 / 47.3; uneven ones keep equal shares (32 of 104
// to 3,936, 28/4 heads, 44 / 104).
template <int D> constexpr int f32_short_tiles() { return D == 64 ? 28 : 18; }
template <int D> constexpr int f32_spare_tiles() { return D == 64 ? 24 : 0; }
// n: the lane's tiles of the first 64 sequences.  Asked before anything else is computed: short
// sequences are over in the time it takes.
template <int D>
__device__ __forceinline__ bool f32_all_short(const DecodeArgs& a, int n) {
  return a.num_seqs <= 64 && __builtin_amdgcn_ballot_w64(n > f32_short_tiles<D>()) == 0;
}
template <int D>
__device__ __forceinline__ bool f32_takes_whole(const DecodeArgs& a, const StreamSizes& z) {
  int64_t most = f32_short_tiles<D>();
  if (z.seqs <= a.waves) {
    const int64_t share = z.slots * 4 / (3 * (int64_t)a.waves) + f32_spare_tiles<D>();
    most = share > most ? share : most;
  }
  return __builtin_amdgcn_ballot_w64(z.longest > most) == 0;
}
// The sizes of a stream whose workgroups take equal shares, or nothing (false) where they take
// whole sequences.
template <int D, int PAD>
__device__ __forceinline__ bool f32_shares(const DecodeArgs& a, int lane, StreamSizes* z) {
  *z = StreamSizes{0, 0, 0};
  for (int base = 0; base < a.num_seqs; base += 64) {
    const int q = base + lane;
    const int n = q < a.num_seqs ? seq_tiles(a, q) : 0;
    if (base == 0 && f32_all_short<D>(a, n)) return false;
    z->slots += __builtin_amdgcn_readlane(wave_incl_scan(stream_slots<PAD>(n), lane), 63);
    add_sizes(*z, n);
  }
  return !f32_takes_whole<D>(a, *z);
}

// Merge of the segment partials: MW waves per (query head, sequence).  A sequence
// whose tiles lie with takers s0 .. s1 of its kv head's stream has its partials in
// segment slots s0 + seq .. s1 + seq; a sequence inside one taker was written by the
// attention kernel, and one with nothing to attend gets zeros here
// (attention.py:307-308 on an empty context).
// Pass 1 (thread-parallel over segments): global max, weights w_p = 2^(m_p - M)
// into LDS, denominator sum_p w_p l_p.  Pass 2: wave w adds w_p acc_p of the parts
// w, w + MW, ..; the first kMergePrefetch of them were loaded together with the (m, l) pairs,
// the rest with independent, unrolled loads; the waves' sums are added in wave order.
constexpr int kMergeMaxParts = 2048;
constexpr int kMergePrefetch = 8;

template <int D, int FMT, int MW, int PAD>
__global__ __launch_bounds__(64 * MW) void paged_decode_merge_kernel(DecodeArgs a) {
  constexpr int PER_LANE = D / 64;
  constexpr int EB = FMT == kFmtF32 ? 4 : 2;   // bytes per element
  __shared__ float wsh[kMergeMaxParts];
  const int head = blockIdx.x, seq = blockIdx.y, lane = threadIdx.x & 63;
  const int wv = MW == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int kvh = head / a.group, hc = head - kvh * a.group;
  // The decode step's new K/V row (ndl_paged_decode_append): the attention kernel attended
  // it from registers; the first query head's wave of each (kv head, sequence) stores it,
  // with the separate append's rule (attention.py:141-154): column min(ctx / bs, W - 1),
  // row ctx % bs, nothing for a negative context or an invalid block id.
  auto store_row = [&] {
    if (a.k_new == nullptr || hc != 0 || wv != 0) return;
    constexpr int EC = 16 / EB;  // elements per 16-byte chunk
    constexpr int CH = D / EC;   // 16-byte chunks per row; lanes < CH: K, < 2 CH: V
    static_assert(2 * CH <= 64, "a lane per chunk of the two rows");
    const int ctx = a.context_lens[seq];
    if (ctx >= 0 && lane < 2 * CH) {
      const int bshift = 4 + a.tile_shift;   // log2(block_size)
      const int pc = ctx >> bshift;
      const int col = pc < a.max_blocks - 1 ? pc : a.max_blocks - 1;
      const int64_t b = a.block_table[(int64_t)seq * a.bt_row_stride + col];
      if (b >= 0 && b < a.num_blocks) {
        const bool is_v = lane >= CH;
        const int ch = is_v ? lane - CH : lane;
        const char* src_row = (const char*)(is_v ? a.v_new : a.k_new) +
                              ((int64_t)seq * (is_v ? a.v_new_stride : a.k_new_stride) +
                               (int64_t)kvh * D) * EB;
        char* row = (char*)const_cast<u16*>(is_v ? a.vplane : a.kplane) +
                    (((b * a.num_kv_heads + kvh) << bshift) * D +
                     (int64_t)(ctx & ((1 << bshift) - 1)) * D) * EB + 16 * ch;
        u32x4 val = ld16(src_row + 16 * ch);
        if (!is_v && a.rope_cos != nullptr) {   // the key row rotated as the attention did
          constexpr int HC = CH / 2;
          const bool first_half = ch < HC;
          const int lo_c = first_half ? ch : ch - HC;
          const u32x4 partner = ld16(src_row + 16 * (ch ^ HC));
          const char* crow = (const char*)a.rope_cos + (int64_t)seq * a.rope_stride * EB + 16 * lo_c;
          const char* srow = (const char*)a.rope_sin + (int64_t)seq * a.rope_stride * EB + 16 * lo_c;
          u32x4 lo, hi;
          rope16<FMT>(first_half ? val : partner, first_half ? partner : val, ld16(crow),
                      ld16(crow + 16 * HC), ld16(srow), ld16(srow + 16 * HC), lo, hi);
          val = first_half ? lo : hi;
        }
        st16(row, val);
      }
    }
  };
  char* dst = (char*)a.out + (((int64_t)seq * a.num_heads + head) * D + lane * PER_LANE) * EB;
  auto store_out = [&](const float (&o)[PER_LANE]) {
    if constexpr (FMT == kFmtF32) {
      if constexpr (PER_LANE == 2)
        *reinterpret_cast<f32x2*>(dst) = f32x2{o[0], o[1]};
      else
        *reinterpret_cast<float*>(dst) = o[0];
    } else {
      using T = Elt<FMT == kFmtF16>;
      if constexpr (PER_LANE == 2)
        *reinterpret_cast<uint32_t*>(dst) = T::pack(o[0], o[1]);
      else
        *reinterpret_cast<u16*>(dst) = T::one(o[0]);
    }
  };
  float acc[PER_LANE];
#pragma unroll
  for (int e = 0; e < PER_LANE; ++e) acc[e] = 0.f;
  // One pass over context_lens (one load per 64 sequences): this sequence's tiles, its first
  // stream tile and the stream's sizes, i.e. what seq_tiles, stream_locate and stream_sizes give.
  int nt = 0;
  int64_t first = 0;
  StreamSizes z{0, 0, 0};
  auto scan = [&] {   // false: the sequences' workgroups wrote everything (float32)
    for (int base = 0; base < a.num_seqs; base += 64) {
      const int q = base + lane;
      const int n = q < a.num_seqs ? seq_tiles(a, q) : 0;
      if constexpr (FMT == kFmtF32) {
        if (base == 0 && f32_all_short<D>(a, n)) return false;
      }
      const int v = stream_slots<PAD>(n);
      const int incl = wave_incl_scan(v, lane);
      if (seq >= base && seq < base + 64) {   // the sequence's tile count and first tile
        nt = __builtin_amdgcn_readlane(n, seq - base);
        first = z.slots + __builtin_amdgcn_readlane(incl - v, seq - base) + PAD;
      }
      z.slots += __builtin_amdgcn_readlane(incl, 63);
      if constexpr (FMT == kFmtF32) add_sizes(z, n);
    }
    if constexpr (FMT == kFmtF32) return !f32_takes_whole<D>(a, z);
    return true;
  };
  if constexpr (FMT == kFmtF32) {
    if (!scan()) return;
    store_row();
  } else {
    store_row();
    scan();
  }
  if (nt == 0) {
    if (wv == 0) store_out(acc);
    return;
  }
  const int64_t chunk = stream_chunk_of(a, z.slots);
  const int64_t s0 = first / chunk, s1 = (first + nt - 1) / chunk;
  if (s0 == s1) return;
  const int nparts = (int)(s1 - s0 + 1);
  const int64_t slot0 = ((int64_t)kvh * a.nseg + s0 + seq) * a.group + hc;
  const int64_t ml_stride = 2 * (int64_t)a.group, acc_stride = (int64_t)a.group * D;
  const float* __restrict__ ml = a.ws_ml + slot0 * 2;
  const float* __restrict__ src = a.ws_acc + slot0 * D + lane * PER_LANE;

  // The first partials do not depend on the weights: load them with the (m, l) pairs.
  float pre[kMergePrefetch][PER_LANE];
#pragma unroll
  for (int u = 0; u < kMergePrefetch; ++u) {
    const int p = wv + MW * u;
#pragma unroll
    for (int e = 0; e < PER_LANE; ++e) pre[u][e] = p < nparts ? src[p * acc_stride + e] : 0.f;
  }

  // Part `tid`'s (m, l) pair (one 8-byte load) serves both passes below; parts from 64 MW on
  // (a sequence over more than 64 MW takers) are read again in the second.
  const int tid = threadIdx.x;
  float m0 = kNegInf, l0 = 0.f;
  if (tid < nparts) {
    const float2 v = *reinterpret_cast<const float2*>(ml + tid * ml_stride);
    m0 = v.x;
    l0 = v.y;
  }
  float mx = m0;
  for (int p = tid + 64 * MW; p < nparts; p += 64 * MW) mx = fmaxf(mx, ml[p * ml_stride]);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) mx = fmaxf(mx, xor_shfl(mx, o));
  __shared__ float sred[2][MW];
  if constexpr (MW > 1) {
    if (lane == 0) sred[0][wv] = mx;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < MW; ++w) mx = fmaxf(mx, sred[0][w]);
  }
  float den = 0.f;
  if (tid < nparts) {
    const float w = (m0 == kNegInf || mx == kNegInf) ? 0.f : fast_exp2(m0 - mx);
    wsh[tid] = w;
    den += w * l0;
  }
  for (int p = tid + 64 * MW; p < nparts; p += 64 * MW) {
    const float mp = ml[p * ml_stride];
    const float w = (mp == kNegInf || mx == kNegInf) ? 0.f : fast_exp2(mp - mx);
    wsh[p] = w;
    den += w * ml[p * ml_stride + 1];
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) den += xor_shfl(den, o);
  if constexpr (MW > 1) {
    if (lane == 0) sred[1][wv] = den;
  }
  __syncthreads();
  if constexpr (MW > 1) {
    den = 0.f;
#pragma unroll
    for (int w = 0; w < MW; ++w) den += sred[1][w];
  }

#pragma unroll
  for (int u = 0; u < kMergePrefetch; ++u)
    if (wv + MW * u < nparts)
#pragma unroll
      for (int e = 0; e < PER_LANE; ++e) acc[e] += wsh[wv + MW * u] * pre[u][e];
  constexpr int UN = MW == 1 ? 4 : 8;   // loads in flight past the prefetched parts
  int p = wv + MW * kMergePrefetch;
  for (; p + MW * (UN - 1) < nparts; p += MW * UN) {
    float v[UN][PER_LANE];
#pragma unroll
    for (int u = 0; u < UN; ++u)
#pragma unroll
      for (int e = 0; e < PER_LANE; ++e) v[u][e] = src[(p + MW * u) * acc_stride + e];
#pragma unroll
    for (int u = 0; u < UN; ++u)
#pragma unroll
      for (int e = 0; e < PER_LANE; ++e) acc[e] += wsh[p + MW * u] * v[u][e];
  }
  for (; p < nparts; p += MW)
#pragma unroll
    for (int e = 0; e < PER_LANE; ++e) acc[e] += wsh[p] * src[p * acc_stride + e];

  if constexpr (MW > 1) {
    __shared__ float ssum[MW][D];
#pragma unroll
    for (int e = 0; e < PER_LANE; ++e) ssum[wv][lane * PER_LANE + e] = acc[e];
    __syncthreads();
    if (wv != 0) return;
#pragma unroll
    for (int w = 1; w < MW; ++w)
#pragma unroll
      for (int e = 0; e < PER_LANE; ++e) acc[e] += ssum[w][lane * PER_LANE + e];
  }
  const float inv = den > 0.f ? 1.f / den : 0.f;
#pragma unroll
  for (int e = 0; e < PER_LANE; ++e) acc[e] *= inv;
  store_out(acc);
}

// Waves per (query head, sequence) of the merge: a sequence has about takers / sequences
// parts, which one wave reads a few at a time (latency-bound: 157 parts of a 20,011-token
// sequence, 32 heads, took 16.2 us, as long as the attention); from kMergeWideParts on eight
// waves share them (that step of 8 layers 283 -> 205 us).  At 4 parts per sequence (64
// sequences, 8 kv heads) the seven idle waves cost more than they save: 73.7 us with one
// wave, 80.2 with eight; a batch of 48 long sequences 308 and 313.
constexpr int kMergeWaves = 8;
constexpr int kMergeWideParts = 16;

template <int FMT, int PAD>
inline int launch_decode_merge(const DecodeArgs& a, int head_dim, hipStream_t s) {
  const dim3 grid((unsigned)a.num_heads, (unsigned)a.num_seqs);
  const bool wide = a.waves / a.num_seqs >= kMergeWideParts;
  if (head_dim == 128) {
    if (wide)
      hipLaunchKernelGGL((paged_decode_merge_kernel<128, FMT, kMergeWaves, PAD>), grid,
                         dim3(64 * kMergeWaves), 0, s, a);
    else
      hipLaunchKernelGGL((paged_decode_merge_kernel<128, FMT, 1, PAD>), grid, dim3(64), 0, s, a);
  } else {
    if (wide)
      hipLaunchKernelGGL((paged_decode_merge_kernel<64, FMT, kMergeWaves, PAD>), grid,
                         dim3(64 * kMergeWaves), 0, s, a);
    else
      hipLaunchKernelGGL((paged_decode_merge_kernel<64, FMT, 1, PAD>), grid, dim3(64), 0, s, a);
  }
  return check_launch();
}

}  // namespace ndl
