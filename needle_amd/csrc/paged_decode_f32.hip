// Paged decode attention in float32 (the reference's --dtype float32), gfx950.
//
// Reference: needle/layers/attention.py:291-310 (_decode_pytorch) in a float32 model
// (needle/args.py:80-84, :143-153; runner.py:31-34, 75-78): per sequence gather K/V blocks,
// expand the GQA group, softmax(q K^T * scale) V, every op in fp32.
//
// A workgroup of kF32Waves waves takes a run of 16-token tiles of a (kv head, sequence), wave
// w its tiles w, w + kF32Waves, ..; the waves combine their (m, l, acc) through LDS, as the
// 16-bit per-sequence split does.  What a sequence costs is the fp32 matrix rate (16 query
// heads' worth of products per tile whatever the group is, 2,048 cycles of a SIMD at head_dim
// 128), so one workgroup per (kv head, sequence) leaves a serving batch waiting for its
// longest sequence on a fraction of the GPU: 12 sequences of up to 4,000 tokens, 4 kv heads,
// 87 us per layer at 0.56 TB/s.  With a workspace the tiles of all sequences are one stream
// (decode_stream.hpp) shared by as many workgroups as can be resident, each taking the
// same number of tiles, and a merge adds the partials: 26.1 us, 1.87 TB/s; what is left is the
// start of each workgroup and the merge (14 us for a single tile per wave).  Where the lengths are short or even the workgroups
// take whole sequences after all (f32_takes_whole).  The products run on v_mfma_f32_16x16x4_f32
// (fp32 operands, fp32 accumulation), the probabilities stay fp32:
//   * S^T = K q^T: M = the tile's 16 tokens, N = the g query heads (padded to 16),
//     K = head_dim in steps of 4.  Lane (i, kk) = (lane % 16, lane / 16) holds
//     K[token i][16 m + 4 kk + e] and q[head i][16 m + 4 kk + e] for m < D/16, e < 4 (one
//     16-byte load per m: 64 contiguous bytes of a row per four lanes); the k order inside
//     the contraction is immaterial as long as both operands use it.
//   * The S^T accumulator puts tokens 4 kk + r of head i in lane (i, kk), which is the B
//     operand (P^T) of O^T = V^T P^T with token 4 kk + t in k-step t: no lane exchange.  The
//     matching A operand is V[4 kk + t][64 g + 4 i + e] (a 16-byte load per (g, t): 256
//     contiguous bytes of a row per sixteen lanes), so O^T row i of group g, MFMA e is head
//     dim d = 64 g + 4 i + e, and lane (i, kk) ends with O[head i][64 g + 16 kk + 4 r + e].
//   * Online softmax in the exp2 domain (scale * log2 e folded), the row max and sum across
//     the four lanes of a head by two lane swaps; the accumulator is rescaled when a head's
//     max moves.
// The fused forms attend the step's row from registers (the new key rotated there) and store it
// in the same call, as the 16-bit kernel does; q is rotated as it is loaded.
#include "decode_stream.hpp"

#include <type_traits>

namespace ndl {

constexpr int kF32Waves = 8;
// Empty stream slots before each sequence (what starting one costs a workgroup: its q rows,
// its table window, its first tile and one more combine, about a round and a half of its
// eight waves), and the fewest slots a workgroup takes (one tile per wave).  12 sequences of
// 100 to 4,000 tokens, 28 / 4 heads of 128, us per layer: 26.5 at 12 empty slots, 27.1 at 8,
// 31 at 4 (at least 8 slots each; 16 the same, 24 31, 32 36).
constexpr int kF32StreamPad = 12;
constexpr int kF32MinChunk = 8;

__device__ __forceinline__ f32x4 ldf4(const float* p) {
  return *reinterpret_cast<const f32x4*>(p);
}

// The launch's arguments, read again where they are used: what a rare path needs (the step's
// row, the output) then holds no scalar registers through the walk.
typedef const __attribute__((address_space(4))) DecodeArgs DecodeArgsConst;
__device__ __forceinline__ DecodeArgsConst& fresh_args() {
  DecodeArgsConst* p = (DecodeArgsConst*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *p;
}

// SPLIT: workgroup sw of a kv head takes stream slots sw*C .. sw*C + C, whatever sequences
// they belong to, or the whole sequences sw, sw + takers, .. where the lengths make that the
// faster one (f32_takes_whole); otherwise one workgroup per (kv head, sequence).  APP: the
// step's row (a.k_new, a.v_new) is attended in place of the pool's stale one; where a workgroup
// has the whole sequence the wave that attends the row also stores it, else the merge kernel
// does.
template <int D, bool ROPE, bool APP, bool SPLIT>
__global__ __launch_bounds__(64 * kF32Waves) void paged_decode_f32_kernel(DecodeArgs a) {
  constexpr int NW = kF32Waves;
  constexpr int QK = D / 16;   // 16-byte pieces of a K row (and of q) per lane
  constexpr int G = D / 64;    // 64-wide head_dim groups of the PV product
  constexpr int E = D / 4;     // accumulator floats per lane
  constexpr int KPW = E / NW;  // accumulator floats per lane each wave finishes
  static_assert(D == 64 || D == 128, "head_dim");
  const int kvh = (int)(blockIdx.x % (unsigned)a.num_kv_heads);
  const int sw = (int)(blockIdx.x / (unsigned)a.num_kv_heads);   // stream taker or sequence
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int i16 = lane & 15, kk = lane >> 4;
  const bool head_ok = i16 < a.group;
  const int head = kvh * a.group + i16;
  const int tshift = a.tile_shift, tmask = (1 << tshift) - 1;
  const int64_t blk_stride = (int64_t)a.num_kv_heads * (16 << tshift) * D;
  const int64_t head_off = (int64_t)kvh * (16 << tshift) * D;
  const float* const kplane = (const float*)a.kplane;
  const float* const vplane = (const float*)a.vplane;
  __shared__ __attribute__((aligned(16))) float sacc[NW * E * 64];
  __shared__ float sm[NW * 16], sl[NW * 16];
  // The split form has no registers to spare: with its arguments held it spilled to memory at
  // head_dim 128 (32 of 1,000 tokens as whole sequences, 28/4 heads: 45.7 us, read again 41.2).
  auto args = [&]() -> decltype(auto) {
    if constexpr (SPLIT)
      return fresh_args();
    else
      return (a);
  };
  bool smem_busy = false;   // an earlier piece's combine may still be reading LDS

  // Tiles lt0 .. lt1 of sequence seq (n_tiles in all), the waves taking every NW-th; every
  // wave of the workgroup calls it together (it has barriers).  whole_seq: std::true_type where
  // these are all its tiles.
  auto piece = [&](auto whole_seq, const int seq, const int lt0, const int lt1, const int n_tiles,
                   const int segid) {
    constexpr bool WHOLE = decltype(whole_seq)::value;
    const int64_t L = attended_len(a, seq);
    const int first = lt0 + wv;
    const int ntw = first < lt1 ? (lt1 - first + NW - 1) / NW : 0;   // this wave's tiles

    // The appended row's tile (attention.py:144-146): row ctx % bs of table column
    // min(ctx / bs, W - 1); ctx >= 0 where a sequence has tiles.
    int app_tile = -1, r_new = 0;
    if constexpr (APP) {
      const int p = a.context_lens[seq];
      const int pc = p >> (4 + tshift);
      if (p >= 0)
        app_tile = ((pc < a.max_blocks - 1 ? pc : a.max_blocks - 1) << tshift) | ((p >> 4) & tmask);
      r_new = p & 15;
    }

    // q^T operand (lanes past the group read the group's first head and zero it)
    f32x4 qv[QK];
    {
      auto&& r = args();
      const float* qrow = (const float*)r.q + (int64_t)seq * r.q_tok_stride +
                          (int64_t)(head_ok ? head : kvh * a.group) * D + 4 * kk;
#pragma unroll
      for (int m = 0; m < QK; ++m) qv[m] = ldf4(qrow + 16 * m);
      if constexpr (ROPE) {
        // element 16 m + 4 kk + e pairs with the same lane's piece m + QK / 2
        const float* crow = (const float*)r.rope_cos + (int64_t)seq * r.rope_stride + 4 * kk;
        const float* srow = (const float*)r.rope_sin + (int64_t)seq * r.rope_stride + 4 * kk;
#pragma unroll
        for (int m = 0; m < QK / 2; ++m) {
          u32x4 lo, hi;
          rope4_f32(__builtin_bit_cast(u32x4, qv[m]), __builtin_bit_cast(u32x4, qv[m + QK / 2]),
                    __builtin_bit_cast(u32x4, ldf4(crow + 16 * m)),
                    __builtin_bit_cast(u32x4, ldf4(crow + 16 * (m + QK / 2))),
                    __builtin_bit_cast(u32x4, ldf4(srow + 16 * m)),
                    __builtin_bit_cast(u32x4, ldf4(srow + 16 * (m + QK / 2))), lo, hi);
          qv[m] = __builtin_bit_cast(f32x4, lo);
          qv[m + QK / 2] = __builtin_bit_cast(f32x4, hi);
        }
      }
#pragma unroll
      for (int m = 0; m < QK; ++m) qv[m] = head_ok ? qv[m] : f32x4{0.f, 0.f, 0.f, 0.f};
    }

    struct Tile {
      f32x4 k[QK];
      f32x4 v[G][4];
      bool bad;
      int64_t off;   // the tile's first element in a plane
    };
    f32x4 acc[G][4];
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[g][e] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = kNegInf, l_run = 0.f;
    const int32_t* bt_row = a.block_table + (int64_t)seq * a.bt_row_stride;

    // The wave's tiles go in windows of 64 (lane l: the block id of the window's tile l).
    for (int w0 = 0; w0 < ntw; w0 += 64) {
      const int cnt = ntw - w0 < 64 ? ntw - w0 : 64;
      const int tl = first + NW * (w0 + (lane < cnt ? lane : cnt - 1));   // the lane's tile
      const int bt_lane = bt_row[tl >> tshift];
      asm volatile("" ::"v"(bt_lane));   // the ids are waited for once per window

      // live = false: a placeholder of the same instructions (every lane reads the tile's
      // first 16 bytes), issued past the window's end so that every compute has the same
      // loads in flight behind it.
      auto load_tile = [&](int it, Tile& t, bool live) {
        const int itc = it < cnt ? it : cnt - 1;
        int64_t blk = __builtin_amdgcn_readlane(bt_lane, itc);
        t.bad = blk < 0 || blk >= a.num_blocks;
        if (t.bad) blk = 0;
        const int tix = first + NW * (w0 + itc);
        t.off = blk * blk_stride + head_off + (int64_t)(tix & tmask) * 16 * D;
        const float* kb = kplane + t.off + (live ? (int64_t)i16 * D + 4 * kk : 0);
        const float* vb = vplane + t.off + (live ? (int64_t)4 * kk * D + 4 * i16 : 0);
#pragma unroll
        for (int m = 0; m < QK; ++m) t.k[m] = ldf4(kb + (live ? 16 * m : 0));
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
          for (int t4 = 0; t4 < 4; ++t4) t.v[g][t4] = ldf4(vb + (live ? t4 * D + 64 * g : 0));
      };
      // The step's row in place of row r_new of its tile (loaded where it is used: one tile
      // of one wave per sequence, and its registers are not held through the walk).
      auto put_new_row = [&](Tile& t) {
        auto&& r = args();
        const float* krow = (const float*)r.k_new + (int64_t)seq * r.k_new_stride +
                            (int64_t)kvh * D + 4 * kk;
        const float* vrow = (const float*)r.v_new + (int64_t)seq * r.v_new_stride +
                            (int64_t)kvh * D + 4 * i16;
        f32x4 kn[QK];
#pragma unroll
        for (int m = 0; m < QK; ++m) kn[m] = ldf4(krow + 16 * m);
        if constexpr (ROPE) {
          const float* crow = (const float*)r.rope_cos + (int64_t)seq * r.rope_stride + 4 * kk;
          const float* srow = (const float*)r.rope_sin + (int64_t)seq * r.rope_stride + 4 * kk;
#pragma unroll
          for (int m = 0; m < QK / 2; ++m) {
            u32x4 lo, hi;
            rope4_f32(__builtin_bit_cast(u32x4, kn[m]), __builtin_bit_cast(u32x4, kn[m + QK / 2]),
                      __builtin_bit_cast(u32x4, ldf4(crow + 16 * m)),
                      __builtin_bit_cast(u32x4, ldf4(crow + 16 * (m + QK / 2))),
                      __builtin_bit_cast(u32x4, ldf4(srow + 16 * m)),
                      __builtin_bit_cast(u32x4, ldf4(srow + 16 * (m + QK / 2))), lo, hi);
            kn[m] = __builtin_bit_cast(f32x4, lo);
            kn[m + QK / 2] = __builtin_bit_cast(f32x4, hi);
          }
        }
        if (i16 == r_new) {
#pragma unroll
          for (int m = 0; m < QK; ++m) t.k[m] = kn[m];
          if constexpr (WHOLE) {
            float* const kd = (float*)r.kplane + t.off + (int64_t)r_new * D + 4 * kk;
#pragma unroll
            for (int m = 0; m < QK; ++m) *reinterpret_cast<f32x4*>(kd + 16 * m) = kn[m];
          }
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const f32x4 vn = ldf4(vrow + 64 * g);
#pragma unroll
          for (int t4 = 0; t4 < 4; ++t4)
            if (4 * kk + t4 == r_new) t.v[g][t4] = vn;
          if constexpr (WHOLE) {
            if (kk == r_new >> 2)
              *reinterpret_cast<f32x4*>((float*)r.vplane + t.off + (int64_t)r_new * D +
                                        4 * i16 + 64 * g) = vn;
          }
        }
      };
      auto compute = [&](int it, Tile& t) {
        const int tix = first + NW * (w0 + it);
        if (APP && tix == app_tile && !t.bad) put_new_row(t);
        f32x4 st = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m = 0; m < QK; ++m)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            st = __builtin_amdgcn_mfma_f32_16x16x4f32(t.k[m][e], qv[m][e], st, 0, 0, 0);
        // st[r]: token tix * 16 + 4 kk + r, head i16
        const int64_t pos0 = (int64_t)tix * 16 + 4 * kk;
        float sc[4];
        float mt = kNegInf;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const bool ok = !t.bad && pos0 + r < L;
          sc[r] = ok ? st[r] * a.scale_log2 : kNegInf;
          mt = fmaxf(mt, sc[r]);
          // rows past the range may hold any bits (NaN * 0 = NaN): cleared
          if (!ok) {
#pragma unroll
            for (int g = 0; g < G; ++g) t.v[g][r] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
        }
        mt = max_xor32(max_xor16(mt));
        const float m_new = fmaxf(m_run, mt);
        const float m_use = m_new == kNegInf ? 0.f : m_new;
        const float alpha = fast_exp2(m_run - m_use);
        float p[4];
        float ps = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          p[r] = fast_exp2(sc[r] - m_use);
          ps += p[r];
        }
        l_run = l_run * alpha + ps;
        m_run = m_new;
        if (__ballot(alpha != 1.f)) {
#pragma unroll
          for (int g = 0; g < G; ++g)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[g][e] *= alpha;
        }
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int t4 = 0; t4 < 4; ++t4)
              acc[g][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(t.v[g][t4][e], p[t4], acc[g][e],
                                                               0, 0, 0);
      };
      // A two-deep ring: one load per trip (placeholders past the window), compute behind it.
      Tile buf[2];
      load_tile(0, buf[0], true);
      for (int it = 0; it < cnt; it += 2) {
        load_tile(it + 1, buf[1], it + 1 < cnt);
        compute(it, buf[0]);
        load_tile(it + 2, buf[0], it + 2 < cnt);
        if (it + 1 < cnt) compute(it + 1, buf[1]);
      }
    }
    l_run = add_xor32(add_xor16(l_run));

    // Combine over the waves: wave w's m, l and accumulators into LDS, one barrier, then
    // wave w sums elements w * KPW .. of every lane over the waves in a fixed order, each
    // term scaled by 2^(m_w - M) (products rounded before the sum).  Lane element
    // x = (4 g + r) * 4 + e holds O[head i16][64 g + 16 kk + 4 r + e].
    if (smem_busy) __syncthreads();
    smem_busy = true;
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int e = 0; e < 4; ++e) sacc[(wv * E + (4 * g + r) * 4 + e) * 64 + lane] = acc[g][e][r];
    if (kk == 0) {
      sm[wv * 16 + i16] = m_run;
      sl[wv * 16 + i16] = l_run;
    }
    __syncthreads();
    if (!head_ok) return;
    float mw[NW];
    float mx = kNegInf;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      mw[w] = sm[w * 16 + i16];
      mx = fmaxf(mx, mw[w]);
    }
    float den = 0.f, o[KPW];
#pragma unroll
    for (int x = 0; x < KPW; ++x) o[x] = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float wt = mw[w] == kNegInf ? 0.f : fast_exp2(mw[w] - mx);
      den += __fmul_rn(sl[w * 16 + i16], wt);
#pragma unroll
      for (int x = 0; x < KPW; ++x) o[x] += __fmul_rn(sacc[(w * E + wv * KPW + x) * 64 + lane], wt);
    }
    // elements wv * KPW .. + KPW: consecutive e of one (g, r)
    const int x0 = wv * KPW;
    const int g = x0 / 16, r = (x0 / 4) % 4, e0 = x0 % 4;
    const int d0 = 64 * g + 16 * kk + 4 * r + e0;
    auto&& y = args();
    float* dst;
    float inv = 1.f;
    if (WHOLE || (lt0 == 0 && lt1 == n_tiles)) {   // the whole sequence: final output
      inv = den > 0.f ? 1.f / den : 0.f;
      dst = (float*)y.out + ((int64_t)seq * y.num_heads + head) * D + d0;
    } else {
      const int64_t slot = ((int64_t)kvh * y.nseg + segid) * a.group + i16;
      dst = y.ws_acc + slot * D + d0;
      if (wv == 0 && kk == 0) {
        y.ws_ml[slot * 2] = mx;
        y.ws_ml[slot * 2 + 1] = den;
      }
    }
    if constexpr (KPW == 4) {
      *reinterpret_cast<f32x4*>(dst) = f32x4{o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv};
    } else {
      static_assert(KPW == 2, "elements per wave");
      *reinterpret_cast<f32x2*>(dst) = f32x2{o[0] * inv, o[1] * inv};
    }
  };

  if constexpr (!SPLIT) {
    const int nt = seq_tiles(a, sw);
    piece(std::true_type{}, sw, 0, nt, nt, 0);
  } else {
    StreamSizes sizes;
    if (!f32_shares<D, kF32StreamPad>(a, lane, &sizes)) {
      for (int seq = sw; seq < a.num_seqs; seq += a.waves) {
        const int nt = seq_tiles(a, seq);
        piece(std::true_type{}, seq, 0, nt, nt, 0);
      }
      return;
    }
    const int64_t chunk = stream_chunk_of(a, sizes.slots);
    const int64_t start = (int64_t)sw * chunk, end = start + chunk;
    int seq;
    int64_t at;
    stream_locate<kF32StreamPad>(a, lane, -1, start, &seq, &at);
    while (seq < a.num_seqs && at < end) {
      const int nt = seq_tiles(a, seq);
      if (nt > 0) {
        const int64_t t0 = at + kF32StreamPad;   // the sequence's first tile
        const int64_t s0 = start > t0 ? start : t0;
        const int64_t s1 = end < t0 + nt ? end : t0 + nt;
        if (s1 > s0)
          piece(std::false_type{}, seq, (int)(s0 - t0), (int)(s1 - t0), nt, sw + seq);
      }
      at += stream_slots<kF32StreamPad>(nt);
      ++seq;
    }
  }
}

// The split of a float32 call: as many workgroups as can be resident at once, shared by the
// kv heads, over the stream of all sequences' tiles.
struct DecodeF32Layout {
  int64_t waves, nseg;
  size_t ml_bytes, bytes;
};
template <int D>
const void* decode_f32_split_fn(bool rope, bool app) {
  return rope ? (const void*)paged_decode_f32_kernel<D, true, true, true>
              : app ? (const void*)paged_decode_f32_kernel<D, false, true, true>
                    : (const void*)paged_decode_f32_kernel<D, false, false, true>;
}
template <int D>
const void* decode_f32_seq_fn(bool rope, bool app) {
  return rope ? (app ? (const void*)paged_decode_f32_kernel<D, true, true, false>
                     : (const void*)paged_decode_f32_kernel<D, true, false, false>)
              : app ? (const void*)paged_decode_f32_kernel<D, false, true, false>
                    : (const void*)paged_decode_f32_kernel<D, false, false, false>;
}
static DecodeF32Layout decode_f32_layout(int num_seqs, int num_heads, int num_kv_heads,
                                         int head_dim) {
  int64_t resident = resident_workgroups(head_dim == 128 ? decode_f32_split_fn<128>(true, true)
                                                         : decode_f32_split_fn<64>(true, true),
                                         64 * kF32Waves);
  if (resident <= 0) resident = 256;
  DecodeF32Layout lay;
  lay.waves = resident / num_kv_heads;
  if (lay.waves < 1) lay.waves = 1;
  if (lay.waves > kMergeMaxParts - 2) lay.waves = kMergeMaxParts - 2;
  lay.nseg = lay.waves + num_seqs;
  const size_t slots = (size_t)num_kv_heads * lay.nseg * (num_heads / num_kv_heads);
  lay.ml_bytes = (slots * 2 * sizeof(float) + 255) & ~(size_t)255;
  lay.bytes = lay.ml_bytes + slots * head_dim * sizeof(float);
  return lay;
}

// Whether a table may be long enough to split (two launches; the lengths then decide on the
// device, f32_takes_whole): up to here one launch of one workgroup per (kv head, sequence) costs
// less whatever the lengths are.  us split / whole, 8 sequences: head_dim 64 (2 kv heads) at 32
// tiles 14.7 / 11.8, 48 15.3 / 14.9, 63 14.4 / 18.0, 125 18.0 / 29.6, 250 18.1 / 51; head_dim 128
// (4 kv heads) at 16 21.3 / 15.3, 32 21.7 / 21.9, 48 22.0 / 27.7, 63 21.3 / 34, 250 40 / 102.
// Pairs that fill most of the GPU gain nothing from a split of short sequences: 14/2 heads of 64,
// 128 sequences of 85 to 996 tokens 24.2 / 20.5, 64 of 1,000 22.5 / 19.3; 28/4 of 128, 64 of 600
// 42.4 / 38.3, 48 of 122 to 595 28.8 / 26.8 (63 tiles, 48 of 86 to 989: 33.2 / 37.5), and from
// two workgroups per CU 128 of 302 to 599 68.3 / 61.1, 32/32 heads, 16 of 1,000 110 / 102.5.
static bool f32_split_takes(int num_seqs, int num_kv_heads, int head_dim, int64_t max_tiles) {
  const int64_t pairs = (int64_t)num_seqs * num_kv_heads;
  if (head_dim == 64) return max_tiles > (pairs >= 128 && pairs <= 256 ? 64 : 48);
  return max_tiles > (pairs >= 512 ? 64 : pairs >= 192 && pairs <= 256 ? 40 : 32);
}

// Batches whose rows are appended by a launch of their own before whole sequences are attended:
// the wave that attends a row it is given finishes later, which three rounds of workgroups wait
// for three times.  us in one launch / two: 100 sequences of 51 to 498 tokens, 32/8 heads of 128,
// 63.7 / 61.3, 32/32 196 / 184; 128 of 300 32/32 302 / 281; 64 of 600 264 / 256; but 32 of 100 to
// 199 57 / 61, 24 of 504 to 996 118 / 128, and 16 of 400 52 / 62.
static bool f32_append_first(int num_seqs, int num_kv_heads) {
  return num_seqs >= 64 && (int64_t)num_seqs * num_kv_heads >= 768;
}

size_t decode_f32_workspace_bytes(int num_seqs, int num_heads, int num_kv_heads, int head_dim,
                                  int64_t max_tiles) {
  if (!f32_split_takes(num_seqs, num_kv_heads, head_dim, max_tiles)) return 256;
  return decode_f32_layout(num_seqs, num_heads, num_kv_heads, head_dim).bytes;
}

int launch_decode_f32(void* out, const void* q, int64_t q_tok_stride, const void* k_new,
                      int64_t k_tok_stride, const void* v_new, int64_t v_tok_stride,
                      const void* cos, const void* sin, int64_t cs_tok_stride, void* kv_cache,
                      int64_t num_blocks, const int32_t* block_table, int64_t bt_row_stride,
                      int max_blocks_per_seq, const int32_t* context_lens, int num_seqs,
                      int num_heads, int num_kv_heads, int head_dim, int block_size, float scale,
                      void* workspace, size_t workspace_bytes,
                      ndl_stream_t stream) {
  if ((q_tok_stride & 3) || (cos != nullptr && (cs_tok_stride & 3))) return NDL_ERR_INVALID_ARG;
  if ((int64_t)num_seqs * num_kv_heads > 0x7fffffff) return NDL_ERR_UNSUPPORTED;
  DecodeArgs a;
  a.out = (u16*)out;
  a.q = (const u16*)q;
  a.q_tok_stride = q_tok_stride;
  a.kplane = (const u16*)kv_cache;
  a.vplane = (const u16*)((const float*)kv_cache +
                          num_blocks * num_kv_heads * (int64_t)block_size * head_dim);
  a.num_blocks = num_blocks;
  a.num_kv_heads = num_kv_heads;
  a.block_table = block_table;
  a.bt_row_stride = bt_row_stride;
  a.max_blocks = max_blocks_per_seq;
  a.tile_shift = block_tile_shift(block_size);
  a.context_lens = context_lens;
  a.num_heads = num_heads;
  a.group = num_heads / num_kv_heads;
  a.scale_log2 = scale * kLog2e;
  a.num_seqs = num_seqs;
  a.chunk = 0;
  a.min_chunk = kF32MinChunk;
  a.waves = 0;
  a.nseg = 0;
  a.ws_ml = nullptr;
  a.ws_acc = nullptr;
  a.k_new = (const u16*)k_new;
  a.v_new = (const u16*)v_new;
  a.k_new_stride = k_tok_stride;
  a.v_new_stride = v_tok_stride;
  a.rope_cos = (const u16*)cos;
  a.rope_sin = (const u16*)sin;
  a.rope_stride = cs_tok_stride;
  const bool rope = cos != nullptr;
  bool app = k_new != nullptr;
  hipStream_t s = (hipStream_t)stream;
  const int64_t max_tiles = (int64_t)max_blocks_per_seq << a.tile_shift;
  bool split = false;
  if (f32_split_takes(num_seqs, num_kv_heads, head_dim, max_tiles) && workspace != nullptr &&
      ((uintptr_t)workspace & 15u) == 0) {
    const DecodeF32Layout lay = decode_f32_layout(num_seqs, num_heads, num_kv_heads, head_dim);
    split = workspace_bytes >= lay.bytes && lay.nseg <= 0x7fffffff;
    a.waves = (int)lay.waves;
    a.nseg = (int)lay.nseg;
    a.ws_ml = (float*)workspace;
    a.ws_acc = (float*)((char*)workspace + lay.ml_bytes);
  }
  if (app && !split && f32_append_first(num_seqs, num_kv_heads)) {
    const int rc = launch_kv_append(kv_cache, num_blocks, num_kv_heads, block_size, head_dim,
                                    k_new, k_tok_stride, v_new, v_tok_stride, block_table,
                                    bt_row_stride, max_blocks_per_seq, nullptr, context_lens,
                                    num_seqs, num_seqs, cos, sin, cs_tok_stride, kFmtF32, stream);
    if (rc != NDL_OK) return rc;
    app = false;
  }
  const void* fn = split ? (head_dim == 128 ? decode_f32_split_fn<128>(rope, app)
                                            : decode_f32_split_fn<64>(rope, app))
                         : (head_dim == 128 ? decode_f32_seq_fn<128>(rope, app)
                                            : decode_f32_seq_fn<64>(rope, app));
  const int64_t grid = (split ? (int64_t)a.waves : (int64_t)num_seqs) * num_kv_heads;
  void* args[] = {&a};
  if (hipLaunchKernel(fn, dim3((unsigned)grid), dim3(64 * kF32Waves), args, 0, s) != hipSuccess) {
    (void)hipGetLastError();
    return NDL_ERR_LAUNCH;
  }
  const int rc = check_launch();
  if (rc != NDL_OK || !split) return rc;
  return launch_decode_merge<kFmtF32, kF32StreamPad>(a, head_dim, s);
}

}  // namespace ndl
