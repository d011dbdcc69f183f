// Attention of several query tokens per sequence on the matrix cores: softmax(q k^T * scale [+ causal
// mask]) v (attention/kernel.py:6-62), the masking of attention.hip, scale > 0. bf16 in and out, over the
// paged KV cache (a conversation's next turn, a prompt fed in chunks; head_dim 64 and 128) or over
// contiguous keys and values (prefill, head_dim 128); fp32 over contiguous keys and values (head_dim 64
// and 128) in the form at the end of this file. What follows is the bf16 form.
//
// Rows: the group = Hq / Hkv query heads that share a KV head are packed with the queries into
// one row index, row p = query p / group of head p % group, so a staged K / V tile serves every
// head of the group (a short chunk of queries still fills the 16-row MFMA tiles: 3 queries of
// 7 heads are 21 rows) and the rows of a tile see almost the same number of keys.
//
// A 256-thread workgroup owns 64 QB rows of one (sequence, KV head) and a range of 64-key tiles
// (grid.z splits the keys when rows alone leave CUs idle; the splits' partial results go to a
// workspace and packed_attention_merge combines them). Wave w owns 16 QB rows. Per tile, staged
// in LDS as K [key][d] and V^T [d][key] while the next tile's loads are in flight:
//   1. S^T = K Q^T with v_mfma_f32_16x16x32_bf16: lane l = 16 g + r holds the scores of row r for
//      keys 4 g + i of each 16-key block;
//   2. online softmax per row in fp32, base 2, with a lazy rescale of the running output;
//   3. O^T += V^T P^T. The probabilities are fp32; each is the exact sum of three bf16 terms (8
//      mantissa bits each, cut by truncation), and all three go through the MFMA, so that nothing is
//      rounded to 16 bits before the output. The row sums are fp32 adds.
// V^T lies in LDS with the 32 keys of an MFMA step permuted (key 16 h + 4 g + i at 8 g + 4 h + i),
// which is the order in which a lane's probabilities stand, so a V fragment is one 16-byte read.
// The 16-byte units of a V^T row are xor-swizzled by d (the 16 rows of a fragment read fall on
// distinct banks, and the 2-key words of the dense form's transposing stores on few).
//
// Bound by the matrix cores (QK once, PV three times for the split) together with the exponentials of
// the same waves. Measured against one wave per row with a scalar dot per key (attention.hip):
//   paged, 2 x 300 new tokens over 3000 and 1500 cached, 28 / 4 heads, head_dim 128: 16.2 ms
//     before, 74 us now (280 TFLOP/s of attention arithmetic; MFMA 22%, VALU 24% busy) and 8.7 us for
//     the merge of 3 splits;
//   dense causal, 2 x 1000 tokens, 28 / 4 heads, head_dim 128: 1.83 ms before, 60 us now.
// Distance from float64 over these: 1.7e-3 (the rounding of the bf16 output) before and now.
#include "packed_attention.h"

#include "common.h"
#include "skinny.h"

using namespace dk;

namespace {

constexpr int kThreads = 256;
constexpr int kTileK = kPackedTileK;
// log2 of the largest probability the lazy rescale lets through before moving the reference
constexpr float kRescaleLog2 = 8.f;

typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));

// keys row i of sequence b sees, in [0, a.keys]
template <bool kPaged>
__device__ __forceinline__ int visibleKeys(const PackedAttentionArgs& a, int64_t past, int i) {
  int64_t n;
  if (kPaged)
    n = past + (a.causal ? i + 1 : a.seq_q);
  else
    n = a.causal ? static_cast<int64_t>(a.keys) - a.seq_q + i + 1 : a.keys;
  return static_cast<int>(n < 0 ? 0 : (n > a.keys ? a.keys : n));
}

template <bool kPaged>
__device__ __forceinline__ int64_t pastOf(const PackedAttentionArgs& a, int64_t b) {
  if (!kPaged) return 0;
  return a.positions != nullptr ? loadIndex(a.positions, a.pos64, b) : a.past;
}

// element of V^T[d][position] in LDS (the d >> 4 term spreads the dense form's transposing stores)
template <bool kPaged>
__device__ __forceinline__ int vtAt(int d, int pos) {
  const int sw = (kPaged ? d >> 1 : (d >> 1) ^ (d >> 4)) & 7;
  return d * kTileK + ((pos >> 3) ^ sw) * 8 + (pos & 7);
}
// position of a tile's key in a V^T row
__device__ __forceinline__ int vtPos(int key) {
  return (key & 32) + ((key >> 2) & 3) * 8 + ((key >> 4) & 1) * 4 + (key & 3);
}

// True if a sum is an infinity or a NaN. An infinite or NaN value always makes it so, but the matrix
// product may give a NaN where the row's own arithmetic has an infinity or a finite result: the key may
// be one that the row does not see (probability 0), and one that it sees meets the terms of p with
// either sign. A workgroup with such a sum redoes its rows key by key.
__device__ __forceinline__ bool nonFinite(const f32x4& v) {
  bool bad = false;
#pragma unroll
  for (int k = 0; k < 4; ++k) bad = bad || (__float_as_uint(v[k]) & 0x7F800000u) == 0x7F800000u;
  return bad;
}

// row of the splits' partial results
__device__ __forceinline__ int64_t partIndex(const PackedAttentionArgs& a, int unit, int rows,
                                             int p) {
  return (static_cast<int64_t>(blockIdx.z) * gridDim.y + unit) * rows + p;
}

template <int D, typename T>
__device__ __forceinline__ T* outRow(const PackedAttentionArgs& a, int b, int kvh,
                                            int group, int p) {
  const int i = p / group, h = kvh * group + p - i * group;
  return static_cast<T*>(a.out) + ((static_cast<int64_t>(b) * a.q_heads + h) * a.seq_q + i) * D;
}

// Row p over the keys [j0, j1) that it sees, by one wave without the matrix cores: lane j scores
// a key, then owns the outputs lane + 64 u. Keys that the row does not see are never touched.
template <int D, bool kPaged, typename T>
__device__ __forceinline__ void rowByKeys(const PackedAttentionArgs& a, int unit, int rows, int p,
                                       int j0, int j1) {
  const int lane = threadIdx.x % kWave, group = a.q_heads / a.kv_heads;
  const int b = unit / a.kv_heads, kvh = unit % a.kv_heads, i = p / group;
  const int lim = visibleKeys<kPaged>(a, pastOf<kPaged>(a, b), i);
  const T* q = static_cast<const T*>(a.q) +
               ((static_cast<int64_t>(b) * a.q_heads + kvh * group + p % group) * a.seq_q + i) * D;
  auto block = [&](int j) {  // first element of the key's (block, head), or of the (b, head)
    if constexpr (kPaged) {
      const int64_t blk = gp(a.block_table)[b * a.max_blocks + j / a.block_size];
      return (blk * a.kv_heads + kvh) * a.block_size * D;
    } else {
      return static_cast<int64_t>(unit) * a.keys * D;
    }
  };
  const int size = kPaged ? a.block_size : a.keys;
  if (j1 > lim) j1 = lim;
  float m = -INFINITY, l = 0.f, acc[D / kWave] = {};
  for (; j0 < j1; j0 += kWave) {
    const int j = j0 + lane;
    float s = -INFINITY;
    if (j < j1) {
      const T* k = static_cast<const T*>(a.k) + block(j) + static_cast<int64_t>(j % size) * D;
      float dot = 0.f;
      for (int d = 0; d < D; ++d) dot = fmaf(ld(q + d), ld(k + d), dot);
      s = dot * a.scale_log2;
    }
    const float next = fmaxf(m, waveMax(s));
    const float base = next == -INFINITY ? 0.f : next;
    const float w = j < j1 ? __builtin_amdgcn_exp2f(s - base) : 0.f;
    const float alpha = __builtin_amdgcn_exp2f(m - base);
    l = l * alpha + waveSum(w);
    m = next;
#pragma unroll
    for (int u = 0; u < D / kWave; ++u) acc[u] *= alpha;
    for (int jj = j0; jj < j1 && jj < j0 + kWave; ++jj) {
      const float pj = __shfl(w, jj - j0, kWave);
      const T* v = static_cast<const T*>(a.v) + block(jj);
#pragma unroll
      for (int u = 0; u < D / kWave; ++u) {
        const int64_t d = lane + u * kWave, at = jj % size;
        acc[u] = fmaf(pj, ld(v + (kPaged ? d * size + at : at * D + d)), acc[u]);
      }
    }
  }
  if (a.splits > 1) {
    const int64_t at = partIndex(a, unit, rows, p);
    if (lane == 0) {
      gp(a.part_ml)[at * 2] = m;
      gp(a.part_ml)[at * 2 + 1] = l;
    }
#pragma unroll
    for (int u = 0; u < D / kWave; ++u) gp(a.part_o)[at * D + lane + u * kWave] = acc[u];
    return;
  }
  const float inv = lim > 0 ? 1.f / l : 0.f;
  T* out = outRow<D, T>(a, b, kvh, group, p);
#pragma unroll
  for (int u = 0; u < D / kWave; ++u) st(out + lane + u * kWave, acc[u] * inv);
}

template <int D, int QB, bool kPaged>
__device__ __forceinline__ void packedAttention(const PackedAttentionArgs& a) {
  static_assert(D == 64 || D == 128, "head_dim");
  constexpr int kTileQ = 64 * QB;
  constexpr int kPitch = D + 8;          // K row pitch: 16 rows start on 16 distinct 4-bank groups
  constexpr int kChunks = D / 8;         // 16-byte chunks per key
  constexpr int kPer = kTileK * kChunks / kThreads;  // chunks of K (and of V) per thread
  constexpr int DT = D / 16, DK = D / 32;
  __shared__ __attribute__((aligned(16))) uint16_t Ks[kTileK * kPitch];
  __shared__ __attribute__((aligned(16))) uint16_t Vt[D * kTileK];
  const int t = threadIdx.x, lane = t % kWave, wave = t / kWave;
  const int r = lane % 16, g = lane / 16;
  const int group = a.q_heads / a.kv_heads;
  const int rows = a.seq_q * group;
  // the (sequence, KV head) is the fast index (consecutive workgroups go to different XCDs, so
  // one pair's tiles meet in one L2 when the pairs are a multiple of the XCDs), the row tile the
  // slow one, last tile first: under a causal mask the longest workgroups start first
  const uint32_t lin = blockIdx.x + gridDim.x * blockIdx.y;
  const int unit = static_cast<int>(lin % gridDim.y);
  const int b = unit / a.kv_heads, kvh = unit - b * a.kv_heads;
  const int p0 = (gridDim.x - 1 - lin / gridDim.y) * kTileQ;
  const int pw = p0 + wave * 16 * QB;  // the wave's first row
  const bool active = pw < rows;       // uniform over the wave
  const int64_t past = pastOf<kPaged>(a, b);
  auto query = [&](int p) { return (p < rows ? p : rows - 1) / group; };

  U128 qf[QB][DK];
  int lim[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const int p = pw + qb * 16 + r < rows ? pw + qb * 16 + r : rows - 1;  // clamped: not stored
    const int i = p / group, h = kvh * group + p - i * group;
    const uint16_t* qp = static_cast<const uint16_t*>(a.q) +
                         ((static_cast<int64_t>(b) * a.q_heads + h) * a.seq_q + i) * D + g * 8;
#pragma unroll
    for (int c = 0; c < DK; ++c) qf[qb][c] = gload16(qp + c * 32);
    lim[qb] = visibleKeys<kPaged>(a, past, i);
  }
  // keys some row of the workgroup sees; keys every row of this wave sees
  const int wg_keys = visibleKeys<kPaged>(a, past, query(p0 + kTileQ - 1));
  const int wave_full = visibleKeys<kPaged>(a, past, query(pw));

  const int all_tiles = (wg_keys + kTileK - 1) / kTileK;
  const int per = (all_tiles + a.splits - 1) / a.splits;
  const int kt0 = static_cast<int>(blockIdx.z) * per;
  const int kt1 = kt0 + per < all_tiles ? kt0 + per : all_tiles;

  // staging. K (both forms) and the paged V^T: chunk c = t + 256 i of the tile; dense V: chunk
  // pairs (keys 2 p and 2 p + 1 at 8 columns), stored transposed as 2-key words
  const int64_t dense_base = static_cast<int64_t>(unit) * a.keys * D;
  U128 kr[kPer], vr[kPer];
  auto fetch = [&](int kt) {
    const int k0 = kt * kTileK;
    if constexpr (kPaged) {
      const int64_t blk = gp(a.block_table)[b * a.max_blocks + k0 / a.block_size];
      const int slot = k0 % a.block_size;
      const int64_t base = (blk * a.kv_heads + kvh) * a.block_size * D;
      const uint16_t* kq = static_cast<const uint16_t*>(a.k) + base + static_cast<int64_t>(slot) * D;
      const uint16_t* vq = static_cast<const uint16_t*>(a.v) + base + slot;
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        const int c = t + i * kThreads;
        kr[i] = gload16(kq + c * 8);
        vr[i] = gload16(vq + static_cast<int64_t>(c / 8) * a.block_size + (c % 8) * 8);
      }
    } else {
      const int64_t at = dense_base + static_cast<int64_t>(k0) * D;
      const uint16_t* kq = static_cast<const uint16_t*>(a.k) + at;
      const uint16_t* vq = static_cast<const uint16_t*>(a.v) + at;
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        const int c = t + i * kThreads;
        const int e = t + (i / 2) * kThreads;
        const int vkey = 2 * (e / kChunks) + i % 2;
        kr[i] = k0 + c / kChunks < a.keys ? gload16(kq + c * 8) : zero16();
        vr[i] = k0 + vkey < a.keys ? gload16(vq + vkey * D + (e % kChunks) * 8) : zero16();
      }
    }
  };
  // In a tile with keys past the last visible one, those values are zeroed (their probabilities
  // are 0, but what a recycled cache block holds there could be an infinity or a NaN).
  auto zeroPast = [&](int k0) {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      if constexpr (kPaged) {
        const int key = k0 + ((t + i * kThreads) % 8) * 8;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const uint32_t lo = key + 2 * w < wg_keys ? 0xFFFFu : 0u;
          const uint32_t hi = key + 2 * w + 1 < wg_keys ? 0xFFFF0000u : 0u;
          vr[i][w] &= lo | hi;
        }
      } else {
        const int key = k0 + 2 * ((t + (i / 2) * kThreads) / kChunks) + i % 2;
        if (key >= wg_keys) vr[i] = zero16();
      }
    }
  };
  auto stash = [&] {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int c = t + i * kThreads;
      *reinterpret_cast<U128*>(&Ks[(c / kChunks) * kPitch + (c % kChunks) * 8]) = kr[i];
    }
    if constexpr (kPaged) {
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        const int c = t + i * kThreads, d = c / 8, key = (c % 8) * 8;
        *reinterpret_cast<uint2*>(&Vt[vtAt<kPaged>(d, vtPos(key))]) = uint2{vr[i][0], vr[i][1]};
        *reinterpret_cast<uint2*>(&Vt[vtAt<kPaged>(d, vtPos(key + 4))]) = uint2{vr[i][2], vr[i][3]};
      }
    } else {
#pragma unroll
      for (int i = 0; i < kPer; i += 2) {
        const int e = t + (i / 2) * kThreads;
        const int pos = vtPos(2 * (e / kChunks)), d0 = (e % kChunks) * 8;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t even = (vr[i][j] & 0xFFFFu) | (vr[i + 1][j] << 16);
          const uint32_t odd = (vr[i][j] >> 16) | (vr[i + 1][j] & 0xFFFF0000u);
          *reinterpret_cast<uint32_t*>(&Vt[vtAt<kPaged>(d0 + 2 * j, pos)]) = even;
          *reinterpret_cast<uint32_t*>(&Vt[vtAt<kPaged>(d0 + 2 * j + 1, pos)]) = odd;
        }
      }
    }
  };

  f32x4 o[QB][DT];  // O^T tiles: d = 16 dt + 4 g + i, row pw + 16 qb + r
  float lsum[QB];   // row sums over the lane group's keys
  float m_run[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    m_run[qb] = -INFINITY;
    lsum[qb] = 0.f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[qb][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  if (kt0 < kt1) fetch(kt0);
  for (int kt = kt0; kt < kt1; ++kt) {
    const int k0 = kt * kTileK;
    if (k0 + kTileK > wg_keys) zeroPast(k0);
    __syncthreads();  // the previous tile is no longer read
    stash();
    __syncthreads();
    if (kt + 1 < kt1) fetch(kt + 1);
    if (!active) continue;

    __builtin_amdgcn_sched_barrier(0);
    // 1. S^T for 4 blocks of 16 keys and each row block
    f32x4 s[QB][4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const uint16_t* krow = &Ks[(kk * 16 + r) * kPitch + g * 8];
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) s[qb][kk] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < DK; ++c) {
        const U128 ka = *reinterpret_cast<const U128*>(krow + c * 32);
#pragma unroll
        for (int qb = 0; qb < QB; ++qb)
          s[qb][kk] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(asBf16x8(ka), asBf16x8(qf[qb][c]),
                                                              s[qb][kk], 0, 0, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    // 2. online softmax per row (keys a row does not see: -inf), reference point in scaled units
    const bool full = k0 + kTileK <= wave_full;  // uniform over the wave: every key visible
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      float tmax = -INFINITY;
      if (!full) {
        const int key0 = k0 + g * 4;
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            s[qb][kk][i] = key0 + kk * 16 + i < lim[qb] ? s[qb][kk][i] : -INFINITY;
      }
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
#pragma unroll
        for (int i = 0; i < 4; ++i) tmax = fmaxf(tmax, s[qb][kk][i]);
      tmax = rowsMax(tmax);  // over the four lane groups: the row's 64 keys
      // the reference moves only when a score passes it by more than kRescaleLog2, so
      // probabilities stay below 2^kRescaleLog2; a row that has seen no key keeps -inf
      const float tm = tmax * a.scale_log2;
      const bool grow = tm > m_run[qb] + kRescaleLog2;  // false while tm = -inf
      if (__builtin_amdgcn_ballot_w64(grow)) {
        const float alpha = grow ? __builtin_amdgcn_exp2f(m_run[qb] - tm) : 1.f;  // 0 from -inf
        m_run[qb] = grow ? tm : m_run[qb];
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[qb][dt] *= alpha;
        lsum[qb] *= alpha;
      }
      const float base = m_run[qb] == -INFINITY ? 0.f : m_run[qb];
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          s[qb][kk][i] = __builtin_amdgcn_exp2f(fmaf(s[qb][kk][i], a.scale_log2, -base));
      const f32x4 part = (s[qb][0] + s[qb][1]) + (s[qb][2] + s[qb][3]);
      lsum[qb] += (part[0] + part[1]) + (part[2] + part[3]);
    }
    __builtin_amdgcn_sched_barrier(0);
    // 3. O^T += V^T P^T, 32 keys per step; each V^T fragment serves every term of every row block
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
      // lane group g: keys 4 g + i of blocks 2 kc and 2 kc + 1; the largest term first. Cut off
      // instead of rounded, a term is one byte permute of two values (2 x 300 queries over 3000
      // keys, head_dim 64: 55 us, 61 with rounded terms)
      bf16x8 pt[3][QB];
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
#pragma unroll
        for (int u = 0; u < 3; ++u) {
          U128 w;
#pragma unroll
          for (int j = 0; j < 4; ++j) {  // keys 2 j and 2 j + 1 of the lane's 8
            f32x4& x = s[qb][2 * kc + j / 2];
            const int i = 2 * (j % 2);
            const uint32_t lo = __float_as_uint(x[i]), hi = __float_as_uint(x[i + 1]);
            w[j] = __builtin_amdgcn_perm(hi, lo, 0x07060302u);  // the upper halves
            x[i] -= __uint_as_float(lo & 0xFFFF0000u);
            x[i + 1] -= __uint_as_float(hi & 0xFFFF0000u);
          }
          pt[u][qb] = asBf16x8(w);
        }
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const U128 va = *reinterpret_cast<const U128*>(&Vt[vtAt<kPaged>(dt * 16 + r, kc * 32 + g * 8)]);
#pragma unroll
        for (int u = 2; u >= 0; --u)
#pragma unroll
          for (int qb = 0; qb < QB; ++qb)
            o[qb][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(asBf16x8(va), pt[u][qb],
                                                                o[qb][dt], 0, 0, 0);
      }
    }
  }

  bool bad = false;
#pragma unroll
  for (int qb = 0; qb < QB; ++qb)
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) bad = bad || nonFinite(o[qb][dt]);
  if (__syncthreads_or(bad)) {
    for (int q = wave; q < kTileQ && p0 + q < rows; q += kThreads / kWave)
      rowByKeys<D, kPaged, bf16>(a, unit, rows, p0 + q, kt0 * kTileK, kt1 * kTileK);
    return;
  }
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const float l = rowsSum(lsum[qb]);
    const int p = pw + qb * 16 + r;
    if (p >= rows) continue;
    if (a.splits > 1) {
      const int64_t at = partIndex(a, unit, rows, p);
      if (g == 0) {
        gp(a.part_ml)[at * 2] = m_run[qb];
        gp(a.part_ml)[at * 2 + 1] = l;
      }
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        *gp(reinterpret_cast<f32x4*>(a.part_o + at * D + dt * 16 + g * 4)) = o[qb][dt];
      continue;
    }
    // a row that sees no key gives zeros; one whose visible scores are all -inf gives NaN
    const float inv = lim[qb] > 0 ? 1.f / l : 0.f;
    uint16_t* orow = outRow<D, uint16_t>(a, b, kvh, group, p) + g * 4;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const uint32_t lo = packBf16x2(o[qb][dt][0] * inv, o[qb][dt][1] * inv);
      const uint32_t hi = packBf16x2(o[qb][dt][2] * inv, o[qb][dt][3] * inv);
      *gp(reinterpret_cast<uint2*>(orow + dt * 16)) = uint2{lo, hi};
    }
  }
}

// ---- fp32, contiguous keys and values --------------------------------------------------------------
// The same rows and tiles with v_mfma_f32_16x16x4_f32 (lane l = 16 g + r supplies A[r][g] and
// B[g][r] and receives D[4 g + i][r]): scores S^T = K Q^T with lane group g on
// the g-th quarter of d, one 16-row block per wave. A lane's scores, keys 4 g + i of each 16-key block, are the B operand of
// O^T += V^T P^T as they stand (step i takes key 4 g + i from every group), so the probabilities
// stay in fp32 registers; V keeps its [key][d] layout, 16 consecutive d per operand row. K and V rows
// are D + 4 floats apart: the rows of a K fragment and the four keys of a V fragment start on
// different banks. Bound by the fp32 matrix instruction (a sixteenth of the bf16 rate) and the
// longest rows: 2 x 500 tokens, 14 / 2 heads, head_dim 64, causal 30 us, 150 with one wave per row and
// a scalar dot.
template <int D>
__device__ __forceinline__ void packedAttentionF32(const PackedAttentionArgs& a) {
  constexpr int kPitch = D + 4, kRowChunks = D / 4, kPer = kTileK * kRowChunks / kThreads;
  constexpr int DT = D / 16, DC = D / 16;  // 16-wide d blocks of O; 4-float chunks per lane group
  __shared__ __attribute__((aligned(16))) float Ks[kTileK * kPitch];
  __shared__ __attribute__((aligned(16))) float Vs[kTileK * kPitch];
  const int t = threadIdx.x, lane = t % kWave, wave = t / kWave;
  const int r = lane % 16, g = lane / 16;
  const int group = a.q_heads / a.kv_heads, rows = a.seq_q * group;
  const uint32_t lin = blockIdx.x + gridDim.x * blockIdx.y;
  const int unit = static_cast<int>(lin % gridDim.y);
  const int b = unit / a.kv_heads, kvh = unit - b * a.kv_heads;
  const int p0 = (gridDim.x - 1 - lin / gridDim.y) * 64, pw = p0 + wave * 16;
  const bool active = pw < rows;  // uniform over the wave
  auto query = [&](int p) { return (p < rows ? p : rows - 1) / group; };
  const int pr = pw + r < rows ? pw + r : rows - 1;  // clamped: not stored
  const int i0 = pr / group;
  f32x4 qf[DC];  // d = g * (D / 4) + 4 c + j
  {
    const int h = kvh * group + pr - i0 * group;
    const float* qp = static_cast<const float*>(a.q) +
                      ((static_cast<int64_t>(b) * a.q_heads + h) * a.seq_q + i0) * D + g * (D / 4);
#pragma unroll
    for (int c = 0; c < DC; ++c) qf[c] = *gp(reinterpret_cast<const f32x4*>(qp + c * 4));
  }
  const int lim = visibleKeys<false>(a, 0, i0);
  const int wg_keys = visibleKeys<false>(a, 0, query(p0 + 63));
  const int wave_full = visibleKeys<false>(a, 0, query(pw));
  const int tiles = (wg_keys + kTileK - 1) / kTileK;

  const int64_t base = static_cast<int64_t>(unit) * a.keys * D;
  f32x4 kr[kPer], vr[kPer];
  auto fetch = [&](int kt) {
    const int k0 = kt * kTileK;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int c = t + i * kThreads;
      const int64_t at = base + static_cast<int64_t>(k0) * D + c * 4;
      const bool in = k0 + c / kRowChunks < a.keys;
      kr[i] = in ? *gp(reinterpret_cast<const f32x4*>(static_cast<const float*>(a.k) + at))
                 : f32x4{0.f, 0.f, 0.f, 0.f};
      vr[i] = in ? *gp(reinterpret_cast<const f32x4*>(static_cast<const float*>(a.v) + at))
                 : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  };
  f32x4 o[DT];  // O^T: d = 16 dt + 4 g + i, row pw + r
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;
  if (tiles > 0) fetch(0);
  for (int kt = 0; kt < tiles; ++kt) {
    const int k0 = kt * kTileK;
    __syncthreads();  // the previous tile is no longer read
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int c = t + i * kThreads, at = (c / kRowChunks) * kPitch + (c % kRowChunks) * 4;
      *reinterpret_cast<f32x4*>(&Ks[at]) = kr[i];
      *reinterpret_cast<f32x4*>(&Vs[at]) = vr[i];
    }
    __syncthreads();
    if (kt + 1 < tiles) fetch(kt + 1);
    if (!active) continue;
    f32x4 s[4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      s[kk] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < DC; ++c) {
        const f32x4 kf =
            *reinterpret_cast<const f32x4*>(&Ks[(kk * 16 + r) * kPitch + g * (D / 4) + c * 4]);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          s[kk] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[j], qf[c][j], s[kk], 0, 0, 0);
      }
    }
    if (k0 + kTileK > wave_full) {  // uniform over the wave
      const int key0 = k0 + g * 4;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          s[kk][i] = key0 + kk * 16 + i < lim ? s[kk][i] : -INFINITY;
    }
    float tmax = -INFINITY;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int i = 0; i < 4; ++i) tmax = fmaxf(tmax, s[kk][i]);
    const float tm = rowsMax(tmax) * a.scale_log2;
    const bool grow = tm > m_run + kRescaleLog2;  // false while tm = -inf
    if (__builtin_amdgcn_ballot_w64(grow)) {
      const float alpha = grow ? __builtin_amdgcn_exp2f(m_run - tm) : 1.f;  // 0 from -inf
      m_run = grow ? tm : m_run;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) o[dt] *= alpha;
      l_run *= alpha;
    }
    const float ref = m_run == -INFINITY ? 0.f : m_run;
    float sum = 0.f;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[kk][i] = __builtin_amdgcn_exp2f(fmaf(s[kk][i], a.scale_log2, -ref));
        sum += s[kk][i];
      }
    l_run += sum;  // this lane group's keys; the groups are added at the end
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
          o[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(
              Vs[(kk * 16 + g * 4 + i) * kPitch + dt * 16 + r], s[kk][i], o[dt], 0, 0, 0);
  }
  bool bad = false;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) bad = bad || nonFinite(o[dt]);
  if (__syncthreads_or(bad)) {
    for (int q = wave; q < 64 && p0 + q < rows; q += kThreads / kWave)
      rowByKeys<D, false, float>(a, unit, rows, p0 + q, 0, tiles * kTileK);
    return;
  }
  const float l = rowsSum(l_run);
  if (pw + r >= rows) return;
  const float inv = lim > 0 ? 1.f / l : 0.f;
  float* orow = outRow<D, float>(a, b, kvh, group, pw + r) + g * 4;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) *gp(reinterpret_cast<f32x4*>(orow + dt * 16)) = o[dt] * inv;
}

// Combines the key splits: D / 4 lanes per row, 16 bytes of every split's sums each.
template <int D, bool kPaged>
__device__ __forceinline__ void packedMerge(const PackedAttentionArgs& a, int units) {
  constexpr int kLanes = D / 4, kRows = kThreads / kLanes;
  const int group = a.q_heads / a.kv_heads;
  const int64_t rows = static_cast<int64_t>(a.seq_q) * group, total = rows * units;
  const int d = (threadIdx.x % kLanes) * 4;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * kRows + threadIdx.x / kLanes;
  if (row >= total) return;
  float m = -INFINITY;
  for (int z = 0; z < a.splits; ++z) m = fmaxf(m, gp(a.part_ml)[(z * total + row) * 2]);
  f32x4 acc{0.f, 0.f, 0.f, 0.f};
  float l = 0.f;
  for (int z = 0; z < a.splits; ++z) {
    const int64_t at = z * total + row;
    const float mz = gp(a.part_ml)[at * 2];
    const float w = mz == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mz - m);
    l = fmaf(w, gp(a.part_ml)[at * 2 + 1], l);
    acc += w * *gp(reinterpret_cast<const f32x4*>(a.part_o + at * D + d));
  }
  const int unit = static_cast<int>(row / rows), p = static_cast<int>(row % rows);
  const int b = unit / a.kv_heads, kvh = unit % a.kv_heads;
  const float inv = visibleKeys<kPaged>(a, pastOf<kPaged>(a, b), p / group) > 0 ? 1.f / l : 0.f;
  *gp(reinterpret_cast<uint2*>(outRow<D, uint16_t>(a, b, kvh, group, p) + d)) =
      uint2{packBf16x2(acc[0] * inv, acc[1] * inv), packBf16x2(acc[2] * inv, acc[3] * inv)};
}

}  // namespace

// Grid {ceil(rows / (64 QB)), B Hkv, splits}. At most 256 VGPRs (two workgroups per CU), which
// keeps the MFMA accumulators in VGPRs.
#define DK_PACKED(name, D, QB, PAGED)                                                            \
  extern "C" __global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2))) \
      name(PackedAttentionArgs a) {                                                              \
    packedAttention<D, QB, PAGED>(a);                                                            \
  }
DK_PACKED(packed_attention_paged_d64, 64, 1, true)
DK_PACKED(packed_attention_paged_d64_r128, 64, 2, true)
DK_PACKED(packed_attention_paged_d128, 128, 1, true)
DK_PACKED(packed_attention_paged_d128_r128, 128, 2, true)
DK_PACKED(packed_attention_dense_d128, 128, 1, false)
DK_PACKED(packed_attention_dense_d128_r128, 128, 2, false)

// Grid {ceil(rows / 64), B Hkv}.
extern "C" __global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
    packed_attention_f32_d64(PackedAttentionArgs a) {
  packedAttentionF32<64>(a);
}
extern "C" __global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
    packed_attention_f32_d128(PackedAttentionArgs a) {
  packedAttentionF32<128>(a);
}

// Grid {ceil(B Hq Sq / (1024 / D))}; units = B Hkv.
extern "C" __global__ void __launch_bounds__(kThreads)
    packed_attention_merge_d64(PackedAttentionArgs a, int units) {
  packedMerge<64, true>(a, units);
}
extern "C" __global__ void __launch_bounds__(kThreads)
    packed_attention_merge_d128(PackedAttentionArgs a, int units) {
  packedMerge<128, true>(a, units);
}
