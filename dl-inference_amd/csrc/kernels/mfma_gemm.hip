// 16-bit MFMA GEMMs on gfx950 (linears and the fused projections of many rows; decode sizes use the
// weight-streaming kernels of gemm.hip / decode.hip; fp32: mfma_gemm_f32.hip).
//
//   C[r, c] = sum_k A(r, k) * B(c, k), then an epilogue per output element (bias, ReLU, layout)
//
//  mfma_linear_bf16_<t>, mfma_linear_f16_<t>  16-bit x, w (K % 8 == 0; linear/kernel.py:6-44), MFMA
//                           16x16x32, fp32 accumulation, 16-bit or fp32 out, optional ReLU. (f16,
//                           1000 x 4864 x 896: 252 us on the general kernel of gemm.hip, 19 us here)
//  mfma_linear_residual_bf16_<t>  the same plus a residual add (bf16 out)
//  mfma_gate_up_silu_bf16_<t>     the same over an interleaved gate/up weight, SwiGLU epilogue
//  mfma_qkv_heads_bf16_<t>        q|k|v projection with RoPE into attention's layout
//  *_splitk*                K split over grid.z into a workspace, then a fixed-order sum
//
// Work split: 256 threads own a BM x BN tile of C (4 waves, 2 x 2, each BM/2 x BN/2 as 16 x 16 MFMA
// tiles) and walk K in BK-wide slices, two slices in flight in registers and two LDS buffers, tiles
// ordered by XCD (gemm_tiles.h). Rows and columns past the ends load clamped rows whose results are
// dropped and k past the end loads zeros, so any shape works. Every output is a fixed-order sum:
// results do not depend on timing.
#include "common.h"
#include "gemm_tiles.h"
#include "skinny.h"

using namespace dk;

namespace {

// ---- 16-bit core ---------------------------------------------------------------------------------
// v_mfma_f32_16x16x32_bf16 / _f16 (E = Bf16 / F16): lane l supplies A[l % 16][(l / 16) * 8 + j] and
// B[(l / 16) * 8 + j][l % 16], j < 8. Operands are [rows, K] row-major with K % 8 == 0 and
// 16-byte aligned rows, loaded 8 elements at a time.
//
// Pipeline (one 64-wide K slice per step): the slice being multiplied sits in one of two LDS
// buffers, the next one is written into the other from registers loaded two steps earlier, and
// the loads for the slice after that go out into the registers just written, all interleaved
// with the MFMAs (sched_group_barrier: one LDS read, or one LDS write and one global load, per two
// MFMAs; one per MFMA measured 15% slower on the 8192 x 9728 x 896 gate_up and 10% on down_proj),
// with one barrier per step. LDS rows hold 8 16-byte
// chunks, chunk c of row r at position c ^ ((r >> 1) & 7): the 16 lanes of a fragment read
// (rows r..r+15, one chunk) and the 16 lanes of a stash write (two rows) then fall on 16
// different 4-bank groups of the 64 banks (no conflicts; SQ_LDS_BANK_CONFLICT reads 0).
//
// Tiles in the XCD-grouped order (groupedTile).

// ld: row stride of a and b in elements (K for whole rows; a split-K part passes a and b offset
// to its first column, its own K and the full row stride).
// BK: K columns per slice, 64 or 128 (128 doubles the bytes each workgroup has in flight: the
// decode-sized kernels, whose few workgroups stream the weights).
// kStreamB: b (the weights) is read with nontemporal loads, for the decode-sized kernels, whose
// single row tile reads every weight once (many row tiles re-read them and keep cached loads).
// Each load instruction covers whole 128-byte lines (16 lanes per 256-byte row slice of a
// 128-wide slice); a streaming probe over 1 GiB read 6.5-6.9 TB/s that way against 5.8-6.0 with
// cached loads.
// G: groups of 256 threads that take equal runs of K slices of the same tile, each with operand
// buffers of its own; the epilogue adds the groups' sums in group order. One group walks K one slice
// per load and LDS round trip (about 550 cycles for 64 x 64, of which 256 are the slice's 16 KB at
// 64 bytes a cycle), so a grid that leaves CUs with one workgroup gains from a second group.
template <int BM, int BN, int BK = 64, bool kStreamB = false, class E = Bf16, int G = 1, class Epi>
__device__ __forceinline__ void gemm16(const uint16_t* a, const uint16_t* b, int64_t R,
                                       int64_t Cn, int64_t K, int64_t ld, const Epi& epi) {
  static_assert(BK == 64 || BK == 128, "slice width");
  constexpr int TM = BM / 32, TN = BN / 32;
  constexpr int VPR = BK / 8;  // 16-byte chunks per tile row
  constexpr int AV = BM * VPR / kGemmThreads, BV = BN * VPR / kGemmThreads;
  // the two operand buffers, then (after the last slice) the fp32 accumulator tile of the
  // epilogue, row pitch BN + 4 floats (the 4 row groups of an MFMA tile store land 16 banks apart)
  constexpr int CP = BN + 4;
  constexpr int kOperandBytes = 2 * (BM + BN) * BK * 2, kTileBytes = BM * CP * 4;
  constexpr int kGroupBytes = kOperandBytes > kTileBytes ? kOperandBytes : kTileBytes;
  constexpr int kThreads = G * kGemmThreads;
  __shared__ __attribute__((aligned(16))) uint8_t smem[G * kGroupBytes];
  const int t = threadIdx.x % kGemmThreads, lane = t % kWave;
  // uniform over the wave
  const int wave = __builtin_amdgcn_readfirstlane(t / kWave);
  const int grp = G == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / kGemmThreads);
  uint16_t* const As0 = reinterpret_cast<uint16_t*>(smem + grp * kGroupBytes);
  uint16_t* const Bs0 = As0 + BM * BK;
  uint16_t* const As1 = Bs0 + BN * BK;
  uint16_t* const Bs1 = As1 + BM * BK;
  const int wr = wave / 2, wc = wave % 2;
  int64_t r0, c0;
  groupedTile(BM, BN, r0, c0);
  // the group's slices; every group makes the same number of steps (and barriers), the last one's
  // steps past K multiply zeros
  const int64_t slices = (K + BK - 1) / BK, nk = (slices + G - 1) / G;
  int64_t whole = K;  // columns that every group has
  if constexpr (G > 1) {
    const int64_t per = nk * BK;
    whole = K - (G - 1) * per;
    a += grp * per;
    b += grp * per;
    K -= grp * per;
    K = K < per ? K : per;
  }
  // 64-wide slices: rows of 128 bytes, two rows fill the 64 banks, chunk c at c ^ ((r >> 1) & 7);
  // 128-wide: rows of 256 bytes, chunk c of 16 at c ^ (r & 15)
  auto at = [](int row, int c) {
    return row * BK + (BK == 64 ? c ^ ((row >> 1) & 7) : c ^ (row & 15)) * 8;
  };
  // the thread's source rows, clamped into range (a clamped row loads a real row whose results
  // the epilogue drops); k past K loads zeros, in the last slice only
  const uint16_t* pa[AV];
  const uint16_t* pb[BV];
  const int kc = (t % VPR) * 8;
#pragma unroll
  for (int i = 0; i < AV; ++i) {
    const int64_t row = r0 + (t + i * kGemmThreads) / VPR;
    pa[i] = a + (row < R ? row : R - 1) * ld + kc;
  }
#pragma unroll
  for (int i = 0; i < BV; ++i) {
    const int64_t row = c0 + (t + i * kGemmThreads) / VPR;
    pb[i] = b + (row < Cn ? row : Cn - 1) * ld + kc;
  }
  auto loadB = [](const uint16_t* p) {
    if constexpr (kStreamB)
      return __builtin_nontemporal_load(gp(reinterpret_cast<const U128*>(p)));
    else
      return gload16(p);
  };
  auto fetch = [&](U128 (&xa)[AV], U128 (&xb)[BV], int64_t k0) {
    if (k0 + BK <= K) {
#pragma unroll
      for (int i = 0; i < AV; ++i) xa[i] = gload16(pa[i] + k0);
#pragma unroll
      for (int i = 0; i < BV; ++i) xb[i] = loadB(pb[i] + k0);
    } else {
      const bool in = k0 + kc < K;
#pragma unroll
      for (int i = 0; i < AV; ++i) xa[i] = in ? gload16(pa[i] + k0) : zero16();
#pragma unroll
      for (int i = 0; i < BV; ++i) xb[i] = in ? loadB(pb[i] + k0) : zero16();
    }
  };
  auto fetchWhole = [&](U128 (&xa)[AV], U128 (&xb)[BV], int64_t k0) {
#pragma unroll
    for (int i = 0; i < AV; ++i) xa[i] = gload16(pa[i] + k0);
#pragma unroll
    for (int i = 0; i < BV; ++i) xb[i] = loadB(pb[i] + k0);
  };
  auto stash = [&](const U128 (&xa)[AV], const U128 (&xb)[BV], uint16_t* as, uint16_t* bs) {
#pragma unroll
    for (int i = 0; i < AV; ++i) {
      const int e = t + i * kGemmThreads;
      *reinterpret_cast<U128*>(&as[at(e / VPR, e % VPR)]) = xa[i];
    }
#pragma unroll
    for (int i = 0; i < BV; ++i) {
      const int e = t + i * kGemmThreads;
      *reinterpret_cast<U128*>(&bs[at(e / VPR, e % VPR)]) = xb[i];
    }
  };
  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int fr = lane % 16, fk = lane / 16;
  auto frags = [&](const uint16_t* as, const uint16_t* bs, int s, U128 (&fa)[TM],
                   U128 (&fb)[TN]) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
      fa[i] = *reinterpret_cast<const U128*>(&as[at(wr * (BM / 2) + i * 16 + fr, s * 4 + fk)]);
#pragma unroll
    for (int j = 0; j < TN; ++j)
      fb[j] = *reinterpret_cast<const U128*>(&bs[at(wc * (BN / 2) + j * 16 + fr, s * 4 + fk)]);
  };
  auto mma = [&](const U128 (&fa)[TM], const U128 (&fb)[TN]) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        acc[i][j] = E::mma(fa[i], fb[j], acc[i][j]);
  };
  constexpr int kMm = TM * TN, kRd = TM + TN, kWr = AV + BV;
  static_assert(kMm >= kRd && (BK == 128 ? 2 * kMm >= kWr : kMm >= kWr),
                "MFMAs to interleave the memory instructions with");
  // A step whose stash and fetch both cover a whole slice: multiply (as, bs); write (xa, xb),
  // the next slice, into (na, nb); load slice k0f into (xa, xb) once written.
  auto wholeStep = [&](const uint16_t* as, const uint16_t* bs, U128 (&xa)[AV], U128 (&xb)[BV],
                       uint16_t* na, uint16_t* nb, int64_t k0f) {
    if constexpr (BK == 128) {
      // four 32-column sub-slices, fragments double-buffered in registers: each sub-slice's
      // reads go out during the MFMAs of the one before, the stash and the next loads during
      // the last two
      U128 fa[2][TM], fb[2][TN];
      frags(as, bs, 0, fa[0], fb[0]);
      frags(as, bs, 1, fa[1], fb[1]);
      mma(fa[0], fb[0]);
      frags(as, bs, 2, fa[0], fb[0]);
#pragma unroll
      for (int i = 0; i < kRd; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      }
      mma(fa[1], fb[1]);
      frags(as, bs, 3, fa[1], fb[1]);
#pragma unroll
      for (int i = 0; i < kRd; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 1);
      }
      stash(xa, xb, na, nb);
      fetchWhole(xa, xb, k0f);
      mma(fa[0], fb[0]);
      mma(fa[1], fb[1]);
#pragma unroll
      for (int i = 0; i < kWr / 2; ++i) {  // two LDS writes and two loads per MFMA
        __builtin_amdgcn_sched_group_barrier(0x200, 2, 2);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 2);
        __builtin_amdgcn_sched_group_barrier(0x020, 2, 2);
      }
      __syncthreads();
      return;
    }
    U128 fa0[TM], fb0[TN], fa1[TM], fb1[TN];
    frags(as, bs, 0, fa0, fb0);
    frags(as, bs, 1, fa1, fb1);
    mma(fa0, fb0);
#pragma unroll
    for (int i = 0; i < kRd; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one LDS read
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);  // two MFMAs
    }
    if constexpr (kMm > kRd) __builtin_amdgcn_sched_group_barrier(0x008, kMm - kRd, 0);
    stash(xa, xb, na, nb);
    fetchWhole(xa, xb, k0f);
    mma(fa1, fb1);
#pragma unroll
    for (int i = 0; i < kWr; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x200, 1, 1);  // one LDS write
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 1);  // two MFMAs
      __builtin_amdgcn_sched_group_barrier(0x020, 1, 1);  // one global load
    }
    if constexpr (kMm > kWr) __builtin_amdgcn_sched_group_barrier(0x008, kMm - kWr, 1);
    __syncthreads();
  };
  // step s of nk near the end: stash and fetch only what exists
  auto tailStep = [&](const uint16_t* as, const uint16_t* bs, U128 (&xa)[AV], U128 (&xb)[BV],
                      uint16_t* na, uint16_t* nb, int64_t s, int64_t nk) {
    U128 fa[TM], fb[TN];
#pragma unroll
    for (int sub = 0; sub < BK / 32; ++sub) {
      frags(as, bs, sub, fa, fb);
      mma(fa, fb);
    }
    if (s + 1 < nk) stash(xa, xb, na, nb);
    __syncthreads();
    if (s + 3 < nk) fetch(xa, xb, (s + 3) * BK);
  };
  // slice j lives in registers j % 2 and LDS buffer j % 2
  U128 ra0[AV], rb0[BV], ra1[AV], rb1[BV];
  fetch(ra0, rb0, 0);
  if (nk > 1) fetch(ra1, rb1, BK);
  stash(ra0, rb0, As0, Bs0);
  __syncthreads();
  if (nk > 2) fetch(ra0, rb0, 2 * BK);
  int64_t s = 0;
  for (; (s + 5) * BK <= whole; s += 2) {  // steps s, s + 1 fetch slices s + 3, s + 4: all whole
    wholeStep(As0, Bs0, ra1, rb1, As1, Bs1, (s + 3) * BK);
    wholeStep(As1, Bs1, ra0, rb0, As0, Bs0, (s + 4) * BK);
  }
  for (; s < nk; s += 2) {
    tailStep(As0, Bs0, ra1, rb1, As1, Bs1, s, nk);
    if (s + 1 < nk) tailStep(As1, Bs1, ra0, rb0, As0, Bs0, s + 1, nk);
  }
  // Epilogue through LDS (every step ended with a barrier, so the operand buffers are free): the
  // accumulators go to LDS as fp32, then each thread takes runs of 8 consecutive columns of a
  // row, so bias / residual loads and output stores are 16-byte vectors. Runs that cross the
  // right edge, and outputs the vector forms cannot address, go element by element through the
  // same arithmetic.
  float* const ct = reinterpret_cast<float*>(smem);
  constexpr int kNextGroup = kGroupBytes / 4;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        ct[grp * kNextGroup + (wr * (BM / 2) + i * 16 + fk * 4 + v) * CP + wc * (BN / 2) + j * 16 +
           fr] = acc[i][j][v];
  __syncthreads();
  auto sum = [&](int at) {
    float v = ct[at];
#pragma unroll
    for (int q = 1; q < G; ++q) v += ct[q * kNextGroup + at];
    return v;
  };
  const int te = threadIdx.x;
  const bool vec = epi.vectorOk();
  if constexpr (Epi::kPairs) {
    // [gate 16 | up 16] column groups: run h (0, 1) of group b pairs gate columns 32 b + 8 h ..
    // with up columns 32 b + 16 + 8 h ..
    constexpr int kRuns = BM * BN / 16;
    static_assert(BN % 32 == 0, "pair runs");
#pragma unroll
    for (int q = 0; q < (kRuns + kThreads - 1) / kThreads; ++q) {
      const int e = te + q * kThreads;
      if (kRuns % kThreads != 0 && e >= kRuns) break;
      const int row = e / (BN / 16), p = e % (BN / 16);
      const int cg = (p / 2) * 32 + (p % 2) * 8;
      const int64_t grow = r0 + row, gcol = c0 + cg;
      if (grow >= R) continue;
      float g[8], u[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        g[k] = sum(row * CP + cg + k);
        u[k] = sum(row * CP + cg + 16 + k);
      }
      if (vec && gcol + 24 <= Cn) {
        epi.pair8(grow, gcol, g, u);
      } else {
#pragma unroll
        for (int k = 0; k < 8; ++k)
          if (gcol + 16 + k < Cn) epi.pair(grow, gcol + k, g[k], u[k]);
      }
    }
  } else {
    // a thread's runs: rows row0 + q * kRowStep, all at column run c8. The
    // loads of every run go out before any result is stored: the compiler must assume a store
    // may alias a later run's input, so a load-compute-store loop per run waited for each load.
    constexpr int kRuns = BM * BN / 8, kPer = (kRuns + kThreads - 1) / kThreads;
    static_assert(kThreads % (BN / 8) == 0, "runs");
    const int c8 = (te % (BN / 8)) * 8, row0 = te / (BN / 8);
    constexpr int kRowStep = kThreads / (BN / 8);
    if (kRuns < kThreads && row0 >= BM) return;  // more threads than runs
    const int64_t gcol = c0 + c8;
    // (vector-only epilogues have Cn % 8 == 0: a run is inside the columns or past them)
    if (Epi::kVectorOnly ? gcol < Cn : vec && gcol + 8 <= Cn) {
      const auto cd = epi.column(gcol);
      typename Epi::Run rd[kPer];
#pragma unroll
      for (int q = 0; q < kPer; ++q) {
        const int64_t grow = r0 + row0 + q * kRowStep;
        if (grow < R) rd[q] = epi.fetch(grow, gcol);
      }
#pragma unroll
      for (int q = 0; q < kPer; ++q) {
        const int row = row0 + q * kRowStep;
        const int64_t grow = r0 + row;
        if (grow >= R) continue;
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = sum(row * CP + c8 + k);
        epi.vec8(grow, gcol, v, cd, rd[q]);
      }
    } else if constexpr (!Epi::kVectorOnly) {
#pragma unroll
      for (int q = 0; q < kPer; ++q) {
        const int row = row0 + q * kRowStep;
        const int64_t grow = r0 + row;
        if (grow >= R) continue;
#pragma unroll
        for (int k = 0; k < 8; ++k)
          if (gcol + k < Cn) epi(grow, gcol + k, sum(row * CP + c8 + k));
      }
    }
  }
}

// ---- epilogues ---------------------------------------------------------------------------------
// Scalar form epi(row, col, v) for any output; the bf16 GEMM also calls vec8(row, col, v[8]) (or
// pair8 for kPairs) for 8 consecutive columns when vectorOk(): the same arithmetic per element,
// with 16-byte loads and stores.

__device__ __forceinline__ bool aligned16(const void* p) {
  return (reinterpret_cast<uintptr_t>(p) & 15u) == 0;
}
// 8 bf16 of a 16-byte vector as floats
__device__ __forceinline__ void unpackBf16x8(const U128& w, float (&f)[8]) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    f[2 * k] = __uint_as_float(w[k] << 16);
    f[2 * k + 1] = __uint_as_float(w[k] & 0xFFFF0000u);
  }
}
__device__ __forceinline__ U128 packBf16x8(const float (&f)[8]) {
  return U128{packBf16x2(f[0], f[1]), packBf16x2(f[2], f[3]), packBf16x2(f[4], f[5]),
              packBf16x2(f[6], f[7])};
}

__device__ __forceinline__ void unpack16x8(const U128& w, float (&f)[8], bf16) {
  unpackBf16x8(w, f);
}
__device__ __forceinline__ void unpack16x8(const U128& w, float (&f)[8], f16) {
  const f16x8 h = __builtin_bit_cast(f16x8, w);
#pragma unroll
  for (int k = 0; k < 8; ++k) f[k] = static_cast<float>(h[k]);
}
__device__ __forceinline__ U128 pack16x8(const float (&f)[8], bf16) { return packBf16x8(f); }
__device__ __forceinline__ U128 pack16x8(const float (&f)[8], f16) {
  f16x8 h;
#pragma unroll
  for (int k = 0; k < 8; ++k) h[k] = static_cast<f16>(f[k]);
  return __builtin_bit_cast(U128, h);
}

__device__ __forceinline__ uint2 pack16x4(const float (&f)[4], bf16) {
  return uint2{packBf16x2(f[0], f[1]), packBf16x2(f[2], f[3])};
}
__device__ __forceinline__ uint2 pack16x4(const float (&f)[4], f16) {
  typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
  return __builtin_bit_cast(uint2, f16x4{static_cast<f16>(f[0]), static_cast<f16>(f[1]),
                                         static_cast<f16>(f[2]), static_cast<f16>(f[3])});
}

// out[row * ldo + col] = act(v + bias[col]) of 16-bit operands (T = bf16 or f16), the output type
// chosen at run time (one copy of the GEMM per kernel: two inlined copies, one per output type, took the kernel past 256
// registers)
template <typename T>
struct RowMajorOut16OrF32 {
  static constexpr bool kPairs = false;
  static constexpr bool kVectorOnly = false;
  void* out;
  const T* bias;
  int64_t ldo;
  int relu, out_f32;
  __device__ __forceinline__ void operator()(int64_t row, int64_t col, float v) const {
    if (bias != nullptr) v += ld(bias + col);
    if (relu) v = fmaxf(v, 0.f);
    if (out_f32)
      st(static_cast<float*>(out) + row * ldo + col, v);
    else
      st(static_cast<T*>(out) + row * ldo + col, v);
  }
  __device__ __forceinline__ bool vectorOk() const {
    return ldo % 8 == 0 && aligned16(out) && aligned16(bias);
  }
  struct Run {};
  __device__ __forceinline__ U128 column(int64_t col) const {
    return bias != nullptr ? gload16(bias + col) : zero16();
  }
  __device__ __forceinline__ Run fetch(int64_t, int64_t) const { return {}; }
  __device__ __forceinline__ void vec8(int64_t row, int64_t col, float (&v)[8], const U128& bw,
                                       const Run&) const {
    if (bias != nullptr) {
      float b[8];
      unpack16x8(bw, b, T{});
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] += b[k];
    }
    if (relu)
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = fmaxf(v[k], 0.f);
    if (out_f32) {
      float* o = static_cast<float*>(out) + row * ldo + col;
      *gp(reinterpret_cast<U128*>(o)) = U128{__float_as_uint(v[0]), __float_as_uint(v[1]),
                                             __float_as_uint(v[2]), __float_as_uint(v[3])};
      *gp(reinterpret_cast<U128*>(o + 4)) = U128{__float_as_uint(v[4]), __float_as_uint(v[5]),
                                                 __float_as_uint(v[6]), __float_as_uint(v[7])};
    } else {
      *gp(reinterpret_cast<U128*>(static_cast<T*>(out) + row * ldo + col)) = pack16x8(v, T{});
    }
  }
};

using RowMajorOutBf16OrF32 = RowMajorOut16OrF32<bf16>;

// out[row, col] = bf16(residual[row, col] + bf16(v + bias[col])): a linear whose output is
// added to the residual stream, rounded where the unfused graph rounds (linear, then add).
struct ResidualOut {
  static constexpr bool kPairs = false;
  static constexpr bool kVectorOnly = false;
  bf16* out;
  const bf16* residual;
  const bf16* bias;
  int64_t ldo;
  __device__ __forceinline__ void operator()(int64_t row, int64_t col, float v) const {
    if (bias != nullptr) v += ld(bias + col);
    const float o = Num<bf16>::round(v);
    st(out + row * ldo + col, ld(residual + row * ldo + col) + o);
  }
  __device__ __forceinline__ bool vectorOk() const {
    return ldo % 8 == 0 && aligned16(out) && aligned16(residual) && aligned16(bias);
  }
  using Run = U128;  // the residual run
  __device__ __forceinline__ U128 column(int64_t col) const {
    return bias != nullptr ? gload16(bias + col) : zero16();
  }
  __device__ __forceinline__ Run fetch(int64_t row, int64_t col) const {
    return gload16(residual + row * ldo + col);
  }
  __device__ __forceinline__ void vec8(int64_t row, int64_t col, float (&v)[8], const U128& bw,
                                       const Run& rw) const {
    if (bias != nullptr) {
      float b[8];
      unpackBf16x8(bw, b);
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] += b[k];
    }
    float r[8];
    unpackBf16x8(rw, r);
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = r[k] + Num<bf16>::round(v[k]);
    *gp(reinterpret_cast<U128*>(out + row * ldo + col)) = packBf16x8(v);
  }
};

// SwiGLU of a [gate 16 | up 16]-interleaved weight (the layout of the fused decode weights):
// C columns 32 b + j (gate) and 32 b + 16 + j (up) give act[row, 16 b + j] =
// bf16(bf16(silu(bf16(gate))) * bf16(up)), the rounding points of the unfused linear, silu and
// mul nodes.
struct SwiGluOut {
  static constexpr bool kPairs = true;
  static constexpr bool kVectorOnly = false;
  bf16* out;
  int64_t ffn;
  __device__ __forceinline__ void pair(int64_t row, int64_t col, float gate, float up) const {
    FP_EXACT;
    const float g = Num<bf16>::round(gate), u = Num<bf16>::round(up);
    const float sg = Num<bf16>::round(g / (1.0f + expf(-g)));
    st(out + row * ffn + (col / 32) * 16 + col % 16, sg * u);
  }
  __device__ __forceinline__ bool vectorOk() const { return ffn % 8 == 0 && aligned16(out); }
  // gate columns col .. col + 7 (col % 16 == 0 or 8) with up columns col + 16 .. col + 23
  __device__ __forceinline__ void pair8(int64_t row, int64_t col, const float (&gate)[8],
                                        const float (&up)[8]) const {
    FP_EXACT;
    float o[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float g = Num<bf16>::round(gate[k]), u = Num<bf16>::round(up[k]);
      const float sg = Num<bf16>::round(g / (1.0f + expf(-g)));
      o[k] = sg * u;
    }
    *gp(reinterpret_cast<U128*>(out + row * ffn + (col / 32) * 16 + col % 16)) = packBf16x8(o);
  }
};

// The q|k|v projection of a prefill prompt straight into attention's layout: C row = token
// (b, s) of [B, S], C column = (q | k | v, head, d) of the packed [q; k; v] weight. Each value is
// rounded as the linear node rounds it (bf16(v + bias)); q and k then get the interleaved RoPE of
// position start_pos + s, rounded as the rotary node rounds it (pairs (2p, 2p + 1), positions
// outside the table copied unchanged); results go to q [B, Hq, S, D], k and v [B, Hkv, S, D]
// (rotary/kernel.py:6-35, and the reshape + transpose nodes a prompt needs). Vector form only:
// the host requires D % 8 == 0 and 16-byte aligned pointers (cos/sin too), so every 8-column
// run lies in one head (or past the last column, where gemm16 skips it) and reads 16 bytes of each
// table row.
struct QkvHeadsOut {
  static constexpr bool kPairs = false;
  static constexpr bool kVectorOnly = true;
  bf16* q;
  bf16* k;
  bf16* v;
  const bf16* bias;
  const float* cosT;
  const float* sinT;
  int64_t seq, max_pos, start_pos;
  int q_heads, kv_heads, head_dim;
  __device__ __forceinline__ bool vectorOk() const { return true; }
  __device__ __forceinline__ void operator()(int64_t, int64_t, float) const {}
  // column-invariant part of a run: the bias and where the run goes
  struct Col {
    U128 bias;
    bf16* base;
    uint32_t heads, h, d;
  };
  struct Run {  // the table rows of the run's position
    U128 cs, sn;
  };
  __device__ __forceinline__ Col column(int64_t col) const {
    // 32-bit index arithmetic (the host bounds rows, columns and seq below 2^31)
    const uint32_t qw = static_cast<uint32_t>(q_heads * head_dim);
    const uint32_t kw = static_cast<uint32_t>(kv_heads * head_dim);
    const uint32_t cu = static_cast<uint32_t>(col);
    Col c;
    c.bias = gload16(bias + col);
    uint32_t rel;
    if (cu < qw) {
      c.base = q, rel = cu, c.heads = q_heads;
    } else if (cu < qw + kw) {
      c.base = k, rel = cu - qw, c.heads = kv_heads;
    } else {
      c.base = v, rel = cu - qw - kw, c.heads = kv_heads;
    }
    c.h = rel / static_cast<uint32_t>(head_dim);
    c.d = rel - c.h * static_cast<uint32_t>(head_dim);
    return c;
  }
  __device__ __forceinline__ int64_t position(int64_t row) const {
    return start_pos + static_cast<uint32_t>(row) % static_cast<uint32_t>(seq);
  }
  __device__ __forceinline__ Run fetch(int64_t row, int64_t col) const {
    // pairs d / 2 .. d / 2 + 3: 16 bytes of each table row (head_dim / 2 % 4 == 0); col is
    // recomputed into the head offset the way column() does
    const uint32_t hd = static_cast<uint32_t>(head_dim);
    const uint32_t qkw = static_cast<uint32_t>((q_heads + kv_heads) * head_dim);
    const int64_t pos = position(row);
    Run r{zero16(), zero16()};
    if (static_cast<uint32_t>(col) < qkw && pos >= 0 && pos < max_pos) {
      const int64_t at = pos * (head_dim / 2) + (static_cast<uint32_t>(col) % hd) / 2;
      r.cs = gload16(cosT + at);
      r.sn = gload16(sinT + at);
    }
    return r;
  }
  __device__ __forceinline__ void vec8(int64_t row, int64_t, float (&x)[8], const Col& c,
                                       const Run& r) const {
    FP_EXACT;
    float b8[8];
    unpackBf16x8(c.bias, b8);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = Num<bf16>::round(x[e] + b8[e]);
    const uint32_t ru = static_cast<uint32_t>(row), sq = static_cast<uint32_t>(seq);
    const uint32_t b = ru / sq, s = ru - b * sq;
    const int64_t pos = start_pos + s;
    if (c.base != v && pos >= 0 && pos < max_pos) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float cs = __uint_as_float(r.cs[j]), sn = __uint_as_float(r.sn[j]);
        const float x0 = x[2 * j], x1 = x[2 * j + 1];
        x[2 * j] = x0 * cs - x1 * sn;
        x[2 * j + 1] = x0 * sn + x1 * cs;
      }
    }
    const uint64_t off =
        (static_cast<uint64_t>(b * c.heads + c.h) * sq + s) * static_cast<uint32_t>(head_dim) + c.d;
    *gp(reinterpret_cast<U128*>(c.base + off)) = packBf16x8(x);
  }
};

}  // namespace

// Two workgroups per CU (the LDS of two fits) and at most 256 VGPRs a lane: the compiler then
// keeps the accumulators in VGPRs and gives the two register stages and both sub-slices'
// fragments room without spilling.
#define DK_BF16_OCCUPANCY __attribute__((amdgpu_waves_per_eu(2)))

// Names: _t64 and _t128 tiles, _t64_g2 with two K groups per workgroup (gemm16's G), _t64_stream
// with 128-wide slices and nontemporal weight loads (one row tile over a large weight).
#define DK_MFMA_LINEAR16(name, T, E, TILE, G, S)                                                  \
  extern "C" __global__ void __launch_bounds__(G* kGemmThreads) DK_BF16_OCCUPANCY               \
      name(const uint16_t* x, const uint16_t* w, const uint16_t* bias, void* out, int64_t M,    \
           int64_t N, int64_t K, int out_f32, int relu) {                                       \
    gemm16<TILE, TILE, S ? 128 : 64, S, E, G>(                                                            \
        x, w, M, N, K, K,                                                                       \
        RowMajorOut16OrF32<T>{out, reinterpret_cast<const T*>(bias), N, relu, out_f32});        \
  }

DK_MFMA_LINEAR16(mfma_linear_bf16_t64, bf16, Bf16, 64, 1, false)
DK_MFMA_LINEAR16(mfma_linear_bf16_t64_g2, bf16, Bf16, 64, 2, false)
DK_MFMA_LINEAR16(mfma_linear_bf16_t64_stream, bf16, Bf16, 64, 1, true)
DK_MFMA_LINEAR16(mfma_linear_bf16_t128, bf16, Bf16, 128, 1, false)
DK_MFMA_LINEAR16(mfma_linear_f16_t64, f16, F16, 64, 1, false)
DK_MFMA_LINEAR16(mfma_linear_f16_t64_g2, f16, F16, 64, 2, false)
DK_MFMA_LINEAR16(mfma_linear_f16_t64_stream, f16, F16, 64, 1, true)
DK_MFMA_LINEAR16(mfma_linear_f16_t128, f16, F16, 128, 1, false)

// bf16 linear + residual (bf16 out) and SwiGLU of an interleaved gate/up weight (N = 2 * ffn,
// ffn % 16 == 0): the ResidualOut and SwiGluOut epilogues above.
#define DK_MFMA_BF16_FUSED(SUFFIX, TILE, G, S)                                                  \
  extern "C" __global__ void __launch_bounds__(G* kGemmThreads) DK_BF16_OCCUPANCY               \
      mfma_linear_residual_bf16_##SUFFIX(                                                      \
      const uint16_t* x, const uint16_t* w, const uint16_t* bias, const uint16_t* residual,    \
      uint16_t* out, int64_t M, int64_t N, int64_t K) {                                        \
    gemm16<TILE, TILE, S ? 128 : 64, S, Bf16, G>(x, w, M, N, K, K,                                       \
                                       ResidualOut{reinterpret_cast<bf16*>(out),               \
                                                   reinterpret_cast<const bf16*>(residual),    \
                                                   reinterpret_cast<const bf16*>(bias), N});   \
  }                                                                                            \
  extern "C" __global__ void __launch_bounds__(G* kGemmThreads) DK_BF16_OCCUPANCY               \
      mfma_gate_up_silu_bf16_##SUFFIX(                                                         \
      const uint16_t* x, const uint16_t* w_gate_up, uint16_t* out, int64_t M, int64_t ffn,      \
      int64_t K) {                                                                             \
    gemm16<TILE, TILE, S ? 128 : 64, S, Bf16, G>(x, w_gate_up, M, 2 * ffn, K, K,                         \
                                       SwiGluOut{reinterpret_cast<bf16*>(out), ffn});           \
  }

DK_MFMA_BF16_FUSED(t64, 64, 1, false)
DK_MFMA_BF16_FUSED(t64_g2, 64, 2, false)
DK_MFMA_BF16_FUSED(t64_stream, 64, 1, true)
DK_MFMA_BF16_FUSED(t128, 128, 1, false)

// q|k|v projection + RoPE + head layout of a prefill prompt (QkvHeadsOut): x [B * S, K],
// w_qkv [(Hq + 2 Hkv) D, K], b_qkv [(Hq + 2 Hkv) D].
#define DK_MFMA_QKV_HEADS(SUFFIX, TILE, G, S)                                                      \
  extern "C" __global__ void __launch_bounds__(G* kGemmThreads) DK_BF16_OCCUPANCY              \
      mfma_qkv_heads_bf16_##SUFFIX(const uint16_t* x, const uint16_t* w_qkv, const uint16_t* b_qkv, \
                                const float* cos, const float* sin, int64_t max_pos,           \
                                uint16_t* q, uint16_t* k, uint16_t* v, int64_t M, int64_t K,   \
                                int64_t seq, int64_t start_pos, int q_heads, int kv_heads,     \
                                int head_dim) {                                                \
    const int64_t n = static_cast<int64_t>(q_heads + 2 * kv_heads) * head_dim;                 \
    gemm16<TILE, TILE, S ? 128 : 64, S, Bf16, G>(x, w_qkv, M, n, K, K,                                                     \
                     QkvHeadsOut{reinterpret_cast<bf16*>(q), reinterpret_cast<bf16*>(k),       \
                                 reinterpret_cast<bf16*>(v),                                   \
                                 reinterpret_cast<const bf16*>(b_qkv), cos, sin, seq, max_pos, \
                                 start_pos, q_heads, kv_heads, head_dim});                     \
  }

DK_MFMA_QKV_HEADS(t64, 64, 1, false)
DK_MFMA_QKV_HEADS(t64_g2, 64, 2, false)
DK_MFMA_QKV_HEADS(t64_stream, 64, 1, true)
DK_MFMA_QKV_HEADS(t128, 128, 1, false)

// bf16 linear with K split over grid.z (decode-sized m with few output tiles): part z covers
// columns [z * per, min(K, (z + 1) * per)) (per % 64 == 0) and writes its fp32 sums to
// part[z][M][N]; splitk_reduce_bf16 then adds the parts in z order.
extern "C" __global__ void __launch_bounds__(kGemmThreads) DK_BF16_OCCUPANCY
    mfma_linear_bf16_splitk_t64(const uint16_t* x, const uint16_t* w, float* part, int64_t M,
                                int64_t N, int64_t K, int64_t per) {
  const int64_t k0 = static_cast<int64_t>(blockIdx.z) * per;
  const int64_t len = K - k0 < per ? K - k0 : per;
  float* const out = part + static_cast<int64_t>(blockIdx.z) * M * N;
  gemm16<64, 64, 128, true>(x + k0, w + k0, M, N, len, K,
                              RowMajorOutBf16OrF32{out, nullptr, N, 0, 1});
}

// The same for more than 64 rows: several row tiles read each weight (cached loads).
#define DK_MFMA_SPLITK16(name, E, T)                                                            \
  extern "C" __global__ void __launch_bounds__(kGemmThreads) DK_BF16_OCCUPANCY                  \
      name(const uint16_t* x, const uint16_t* w, float* part, int64_t M, int64_t N, int64_t K,  \
           int64_t per) {                                                                       \
    const int64_t k0 = static_cast<int64_t>(blockIdx.z) * per;                                  \
    const int64_t len = K - k0 < per ? K - k0 : per;                                            \
    float* const out = part + static_cast<int64_t>(blockIdx.z) * M * N;                         \
    gemm16<64, 64, 64, false, E>(x + k0, w + k0, M, N, len, K,                                  \
                                 RowMajorOut16OrF32<T>{out, nullptr, N, 0, 1});                 \
  }
DK_MFMA_SPLITK16(mfma_linear_bf16_splitk_rows_t64, Bf16, bf16)
DK_MFMA_SPLITK16(mfma_linear_f16_splitk_rows_t64, F16, f16)

extern "C" __global__ void __launch_bounds__(kGemmThreads) DK_BF16_OCCUPANCY
    mfma_linear_f16_splitk_t64(const uint16_t* x, const uint16_t* w, float* part, int64_t M,
                               int64_t N, int64_t K, int64_t per) {
  const int64_t k0 = static_cast<int64_t>(blockIdx.z) * per;
  const int64_t len = K - k0 < per ? K - k0 : per;
  float* const out = part + static_cast<int64_t>(blockIdx.z) * M * N;
  gemm16<64, 64, 128, true, F16>(x + k0, w + k0, M, N, len, K,
                                 RowMajorOut16OrF32<f16>{out, nullptr, N, 0, 1});
}

// out[m, n] = T(v + bias[n]) (or fp32, optional ReLU), or with a residual T(residual[m, n] +
// T(v + bias[n])), v = the sum of the split parts in split order: the rounding points of
// RowMajorOut16OrF32 and ResidualOut. Four columns per thread where the rows allow it.
template <typename T>
__device__ __forceinline__ void splitkReduce16(const float* part, const T* bias, const T* residual,
                                               void* out, int64_t M, int64_t N, int splits,
                                               int out_f32, int relu) {
  const int64_t total = M * N;
  auto finish = [&](int64_t e, int64_t col, float v) {
    if (bias != nullptr) v += ld(bias + col);
    if (residual != nullptr) v = ld(residual + e) + Num<T>::round(v);
    return relu ? fmaxf(v, 0.f) : v;
  };
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  const int64_t first = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (N % 4 == 0 && aligned16(part) && aligned16(out)) {
    for (int64_t e = first * 4; e < total; e += stride * 4) {
      f32x4 v = *gp(reinterpret_cast<const f32x4*>(part + e));
#pragma unroll 4
      for (int z = 1; z < splits; ++z)
        v += *gp(reinterpret_cast<const f32x4*>(part + z * total + e));
      const int64_t col = e % N;
      float r[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) r[k] = finish(e + k, col + k, v[k]);
      if (out_f32) {
        *gp(reinterpret_cast<f32x4*>(static_cast<float*>(out) + e)) = f32x4{r[0], r[1], r[2], r[3]};
      } else {
        *gp(reinterpret_cast<uint2*>(static_cast<T*>(out) + e)) = pack16x4(r, T{});
      }
    }
    return;
  }
  for (int64_t e = first; e < total; e += stride) {
    float v = gp(part)[e];
    for (int z = 1; z < splits; ++z) v += gp(part)[z * total + e];
    v = finish(e, e % N, v);
    if (out_f32)
      st(static_cast<float*>(out) + e, v);
    else
      st(static_cast<T*>(out) + e, v);
  }
}
extern "C" __global__ void __launch_bounds__(256)
    splitk_reduce_bf16(const float* part, const bf16* bias, const bf16* residual, void* out,
                       int64_t M, int64_t N, int splits, int out_f32, int relu) {
  splitkReduce16(part, bias, residual, out, M, N, splits, out_f32, relu);
}
extern "C" __global__ void __launch_bounds__(256)
    splitk_reduce_f16(const float* part, const f16* bias, const f16* residual, void* out,
                      int64_t M, int64_t N, int splits, int out_f32, int relu) {
  splitkReduce16(part, bias, residual, out, M, N, splits, out_f32, relu);
}

// The split parts of the [q | k | v] projection of decode rows (one new token per row): each
// value is the sum of its parts in split order plus the bias, rounded to bf16 (the linear
// output); q and k columns are then rotated as interleaved pairs in fp32 and rounded again
// (rotary/kernel.py:6-35; no rotation at positions >= max_pos); q goes to q_out [M, Hq, D], k and
// v into the paged cache at the row's position (k_pool [block, Hkv, slot, D], v_pool [block, Hkv,
// D, slot]; rows whose position is negative or past the cache write nothing). The arithmetic is
// that of the qkv_rope_append decode kernels. One thread per (row, column pair): part reads and
// q / k stores are coalesced along the row.
extern "C" __global__ void __launch_bounds__(256)
    splitk_reduce_qkv_rope_append(const float* part, int splits, const uint16_t* bias,
                                  const float* cos_t, const float* sin_t, int64_t max_pos,
                                  const void* positions, int pos64, uint16_t* q_out,
                                  uint16_t* k_pool, uint16_t* v_pool, const int32_t* block_table,
                                  int64_t block_size, int64_t max_blocks, int M, int Hq, int Hkv,
                                  int D) {
  FP_EXACT;
  const int64_t N = static_cast<int64_t>(Hq + 2 * Hkv) * D;
  const int64_t pairs = N / 2;
  const int64_t total = static_cast<int64_t>(M) * pairs;
  const int64_t plane = static_cast<int64_t>(M) * N;
  const int64_t q_rows = static_cast<int64_t>(Hq) * D;
  const int64_t k_rows = static_cast<int64_t>(Hkv) * D;
  const int64_t capacity = max_blocks * block_size;
  for (int64_t e = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; e < total;
       e += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int m = static_cast<int>(e / pairs);
    const int64_t n = 2 * (e % pairs);
    const int64_t pos = loadIndex(positions, pos64, m);
    if (pos < 0) continue;
    const int64_t at = static_cast<int64_t>(m) * N + n;
    f32x2_t s = *gp(reinterpret_cast<const f32x2_t*>(part + at));
    for (int z = 1; z < splits; ++z) {
      const f32x2_t p = *gp(reinterpret_cast<const f32x2_t*>(part + z * plane + at));
      s.x += p.x;
      s.y += p.y;
    }
    if (bias != nullptr) {
      s.x += bf16ToFloat(gp(bias)[n]);
      s.y += bf16ToFloat(gp(bias)[n + 1]);
    }
    float v0 = Num<bf16>::round(s.x), v1 = Num<bf16>::round(s.y);
    const bool is_q = n < q_rows;
    const bool is_k = !is_q && n < q_rows + k_rows;
    const int64_t local = is_q ? n : (is_k ? n - q_rows : n - q_rows - k_rows);
    const int head = static_cast<int>(local / D);
    const int d = static_cast<int>(local % D);
    if ((is_q || is_k) && pos < max_pos) {
      const int64_t c = pos * (D / 2) + d / 2;
      const float cs = gp(cos_t)[c], sn = gp(sin_t)[c];
      const float r0 = v0 * cs - v1 * sn;
      const float r1 = v0 * sn + v1 * cs;
      v0 = r0;
      v1 = r1;
    }
    const uint32_t packed = packBf16x2(v0, v1);
    if (is_q) {
      *gp(reinterpret_cast<uint32_t*>(q_out + (static_cast<int64_t>(m) * Hq + head) * D + d)) =
          packed;
      continue;
    }
    if (pos >= capacity) continue;
    const int64_t blk = gp(block_table)[m * max_blocks + pos / block_size];
    const int64_t off = pos % block_size;
    if (is_k) {
      *gp(reinterpret_cast<uint32_t*>(k_pool + ((blk * Hkv + head) * block_size + off) * D + d)) =
          packed;
    } else {
      uint16_t* dst = v_pool + ((blk * Hkv + head) * D + d) * block_size + off;
      *gp(dst) = static_cast<uint16_t>(packed);
      *gp(dst + block_size) = static_cast<uint16_t>(packed >> 16);
    }
  }
}

// Split parts of a residual projection (o_proj, down_proj) of decode rows, then the RMSNorm that
// follows it: h = bf16(residual + bf16(sum of the parts in split order + bias)) (the values of
// splitk_reduce_bf16) and xn = bf16(h * rsqrt(mean(h^2) + eps) * norm_w)
// (rms_norm/kernel.py:6-14). One workgroup per row, h held in registers between the two; rows of
// N <= 4096 columns (N % 8 == 0), at most kMaxParts parts (2, 4 or 8: the kernel suffix). Every
// part of every chunk is requested before the first is added (the index of parts past `splits`
// is clamped and their sums discarded), so a row costs one memory round trip, not one per part,
// and the smallest kMaxParts that holds the parts keeps the surplus loads few.
constexpr int kResNormChunks = 2;
template <int kMaxParts>
__device__ __forceinline__ void splitkReduceResidualNorm(const float* part, int splits,
                                                         const uint16_t* bias,
                                                         const uint16_t* residual,
                                                         const uint16_t* norm_w, uint16_t* h_out,
                                                         uint16_t* xn_out, int M, int N,
                                                         float eps) {
  FP_EXACT;
  __shared__ float wave_sq[256 / kWave];
  const int m = blockIdx.x;
  const int chunks = N / 8;
  const int64_t plane = static_cast<int64_t>(M) * N;
  uint32_t h[kResNormChunks][4];
  float sq = 0.f;
#pragma unroll
  for (int c = 0; c < kResNormChunks; ++c) {
    const int i = threadIdx.x + c * 256;
    if (i >= chunks) break;
    const int64_t at = static_cast<int64_t>(m) * N + i * 8;
    f32x4 p[kMaxParts][2];
#pragma unroll
    for (int z = 0; z < kMaxParts; ++z) {
      const int64_t zz = z < splits ? z : splits - 1;
      p[z][0] = *gp(reinterpret_cast<const f32x4*>(part + zz * plane + at));
      p[z][1] = *gp(reinterpret_cast<const f32x4*>(part + zz * plane + at + 4));
    }
    const U128 r = gload16(residual + at);
    U128 b = U128{0u, 0u, 0u, 0u};
    if (bias != nullptr) b = gload16(bias + i * 8);
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = p[0][e / 4][e % 4];
#pragma unroll
    for (int z = 1; z < kMaxParts; ++z)
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = z < splits ? v[e] + p[z][e / 4][e % 4] : v[e];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float lo = v[2 * k], hi = v[2 * k + 1];
      if (bias != nullptr) {
        lo += __uint_as_float(b[k] << 16);
        hi += __uint_as_float(b[k] & 0xFFFF0000u);
      }
      lo = __uint_as_float(r[k] << 16) + Num<bf16>::round(lo);
      hi = __uint_as_float(r[k] & 0xFFFF0000u) + Num<bf16>::round(hi);
      h[c][k] = packBf16x2(lo, hi);
      const float hl = __uint_as_float(h[c][k] << 16), hh = __uint_as_float(h[c][k] & 0xFFFF0000u);
      sq += hl * hl;
      sq += hh * hh;
    }
    *gp(reinterpret_cast<U128*>(h_out + at)) = U128{h[c][0], h[c][1], h[c][2], h[c][3]};
  }
  sq = waveSum(sq);
  if (threadIdx.x % kWave == 0) wave_sq[threadIdx.x / kWave] = sq;
  __syncthreads();
  float total = 0.f;
#pragma unroll
  for (int w = 0; w < 256 / kWave; ++w) total += wave_sq[w];
  const float inv = 1.0f / sqrtf(total / static_cast<float>(N) + eps);
#pragma unroll
  for (int c = 0; c < kResNormChunks; ++c) {
    const int i = threadIdx.x + c * 256;
    if (i >= chunks) break;
    const U128 w = gload16(norm_w + i * 8);
    uint32_t o[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float hl = __uint_as_float(h[c][k] << 16), hh = __uint_as_float(h[c][k] & 0xFFFF0000u);
      o[k] = packBf16x2(hl * inv * __uint_as_float(w[k] << 16),
                        hh * inv * __uint_as_float(w[k] & 0xFFFF0000u));
    }
    *gp(reinterpret_cast<U128*>(xn_out + static_cast<int64_t>(m) * N + i * 8)) =
        U128{o[0], o[1], o[2], o[3]};
  }
}

#define DK_RESNORM(P)                                                                            \
  extern "C" __global__ void __launch_bounds__(256) splitk_reduce_residual_norm_p##P(           \
      const float* part, int splits, const uint16_t* bias, const uint16_t* residual,             \
      const uint16_t* norm_w, uint16_t* h_out, uint16_t* xn_out, int M, int N, float eps) {      \
    splitkReduceResidualNorm<P>(part, splits, bias, residual, norm_w, h_out, xn_out, M, N, eps); \
  }
DK_RESNORM(2)
DK_RESNORM(4)
DK_RESNORM(8)
