// fp32 MFMA GEMMs of the generic operators on gfx950.
//
//   C[r, c] = sum_k A(r, k) * B(c, k), then bias, ReLU and the output's layout
//
//  mfma_linear_f32_<g>   A = x [M, K], B = w [N, K] (linear/kernel.py:6-44)
//  mfma_matmul_f32_<g>   A = a [M, K], B = b [K, N] (matmul/kernel.py:6-40)
//  mfma_conv2d_f32_<g>   im2col-free conv2d (conv2d/kernel.py:6-49): A = weight [OC, C*KH*KW] rows,
//                        B = the input patch of each output pixel, gathered from NCHW x while
//                        staging (never materialised); out NCHW
//
// The products run on the bf16 matrix cores as sums of three terms (below), eight instructions at
// sixteen times the rate of the fp32 one, so a 64 x 64 tile is bound by staging as much as by the
// matrix cores (over 1000 x 4864 x 896: vector instructions 47%, LDS 32%, matrix cores 41% busy; at 4096^3
// the products run at 1140 TFLOP/s of bf16, near what a library product reaches): one tile size, fine enough that a few hundred tiles spread over 256 CUs. What overlaps
// loads, staging and products are three workgroups per CU or, when the tiles are few, G = 2 groups of
// 256 threads that share a tile's K (_g2). Each group stages 32-wide K slices through LDS buffers of
// its own, two slices in flight in registers, and the epilogue adds the groups' tiles in group order.
// grid.z > 1 splits K further into a workspace (part); splitk_reduce_f32 / conv_splitk_reduce_f32 add
// the parts in order. Every output is a fixed-order sum: results do not depend on timing.
//
// Measured in us, before (fp32 instruction, 4-byte loads) and now: linear 1000 x 4864 x 896 153 / 73,
// 1000 x 896 x 4864 132 / 76, 8192 x 4864 x 896 700 / 514, 4096^3 1297 / 965, 3 x 4096 x 16384 103 / 45;
// conv 384 x 4096 pixels x 1728 159 / 55 (with the sum of its parts), 256 x 6272 pixels x 2304 200 / 84.
//
//  _m16: 16 rows of A against 64 of B (a decode-sized x); _stream: nontemporal weight loads.
//  _scalar: rows that are not 16-byte aligned or K % 4 != 0 (4-byte loads); convs of windows or images
//        that the gather through a buffer does not hold.
#include <type_traits>

#include "common.h"
#include "gemm_tiles.h"
#include "skinny.h"

using namespace dk;

namespace {

constexpr int kBK = 32;            // K slice
constexpr int kChunks = kBK / 4;   // 4-wide chunks of a slice
constexpr int kPitch = kBK + 4;    // LDS row pitch of fp32 rows in floats

// ---- operand sources -------------------------------------------------------------------------
// A thread stages chunks (4 consecutive k of one row). begin() fixes its rows (rows past the end are
// clamped: their results are dropped), chunk<kWhole>(i, k0, tab) loads chunk i of the slice at k0,
// zeros past K; kWhole: the slice ends within K, and the loads are free of branches (a load behind a
// branch made every step wait for the loads it had just issued: 1900 instead of 1200 cycles a step).

// p[row * ld + k], lanes along k: chunk i = row t / 8 + 32 i, k 4 (t % 8)
template <int ROWS, bool kVec, bool kStream>
struct RowsK {
  static constexpr int kCount = ROWS * kChunks >= kGemmThreads ? ROWS * kChunks / kGemmThreads : 1;
  static constexpr bool kTable = false;
  const float* p;
  int64_t rows, K, ld;
  const float* at[kCount];
  int kc;
  __device__ __forceinline__ void begin(int64_t r0, int t) {
    kc = (t % kChunks) * 4;
#pragma unroll
    for (int i = 0; i < kCount; ++i) {
      const int64_t row = r0 + t / kChunks + i * (kGemmThreads / kChunks);
      at[i] = p + (row < rows ? row : rows - 1) * ld + kc;
    }
  }
  __device__ __forceinline__ static int row(int t, int i) {
    return t / kChunks + i * (kGemmThreads / kChunks);
  }
  __device__ __forceinline__ static int col(int t, int) { return (t % kChunks) * 4; }
  template <bool kWhole>
  __device__ __forceinline__ f32x4 chunk(int i, int64_t k0, const int2*) const {
    const float* q = at[i] + k0;
    if constexpr (kVec) {
      if (!kWhole && k0 + kc >= K) return f32x4{0.f, 0.f, 0.f, 0.f};
      if constexpr (kStream)
        return __builtin_nontemporal_load(gp(reinterpret_cast<const f32x4*>(q)));
      else
        return *gp(reinterpret_cast<const f32x4*>(q));
    } else {
      f32x4 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = kWhole || k0 + kc + j < K ? gp(q)[j] : 0.f;
      return v;
    }
  }
};

// lanes along rows: chunk i = row t % ROWS, k 4 (t / ROWS + (256 / ROWS) i)
template <int ROWS>
struct AlongRows {
  static constexpr int kCount = ROWS * kChunks / kGemmThreads;
  __device__ __forceinline__ static int row(int t, int) { return t % ROWS; }
  __device__ __forceinline__ static int col(int t, int i) {
    return 4 * (t / ROWS + i * (kGemmThreads / ROWS));
  }
};

// p[k * ld + row] (matmul's b [K, N])
template <int ROWS>
struct KRows : AlongRows<ROWS> {
  static constexpr bool kTable = false;
  const float* p;
  int64_t rows, K, ld;
  int64_t r;
  int t;
  __device__ __forceinline__ KRows(const float* p, int64_t rows, int64_t K, int64_t ld)
      : p(p), rows(rows), K(K), ld(ld) {}
  __device__ __forceinline__ void begin(int64_t r0, int t_) {
    t = t_;
    r = r0 + t % ROWS;
    if (r >= rows) r = rows - 1;
  }
  template <bool kWhole>
  __device__ __forceinline__ f32x4 chunk(int i, int64_t k0, const int2*) const {
    const int64_t k = k0 + this->col(t, i);
    f32x4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = kWhole || k + j < K ? gp(p)[(k + j) * ld + r] : 0.f;
    return v;
  }
};

// Input patch of a zero-padded NCHW conv: row = output pixel (n, oy, ox), k = (c, ky, kx) over
// k_base + [0, K). prepare() tabulates the k of a slice, and an element is a table read and one gather.
// 32-bit index math (the host checks that every index fits).
// kBuffer (KH * KW < 32, the images of a tile below 4 GB): the table holds (byte offset, ky * KW + kx)
// and the pixel a mask of the window positions outside the image; an element is one bit extract, an
// or that sends what is masked out of the buffer's range (which reads as 0) and a buffer load, 4
// vector instructions. Without it two range checks, two selects and 64-bit addresses, about 13: the
// convolutions are bound by vector instructions (57% of the CU cycles with these).
template <int ROWS, bool kBuffer>
struct ConvPatch : AlongRows<ROWS> {
  static constexpr bool kTable = true;
  const float* x;
  int rows, K, k_base, C, H, W, KH, KW, OH, OW, SH, SW, PH, PW;
  int iy0, ix0, base, t;
  unsigned outside;  // kBuffer: bit ky * KW + kx: that position lies outside; bit 31: past K
  bool valid;
  __amdgpu_buffer_rsrc_t images;
  __device__ __forceinline__ ConvPatch(const float* x, int rows, int K, int k_base, int C, int H,
                                       int W, int KH, int KW, int OH, int OW, int SH, int SW,
                                       int PH, int PW)
      : x(x), rows(rows), K(K), k_base(k_base), C(C), H(H), W(W), KH(KH), KW(KW), OH(OH), OW(OW),
        SH(SH), SW(SW), PH(PH), PW(PW) {}
  __device__ __forceinline__ void begin(int64_t r0, int t_) {
    t = t_;
    const int pixel = static_cast<int>(r0) + t % ROWS;
    valid = pixel < rows;
    const int ox = pixel % OW, q = pixel / OW;
    const int oy = q % OH;
    int n = q / OH;
    iy0 = oy * SH - PH;
    ix0 = ox * SW - PW;
    if constexpr (kBuffer) {
      // offsets from the tile's first image
      const int n0 = static_cast<int>(r0) / (OH * OW), last = (rows - 1) / (OH * OW);
      const int64_t chw = static_cast<int64_t>(C) * H * W;
      const int64_t bytes = (last + 1 - n0) * chw * 4;
      n -= n0;
      images = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<float*>(x + n0 * chw), 0,
          static_cast<int>(bytes < 0xFFFFFFFFll ? bytes : 0xFFFFFFFFll), 0x00027000);
      outside = 0x80000000u;
      for (int ky = 0, bit = 0; ky < KH; ++ky)
        for (int kx = 0; kx < KW; ++kx, ++bit) {
          const bool in = valid && static_cast<unsigned>(iy0 + ky) < static_cast<unsigned>(H) &&
                          static_cast<unsigned>(ix0 + kx) < static_cast<unsigned>(W);
          outside |= (in ? 0u : 1u) << bit;
        }
      base = static_cast<int>(static_cast<unsigned>(n * C * H * W + iy0 * W + ix0) * 4u);
    } else {
      base = n * C * H * W + iy0 * W + ix0;
    }
  }
  __device__ __forceinline__ void prepare(int64_t k0, int t, int2* tab) const {
    const int k = static_cast<int>(k0) + t;
    if (t < kBK) {
      const int kk = k_base + k, khw = KH * KW;
      const int c = kk / khw, rem = kk - c * khw;
      const int ky = rem / KW, kx = rem - ky * KW;
      const int at = (c * H + ky) * W + kx;
      if constexpr (kBuffer)
        tab[t] = k < K ? int2{static_cast<int>(static_cast<unsigned>(at) * 4u), rem} : int2{0, 31};
      else
        tab[t] = int2{k < K ? at : -1, (ky << 16) | kx};
    }
  }
  template <bool kWhole>
  __device__ __forceinline__ f32x4 chunk(int i, int64_t, const int2* tab) const {
    const int c0 = this->col(t, i);
    f32x4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int2 e = tab[c0 + j];
      if constexpr (kBuffer) {
        const int out = __builtin_amdgcn_sbfe(static_cast<int>(outside), e.y, 1);  // -1: masked
        const int off = static_cast<int>(static_cast<unsigned>(base) + static_cast<unsigned>(e.x));
        v[j] = __uint_as_float(
            __builtin_amdgcn_raw_buffer_load_b32(images, off | out, 0, 0));
      } else {
        const unsigned iy = iy0 + (static_cast<unsigned>(e.y) >> 16), ix = ix0 + (e.y & 0xFFFF);
        const bool in = valid && e.x >= 0 && iy < static_cast<unsigned>(H) &&
                        ix < static_cast<unsigned>(W);
        const float g = gp(x)[in ? base + e.x : 0];
        v[j] = in ? g : 0.f;
      }
    }
    return v;
  }
};

// ---- core ----------------------------------------------------------------------------------------
// The products run on the bf16 matrix cores, which are 16 times as fast as the fp32 ones: an fp32
// value is the exact sum of three bf16 terms, x = h + m + l (8 mantissa bits each, cut by
// truncation, so that h never overflows), and
//   x y = l m' + m l' + l h' + h l' + m m' + m h' + h m' + h h'  (+ l l', below 2^-30 x y, left out)
// is eight v_mfma_f32_16x16x32_bf16, h h' into one fp32 accumulator and the small products into another
// one: the large sum is then rounded once per 32 products (with one accumulator for all, as often as
// there are products, which showed: 3.9e-7 from float64 over the CNN against 2.2e-7 with the fp32
// instruction). The two smallest products reach 2^-21 x y and always have its sign; without them one
// product was off by up to 8 half-ulps (K = 1: 6.0e-8 in the 2-norm, 2.5e-8 with the fp32 instruction
// and with these two). Distance from float64 over random normal operands, the fp32 instruction / here:
// K = 4 3.9e-8 / 2.6e-8, K = 32 1.0e-7 / 3.9e-8, K = 256 2.8e-7 / 6.3e-8, K = 4864 3.2e-7 / 1.1e-7. They
// cost 12 to 14% where the matrix cores bind (4096^3 841 -> 968 us, 1272 with the fp32 instruction), 1 to
// 8% elsewhere.
// An infinity or NaN among the operands, or a sum past the fp32 range, makes a result of the tile
// non-finite; such a tile is computed again with the fp32 instruction, whose rules for them hold. So is
// a tile with operands below 2^-110, whose last bits lie below the smallest bf16 (2^-133): they are
// what is left in the lower half of the third term.
//
// Staging splits a chunk once for the waves that share it. LDS holds an operand's slice as planes of
// 16-byte runs (8 k of one term), one plane per term and run g of the 32 k, row r of a plane at
// r ^ mask(g): the 16 rows of a fragment read fall on the 16 4-bank groups, and so do the two rows of
// eight chunks that 16 lanes write (in rows of 208 bytes, conflicts were half of the LDS cycles, and
// LDS 73% of the kernel's).
constexpr int kRowBytes = 3 * kBK * 2;

// byte offset of row `row`, run g of term 0, in an operand of ROWS rows; term q is 64 ROWS q further
template <int ROWS>
__device__ __forceinline__ int runAt(int row, int g) {
  const int mask = ((g & 1) << 1) | ((g >> 1) * 12);
  return (g * ROWS + (row ^ mask)) * 16;
}

// lost: the or of the third terms, whose lower halves are what the bf16 terms drop (the upper halves:
// noise). The asm statements are empty: they keep the ors where the values are made. Gathered for all
// chunks at the end of a step, the ors held the values in registers and made 4096^3 6% slower, 500 x 896 x
// 4864 (_g2) 11%; like this 1% and 6%.
__device__ __forceinline__ void split3(const f32x4& v, uint2 (&t)[3], uint32_t& lost) {
  uint32_t h[4], m[4], l[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    h[k] = __float_as_uint(v[k]);
    const float r = v[k] - __uint_as_float(h[k] & 0xFFFF0000u);
    m[k] = __float_as_uint(r);
    l[k] = __float_as_uint(r - __uint_as_float(m[k] & 0xFFFF0000u));
  }
  auto pack = [](const uint32_t (&u)[4]) {  // the upper halves
    return uint2{__builtin_amdgcn_perm(u[1], u[0], 0x07060302u),
                 __builtin_amdgcn_perm(u[3], u[2], 0x07060302u)};
  };
  t[0] = pack(h), t[1] = pack(m), t[2] = pack(l);
  lost |= l[0] | l[1];
  asm("" : "+v"(lost));
  lost |= l[2] | l[3];
  asm("" : "+v"(lost));
}

// WR x WC: the 4 waves of a group over the tile.
template <int BM, int BN, int WR, int WC, int G, class ASrc, class BSrc, class Epi>
__device__ __forceinline__ void gemmF32(ASrc A, BSrc B, int64_t R, int64_t Cn, int64_t K,
                                        const Epi& epi) {
  constexpr int TM = BM / (16 * WR), TN = BN / (16 * WC);
  constexpr int CA = ASrc::kCount, CB = BSrc::kCount;
  // every thread stages chunks of A, of B
  constexpr bool kAllA = BM * kChunks >= kGemmThreads, kAllB = BN * kChunks >= kGemmThreads;
  constexpr int kStage = (BM + BN) * kRowBytes / 4;     // floats of one LDS buffer
  constexpr int CP = BN + 4;                            // pitch of the epilogue's tile
  constexpr int kGroupFloats = 2 * kStage > BM * CP ? 2 * kStage : BM * CP;
  __shared__ __attribute__((aligned(16))) float smem[G * kGroupFloats];
  __shared__ int2 ktab[BSrc::kTable ? G : 1][2][kBK];
  const int t = threadIdx.x % kGemmThreads, lane = t % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(t / kWave);
  const int grp = G == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / kGemmThreads);
  const int wr = wave / WC, wc = wave % WC;
  float* const buf = smem + grp * kGroupFloats;
  int64_t r0, c0;
  groupedTile(BM, BN, r0, c0);
  // the group's slices [first, first + nk); steps past K stage zeros
  const int slices = static_cast<int>((K + kBK - 1) / kBK), nk = (slices + G - 1) / G;
  const int64_t kg = static_cast<int64_t>(grp) * nk * kBK;
  // columns that every group has: the last group's
  const int64_t whole = K - static_cast<int64_t>(G - 1) * nk * kBK;
  // Step j of a group takes slice (j + rot) % nk, rot from the column tile, where every slice is whole
  // and the walk is long: with all workgroups at the same columns, rows that are a power of two apart
  // meet on the same memory channels. 16 rows only (_m16, a stream of weights). In us without / with, 3
  // rows: 4096 x 16384 62 / 45, 4096 x 32768 113 / 83, 8192 x 8192 62 / 47, 6000 x 12288 53 / 51; of 8
  // slices and less 1 to 4% slower.
  int rot = 0;
  if constexpr (G == 4)
    if (nk >= 16 && whole == static_cast<int64_t>(nk) * kBK)
      rot = static_cast<int>((blockIdx.x * 5u) & ((1u << (31 - __builtin_clz(nk))) - 1u));
  A.begin(r0, t);
  B.begin(c0, t);
  f32x4 acc[TM][TN], low[TM][TN];  // the products of the first terms; the others
  // what the bf16 terms drop (split3): one chain of ors per chunk where registers allow, so that none
  // waits for another chunk's load
  constexpr int kLostA = G == 1 ? 1 : CA, kLostB = G == 1 ? 1 : CB;
  uint32_t lost_a[kLostA] = {}, lost_b[kLostB] = {};
  const int fr = lane % 16, fk = lane / 16;

  // acc = the tile's products over the group's slices; exact: with the fp32 instruction
  auto run = [&](auto exact) {
    constexpr bool kExact = decltype(exact)::value;
    auto prepare = [&](int j) {
      if constexpr (BSrc::kTable)
        B.prepare(kg + static_cast<int64_t>(j) * kBK, t, ktab[grp][j & 1]);
    };
    auto fetch = [&](auto all, f32x4 (&ra)[CA], f32x4 (&rb)[CB], int j) {
      constexpr bool kWhole = decltype(all)::value;
      int at = j + rot;
      if (G == 4 && at >= nk) at -= nk;
      const int64_t k0 = kg + static_cast<int64_t>(at) * kBK;
      const int2* tab = nullptr;
      if constexpr (BSrc::kTable) tab = ktab[grp][j & 1];
      // (with fewer A chunks than threads, the spare threads load other rows and drop them)
#pragma unroll
      for (int i = 0; i < CA; ++i) ra[i] = A.template chunk<kWhole>(i, k0, tab);
#pragma unroll
      for (int i = 0; i < CB; ++i) rb[i] = B.template chunk<kWhole>(i, k0, tab);
    };
    auto put = [&](auto rows, float* base, int row, int col, const f32x4& v, uint32_t& lost) {
      if constexpr (kExact) {
        *reinterpret_cast<f32x4*>(&base[row * kPitch + col]) = v;
      } else {
        uint2 term[3];
        split3(v, term, lost);
        constexpr int kRows = decltype(rows)::value;
        char* const p = reinterpret_cast<char*>(base) + runAt<kRows>(row, col / 8) + (col & 4) * 2;
#pragma unroll
        for (int q = 0; q < 3; ++q) *reinterpret_cast<uint2*>(p + q * 64 * kRows) = term[q];
      }
    };
    auto stash = [&](const f32x4 (&ra)[CA], const f32x4 (&rb)[CB], int b) {
      float* const as = buf + b * kStage;
      float* const bs = as + BM * kRowBytes / 4;
      if (kAllA || t < BM * kChunks) {
#pragma unroll
        for (int i = 0; i < CA; ++i)
          put(std::integral_constant<int, BM>{}, as, ASrc::row(t, i), ASrc::col(t, i), ra[i],
              lost_a[i % kLostA]);
      }
      if (kAllB || t < BN * kChunks) {
#pragma unroll
        for (int i = 0; i < CB; ++i)
          put(std::integral_constant<int, BN>{}, bs, BSrc::row(t, i), BSrc::col(t, i), rb[i],
              lost_b[i % kLostB]);
      }
    };
    auto multiply = [&](int b) {
      const float* const as = buf + b * kStage;
      const float* const bs = as + BM * kRowBytes / 4;
      if constexpr (kExact) {
        // v_mfma_f32_16x16x4_f32: lane l supplies A[l % 16][kk] and B[kk][l % 16] for the step's k
        // index kk = l / 16 and receives D[(l / 16) * 4 + i][l % 16], i < 4; step s uses
        // k = 8 (l / 16) + s, so a lane's 8 values are two 16-byte reads
        f32x4 a4[TM][2], b4[TN][2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
          for (int i = 0; i < TM; ++i)
            a4[i][h] = *reinterpret_cast<const f32x4*>(
                &as[((wr * TM + i) * 16 + fr) * kPitch + fk * 8 + h * 4]);
#pragma unroll
          for (int j = 0; j < TN; ++j)
            b4[j][h] = *reinterpret_cast<const f32x4*>(
                &bs[((wc * TN + j) * 16 + fr) * kPitch + fk * 8 + h * 4]);
        }
#pragma unroll
        for (int s = 0; s < 8; ++s)
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                  a4[i][s / 4][s % 4], b4[j][s / 4][s % 4], acc[i][j], 0, 0, 0);
      } else {
        // v_mfma_f32_16x16x32_bf16: lane l supplies A[l % 16][(l / 16) * 8 + j], B alike, j < 8
        const char* const ap = reinterpret_cast<const char*>(as) + runAt<BM>(wr * TM * 16 + fr, fk);
        const char* const bp = reinterpret_cast<const char*>(bs) + runAt<BN>(wc * TN * 16 + fr, fk);
        U128 at[TM][3], bt[TN][3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
#pragma unroll
          for (int i = 0; i < TM; ++i)
            at[i][q] = *reinterpret_cast<const U128*>(ap + q * 64 * BM + i * 256);
#pragma unroll
          for (int j = 0; j < TN; ++j)
            bt[j][q] = *reinterpret_cast<const U128*>(bp + q * 64 * BN + j * 256);
        }
        constexpr int kTerms[7][2] = {{2, 1}, {1, 2}, {2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}};
#pragma unroll
        for (int q = 0; q < 7; ++q)
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
              low[i][j] = Bf16::mma(at[i][kTerms[q][0]], bt[j][kTerms[q][1]], low[i][j]);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = Bf16::mma(at[i][0], bt[j][0], acc[i][j]);
      }
    };
    // Step s multiplies LDS buffer s % 2, writes slice s + 1 (fetched a step ago) into the other one
    // and fetches slice s + 2; the table of slice s + 3 goes where slice s + 1's was.
    f32x4 ra0[CA], rb0[CB], ra1[CA], rb1[CB];
    auto step = [&](auto all, f32x4 (&fa)[CA], f32x4 (&fb)[CB], f32x4 (&na)[CA],
                    f32x4 (&nb)[CB], int s) {
      constexpr bool kWhole = decltype(all)::value;
      if (kWhole || s + 2 < nk) fetch(all, fa, fb, s + 2);
      // the loads stay ahead of the step's work (the compiler sank them to its end, where the next
      // step waited for them: 1700 cycles a step)
      __builtin_amdgcn_sched_barrier(0);
      multiply(s & 1);
      if (kWhole || s + 1 < nk) stash(na, nb, (s + 1) & 1);
      if (BSrc::kTable && s + 3 < nk) prepare(s + 3);
      __syncthreads();
    };
    const std::false_type tail;
    const std::true_type all;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = low[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    prepare(0);
    if (nk > 1) prepare(1);
    if (BSrc::kTable) __syncthreads();
    fetch(tail, ra0, rb0, 0);
    if (nk > 1) fetch(tail, ra1, rb1, 1);
    stash(ra0, rb0, 0);
    if (BSrc::kTable) __syncthreads();  // slice 0's table has been read by every wave
    if (nk > 2) prepare(2);
    __syncthreads();
    int s = 0;
    for (; (s + 4) * kBK <= whole; s += 2) {  // steps s and s + 1 fetch slices s + 2 and s + 3
      step(all, ra0, rb0, ra1, rb1, s);
      step(all, ra1, rb1, ra0, rb0, s + 1);
    }
    for (; s < nk; s += 2) {
      step(tail, ra0, rb0, ra1, rb1, s);
      if (s + 1 < nk) step(tail, ra1, rb1, ra0, rb0, s + 1);
    }
  };
  run(std::false_type{});
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] += low[i][j];
  bool bad = false;
#pragma unroll
  for (int i = 0; i < kLostA; ++i) bad = bad || (lost_a[i] & 0xFFFFu) != 0;
#pragma unroll
  for (int i = 0; i < kLostB; ++i) bad = bad || (lost_b[i] & 0xFFFFu) != 0;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        bad = bad || (__float_as_uint(acc[i][j][v]) & 0x7F800000u) == 0x7F800000u;
  if (__syncthreads_or(bad)) run(std::true_type{});
  // epilogue through LDS (every step ended with a barrier): the groups' tiles, then each thread
  // adds runs of 4 columns
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        buf[((wr * TM + i) * 16 + fk * 4 + v) * CP + (wc * TN + j) * 16 + fr] = acc[i][j][v];
  __syncthreads();
  constexpr int kRuns = BM * BN / 4, kThreads = G * kGemmThreads;
#pragma unroll
  for (int q = 0; q < (kRuns + kThreads - 1) / kThreads; ++q) {
    const int e = static_cast<int>(threadIdx.x) + q * kThreads;
    if (kRuns % kThreads != 0 && e >= kRuns) break;
    const int row = e / (BN / 4), c = (e % (BN / 4)) * 4;
    if (r0 + row >= R || c0 + c >= Cn) continue;
    f32x4 v = *reinterpret_cast<const f32x4*>(&smem[row * CP + c]);
#pragma unroll
    for (int p = 1; p < G; ++p)
      v += *reinterpret_cast<const f32x4*>(&smem[p * kGroupFloats + row * CP + c]);
    epi(r0 + row, c0 + c, v, Cn - (c0 + c) < 4 ? static_cast<int>(Cn - (c0 + c)) : 4);
  }
}

// ---- epilogues: n <= 4 consecutive columns of a row ----------------------------------------------

__device__ __forceinline__ bool aligned16(const void* p) {
  return (reinterpret_cast<uintptr_t>(p) & 15u) == 0;
}

// out[row * ldo + col] = act(v + bias[col])
struct RowMajorOut {
  float* out;
  const float* bias;
  int64_t ldo;
  int relu;
  __device__ __forceinline__ void operator()(int64_t row, int64_t col, f32x4 v, int n) const {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (bias != nullptr && k < n) v[k] += gp(bias)[col + k];
      if (relu) v[k] = fmaxf(v[k], 0.f);
    }
    float* const o = out + row * ldo + col;
    if (n == 4 && aligned16(o)) {
      *gp(reinterpret_cast<f32x4*>(o)) = v;
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (k < n) gp(o)[k] = v[k];
    }
  }
};

// out[n, oc, oy, ox] = act(v + bias[oc]) for C row oc and C column pixel (n, oy, ox)
struct ConvOut {
  float* out;
  const float* bias;
  int OC, OHW;
  int relu;
  __device__ __forceinline__ void operator()(int64_t oc, int64_t pixel, f32x4 v, int n) const {
    const float b = bias != nullptr ? gp(bias)[oc] : 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (bias != nullptr) v[k] += b;
      if (relu) v[k] = fmaxf(v[k], 0.f);
    }
    const int px = static_cast<int>(pixel), img = px / OHW, p = px - img * OHW;
    float* const o = out + (static_cast<int64_t>(img) * OC + oc) * OHW + p;
    if (n == 4 && p + 4 <= OHW && aligned16(o)) {
      *gp(reinterpret_cast<f32x4*>(o)) = v;
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (k < n) {
          const int pk = px + k, ik = pk / OHW;
          gp(out)[(static_cast<int64_t>(ik) * OC + oc) * OHW + (pk - ik * OHW)] = v[k];
        }
    }
  }
};

}  // namespace

#define DK_F32_OCCUPANCY __attribute__((amdgpu_waves_per_eu(2)))

// K range of this workgroup's part (grid.z parts of `per` columns, per % 32 == 0) and where its
// result goes: the output, or part z of the workspace
#define DK_PART(K)                                                              \
  const int64_t kb = static_cast<int64_t>(blockIdx.z) * per;                    \
  const int64_t kl = (K) - kb < per ? (K) - kb : per;                           \
  const bool whole = gridDim.z == 1;

#define DK_LINEAR(name, BM, BN, WR, WC, G, VEC, STREAM)                                         \
  extern "C" __global__ void __launch_bounds__(G* kGemmThreads) DK_F32_OCCUPANCY                                \
      name(const float* x, const float* w, const float* bias, float* out, float* part,          \
           int64_t M, int64_t N, int64_t K, int64_t per, int relu) {                            \
    DK_PART(K)                                                                                  \
    gemmF32<BM, BN, WR, WC, G>(                                                                 \
        RowsK<BM, VEC, false>{x + kb, M, kl, K}, RowsK<BN, VEC, STREAM>{w + kb, N, kl, K}, M, N, \
        kl,                                                                                     \
        RowMajorOut{whole ? out : part + static_cast<int64_t>(blockIdx.z) * M * N,              \
                    whole ? bias : nullptr, N, whole ? relu : 0});                              \
  }
DK_LINEAR(mfma_linear_f32_g1, 64, 64, 2, 2, 1, true, false)
DK_LINEAR(mfma_linear_f32_g2, 64, 64, 2, 2, 2, true, false)
DK_LINEAR(mfma_linear_f32_stream, 64, 64, 2, 2, 2, true, true)
DK_LINEAR(mfma_linear_f32_m16, 16, 64, 1, 4, 4, true, true)
DK_LINEAR(mfma_linear_f32_scalar, 64, 64, 2, 2, 1, false, false)

#define DK_MATMUL(name, G, VEC)                                                                 \
  extern "C" __global__ void __launch_bounds__(G* kGemmThreads) DK_F32_OCCUPANCY                                \
      name(const float* a, const float* b, float* out, int64_t M, int64_t N, int64_t K) {       \
    gemmF32<64, 64, 2, 2, G>(RowsK<64, VEC, false>{a, M, K, K}, KRows<64>(b, N, K, N), M, N, K, \
                             RowMajorOut{out, nullptr, N, 0});                                  \
  }
DK_MATMUL(mfma_matmul_f32_g1, 1, true)
DK_MATMUL(mfma_matmul_f32_g2, 2, true)
DK_MATMUL(mfma_matmul_f32_scalar, 1, false)

#define DK_CONV(name, G, VEC)                                                                   \
  extern "C" __global__ void __launch_bounds__(G* kGemmThreads) DK_F32_OCCUPANCY                                \
      name(const float* x, const float* weight, const float* bias, float* out, float* part,     \
           int N, int C, int H, int W, int OC, int KH, int KW, int OH, int OW, int SH, int SW,  \
           int PH, int PW, int per, int relu) {                                                 \
    const int64_t K = C * KH * KW;                                                              \
    const int pixels = N * OH * OW;                                                             \
    DK_PART(K)                                                                                  \
    const RowsK<64, VEC, false> A{weight + kb, OC, kl, K};                                      \
    const ConvPatch<64, VEC> B(x, pixels, static_cast<int>(kl), static_cast<int>(kb), C, H, W, KH,   \
                          KW, OH, OW, SH, SW, PH, PW);                                          \
    const RowMajorOut parts{part + static_cast<int64_t>(blockIdx.z) * OC * pixels, nullptr,     \
                            pixels, 0};                                                         \
    const ConvOut final{out, bias, OC, OH * OW, relu};                                          \
    gemmF32<64, 64, 2, 2, G>(A, B, OC, pixels, kl,                                              \
                             [&](int64_t r, int64_t c, f32x4 v, int n) {                        \
                               if (whole)                                                       \
                                 final(r, c, v, n);                                             \
                               else                                                             \
                                 parts(r, c, v, n);                                             \
                             });                                                                \
  }
DK_CONV(mfma_conv2d_f32_g1, 1, true)
DK_CONV(mfma_conv2d_f32_g2, 2, true)
DK_CONV(mfma_conv2d_f32_scalar, 1, false)

// out[m, n] = act(sum of the parts in order + bias[n]); four columns per thread where the rows allow
extern "C" __global__ void __launch_bounds__(kGemmThreads)
    splitk_reduce_f32(const float* part, const float* bias, float* out, int64_t M, int64_t N,
                      int splits, int relu) {
  const int64_t total = M * N, stride = static_cast<int64_t>(gridDim.x) * kGemmThreads;
  const int64_t first = static_cast<int64_t>(blockIdx.x) * kGemmThreads + threadIdx.x;
  const RowMajorOut store{out, bias, N, relu};
  if (total % 4 == 0 && aligned16(part)) {
    for (int64_t e = first * 4; e < total; e += stride * 4) {
      f32x4 v = *gp(reinterpret_cast<const f32x4*>(part + e));
#pragma unroll 4
      for (int z = 1; z < splits; ++z)
        v += *gp(reinterpret_cast<const f32x4*>(part + z * total + e));
      if (N % 4 == 0) {
        store(e / N, e % N, v, 4);
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k)
          store((e + k) / N, (e + k) % N, f32x4{v[k], 0.f, 0.f, 0.f}, 1);
      }
    }
    return;
  }
  for (int64_t e = first; e < total; e += stride) {
    f32x4 v{gp(part)[e], 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int z = 1; z < splits; ++z) v[0] += gp(part)[z * total + e];
    store(e / N, e % N, v, 1);
  }
}

// The same for parts [OC][pixels] of a conv, out NCHW.
extern "C" __global__ void __launch_bounds__(kGemmThreads)
    conv_splitk_reduce_f32(const float* part, const float* bias, float* out, int64_t OC,
                           int64_t pixels, int64_t OHW, int splits, int relu) {
  const int64_t total = OC * pixels, stride = static_cast<int64_t>(gridDim.x) * kGemmThreads;
  const int64_t first = static_cast<int64_t>(blockIdx.x) * kGemmThreads + threadIdx.x;
  const ConvOut store{out, bias, static_cast<int>(OC), static_cast<int>(OHW), relu};
  if (pixels % 4 == 0 && aligned16(part)) {
    for (int64_t e = first * 4; e < total; e += stride * 4) {
      f32x4 v = *gp(reinterpret_cast<const f32x4*>(part + e));
#pragma unroll 4
      for (int z = 1; z < splits; ++z)
        v += *gp(reinterpret_cast<const f32x4*>(part + z * total + e));
      store(e / pixels, e % pixels, v, 4);
    }
    return;
  }
  for (int64_t e = first; e < total; e += stride) {
    f32x4 v{gp(part)[e], 0.f, 0.f, 0.f};
    for (int z = 1; z < splits; ++z) v[0] += gp(part)[z * total + e];
    store(e / pixels, e % pixels, v, 1);
  }
}
