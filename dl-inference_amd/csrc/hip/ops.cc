// Kernel entry points of libdli_hip.so (declared in include/dli_hip.h): argument checks,
// launch geometry, and the launch of the matching embedded gfx950 kernel.
#include <cmath>
#include <string>

#include "../kernels/conv_small.h"
#include "../kernels/packed_attention.h"
#include "runtime.h"

namespace dli::hip {
namespace {

// The three float variants of one kernel in one code object.
struct FloatKernels {
  DeviceKernel f32, bf16, f16;
  FloatKernels(const char* module, const char* base)
      : f32(module, intern(base, "_f32")), bf16(module, intern(base, "_bf16")),
        f16(module, intern(base, "_f16")) {}

  DeviceKernel* pick(int dtype) {
    switch (dtype) {
      case DLI_F32: return &f32;
      case DLI_BF16: return &bf16;
      case DLI_F16: return &f16;
      default: return nullptr;
    }
  }

 private:
  static const char* intern(const char* base, const char* suffix) {
    return (new std::string(std::string(base) + suffix))->c_str();  // lives for the process
  }
};

int badDtype(const char* op, int dtype) {
  return fail(DLI_HIP_EINVAL, std::string(op) + ": unsupported dtype code " + std::to_string(dtype));
}

int badArg(const char* op, const char* what) {
  return fail(DLI_HIP_EINVAL, std::string(op) + ": " + what);
}

bool validIndexDtype(int dtype) { return dtype == DLI_I64 || dtype == DLI_I32; }

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Grid-stride launches: enough blocks to fill 256 CUs several times over, capped.
unsigned strideBlocks(int64_t work) {
  const int64_t blocks = (work + 255) / 256;
  return static_cast<unsigned>(blocks < 4096 ? (blocks > 0 ? blocks : 1) : 4096);
}

FloatKernels k_add("elementwise", "add");
FloatKernels k_mul("elementwise", "mul");
FloatKernels k_silu("elementwise", "silu");
FloatKernels k_relu("elementwise", "relu");
FloatKernels k_add16("elementwise", "add16");
FloatKernels k_mul16("elementwise", "mul16");
FloatKernels k_silu16("elementwise", "silu16");
FloatKernels k_relu16("elementwise", "relu16");
FloatKernels k_rotary16("elementwise", "rotary16");
FloatKernels k_bn("elementwise", "batch_norm2d");
FloatKernels k_maxpool("elementwise", "max_pool2d");
FloatKernels k_embedding("elementwise", "embedding");
FloatKernels k_softmax("elementwise", "softmax");
FloatKernels k_transpose("elementwise", "transpose2d");
DeviceKernel k_permute16("elementwise", "permute_0213_u128");
DeviceKernel k_permute2("elementwise", "permute_0213_u16");
FloatKernels k_rotary("elementwise", "rotary");
FloatKernels k_argmax("elementwise", "argmax");
DeviceKernel k_argmax_rows_v4("elementwise", "argmax_f32_rows_v4");
FloatKernels k_rms_norm("norm", "rms_norm");
DeviceKernel k_rms_norm_rows("norm", "rms_norm_rows_bf16_k");
DeviceKernel k_rms_norm_mid_rows("norm", "rms_norm_mid_rows_bf16_k");
DeviceKernel k_rms_norm_wide_rows("norm", "rms_norm_wide_rows_bf16_k");
DeviceKernel k_kv_append_tiles("attention", "kv_append_tiles_bf16_k");
FloatKernels k_gemm("gemm", "gemm_tiled");
// [16 waves][16 MB rows: MB = 1, 2, 4]
DeviceKernel k_skinny_bf16[2][3] = {{{"gemm", "skinny_linear_bf16_m1"},
                                     {"gemm", "skinny_linear_bf16_m2"},
                                     {"gemm", "skinny_linear_bf16_m4"}},
                                    {{"gemm", "skinny_linear_bf16_w16_m1"},
                                     {"gemm", "skinny_linear_bf16_w16_m2"},
                                     {"gemm", "skinny_linear_bf16_w16_m4"}}};
DeviceKernel k_skinny_f16[2][3] = {{{"gemm", "skinny_linear_f16_m1"},
                                    {"gemm", "skinny_linear_f16_m2"},
                                    {"gemm", "skinny_linear_f16_m4"}},
                                   {{"gemm", "skinny_linear_f16_w16_m1"},
                                    {"gemm", "skinny_linear_f16_w16_m2"},
                                    {"gemm", "skinny_linear_f16_w16_m4"}}};
FloatKernels k_attention("attention", "attention");
FloatKernels k_paged_attention("attention", "paged_attention");
FloatKernels k_kv_append("attention", "kv_append");
FloatKernels k_conv2d("conv", "conv2d");
DeviceKernel k_flash_attention("flash_attention", "flash_attention_bf16");
DeviceKernel k_flash_attention_q32("flash_attention", "flash_attention_bf16_q32");
DeviceKernel k_packed_paged64("packed_attention", "packed_attention_paged_d64");
DeviceKernel k_packed_paged64_r128("packed_attention", "packed_attention_paged_d64_r128");
DeviceKernel k_packed_paged128("packed_attention", "packed_attention_paged_d128");
DeviceKernel k_packed_paged128_r128("packed_attention", "packed_attention_paged_d128_r128");
DeviceKernel k_packed_dense128("packed_attention", "packed_attention_dense_d128");
DeviceKernel k_packed_dense128_r128("packed_attention", "packed_attention_dense_d128_r128");
DeviceKernel k_packed_f32_64("packed_attention", "packed_attention_f32_d64");
DeviceKernel k_packed_f32_128("packed_attention", "packed_attention_f32_d128");
DeviceKernel k_packed_merge64("packed_attention", "packed_attention_merge_d64");
DeviceKernel k_packed_merge128("packed_attention", "packed_attention_merge_d128");
DeviceKernel k_conv_small9("conv", "conv2d_small_f32_p9");
DeviceKernel k_conv_small27("conv", "conv2d_small_f32_p27");
// [tile form: TileForm16]
DeviceKernel k_mfma_bf16[4] = {{"mfma_gemm", "mfma_linear_bf16_t64"},
                               {"mfma_gemm", "mfma_linear_bf16_t64_g2"},
                               {"mfma_gemm", "mfma_linear_bf16_t64_stream"},
                               {"mfma_gemm", "mfma_linear_bf16_t128"}};
DeviceKernel k_mfma_f16[4] = {{"mfma_gemm", "mfma_linear_f16_t64"},
                              {"mfma_gemm", "mfma_linear_f16_t64_g2"},
                              {"mfma_gemm", "mfma_linear_f16_t64_stream"},
                              {"mfma_gemm", "mfma_linear_f16_t128"}};
DeviceKernel k_mfma_linres[4] = {{"mfma_gemm", "mfma_linear_residual_bf16_t64"},
                                 {"mfma_gemm", "mfma_linear_residual_bf16_t64_g2"},
                                 {"mfma_gemm", "mfma_linear_residual_bf16_t64_stream"},
                                 {"mfma_gemm", "mfma_linear_residual_bf16_t128"}};
DeviceKernel k_mfma_bf16_splitk("mfma_gemm", "mfma_linear_bf16_splitk_t64");
DeviceKernel k_mfma_bf16_rows("mfma_gemm", "mfma_linear_bf16_splitk_rows_t64");
DeviceKernel k_splitk_reduce_bf16("mfma_gemm", "splitk_reduce_bf16");
DeviceKernel k_mfma_f16_splitk("mfma_gemm", "mfma_linear_f16_splitk_t64");
DeviceKernel k_mfma_f16_rows("mfma_gemm", "mfma_linear_f16_splitk_rows_t64");
DeviceKernel k_splitk_reduce_f16("mfma_gemm", "splitk_reduce_f16");
// fp32 GEMMs by K groups per workgroup (FormF32)
constexpr const char* kF32 = "mfma_gemm_f32";
DeviceKernel k_f32_linear[5] = {{kF32, "mfma_linear_f32_g1"},
                                {kF32, "mfma_linear_f32_g2"},
                                {kF32, "mfma_linear_f32_scalar"},
                                {kF32, "mfma_linear_f32_stream"},
                                {kF32, "mfma_linear_f32_m16"}};
DeviceKernel k_f32_matmul[3] = {{kF32, "mfma_matmul_f32_g1"},
                                {kF32, "mfma_matmul_f32_g2"},
                                {kF32, "mfma_matmul_f32_scalar"}};
DeviceKernel k_f32_conv[3] = {{kF32, "mfma_conv2d_f32_g1"},
                              {kF32, "mfma_conv2d_f32_g2"},
                              {kF32, "mfma_conv2d_f32_scalar"}};
DeviceKernel k_splitk_reduce(kF32, "splitk_reduce_f32");
DeviceKernel k_conv_splitk_reduce(kF32, "conv_splitk_reduce_f32");

// Form of an fp32 GEMM (mfma_gemm_f32.hip): kernel index, threads, K parts of `per` columns.
enum FormF32 { kG1 = 0, kG2 = 1, kScalar = 2, kStream = 3, kM16 = 4 };
struct PlanF32 {
  int form;
  unsigned threads;
  int64_t tile_rows, parts, per;
};
// `vec`: rows of 16-byte chunks (K % 4 == 0, aligned); `linear`: the forms of a few rows exist; at
// most max_parts parts.
//
// Three workgroups of one K group (_g1) fit a CU and overlap each other's loads, staging and matrix
// instructions; where the tiles alone are fewer, K parts make up for it, or, where the parts' traffic
// would cost more, a second K group in the workgroup. In us, parts with their sum: conv 384 x 4096 pixels
// x 1728 (384 tiles) 65 in one part, 55 in two; 256 x 4096 x 3456 (256 tiles) 73 with two groups, 69 in
// three parts of one; linear 1000 x 896 x 4864 (224 tiles) 76 with two groups, 97 with one, 79 in parts;
// 1000 x 896 x 896 17 with two groups, 21 with one, 24 in parts; convs of 3 images (12 to 24 tiles) are
// even: 13.5 with two groups and 12.8 with one for 384 x 192 x 1728, 15.4 either way for 256 x 192 x 3456.
constexpr int64_t kMaxPartsF32 = 16;
PlanF32 planF32(int64_t rows, int64_t cols, int64_t k, bool vec, bool linear, int64_t max_parts) {
  PlanF32 p{kG1, 256, 64, 1, k};
  const int64_t tiles = ((rows + 63) / 64) * ((cols + 63) / 64);
  const int64_t slices = (k + 31) / 32;
  const bool many = !linear && tiles >= 128 && vec;  // parts of one group
  int groups = 1;
  if (!vec) {
    p.form = kScalar;
  } else if (slices <= 1) {
    // one slice is one group's: the others would only add their start (K = 16 in us, several groups /
    // one: linear 16 x 16 4.7 / 3.7, 64 x 1000 4.9 / 4.5; matmul 64 x 1000 4.8 / 4.3)
  } else if (linear && rows <= 16) {
    p.form = kM16, p.tile_rows = 16, groups = 4;
  } else if (linear && rows <= 64) {
    p.form = kStream, groups = 2;
  } else if (tiles <= 256 && !many) {
    p.form = kG2, groups = 2;
  }
  p.threads = 256u * groups;
  // at least two slices per group (six where a workgroup has one)
  int64_t s = (many ? 768 : 256) / tiles;
  const int64_t least = many ? 6 : 2 * groups;
  if (s > slices / least) s = slices / least;
  if (s > max_parts) s = max_parts;
  if (s > 1) {
    p.per = (slices + s - 1) / s * 32;
    p.parts = (k + p.per - 1) / p.per;
  } else if (many && tiles <= 256 && slices > 1) {
    p.form = kG2, p.threads = 512;
  }
  return p;
}
// A conv on the 16-byte / buffer forms: whole 4-wide chunks of weight rows, a window of less than 32
// positions (bits of a mask), and the images under a tile's 64 pixels within a buffer's 4 GB.
bool convVec(int64_t n, int64_t c, int64_t h, int64_t w, int64_t patch, int64_t window,
             int64_t out_pixels) {
  int64_t images = 63 / out_pixels + 2;
  if (images > n) images = n;
  return patch % 4 == 0 && window < 32 && images * c * h * w < (int64_t{1} << 30);
}

// parts that a workspace holds
int64_t partsHeldF32(const void* workspace, size_t bytes, int64_t rows, int64_t cols) {
  const auto held = static_cast<int64_t>(bytes / sizeof(float)) / (rows * cols);
  return workspace == nullptr || held < 1 ? 1 : (held < kMaxPartsF32 ? held : kMaxPartsF32);
}
size_t partBytesF32(const PlanF32& p, int64_t rows, int64_t cols) {
  return p.parts > 1 ? static_cast<size_t>(p.parts * rows * cols) * sizeof(float) : 0;
}

constexpr int64_t kMaxGridY = 65535;

// fp32 linear and matmul: 64-row tiles in grid.y, in two launches past what that holds (the rows of the
// 128-row tiles that these calls had).
constexpr int64_t kGridRowsF32 = 64 * kMaxGridY, kMaxRowsF32 = 2 * kGridRowsF32;
template <class Launch>
int byRowsF32(const void* x, void* out, int64_t m, int64_t n, int64_t k, const Launch& go) {
  for (int64_t r = 0; r < m; r += kGridRowsF32)
    if (int rc = go(static_cast<const float*>(x) + r * k, static_cast<float*>(out) + r * n,
                    m - r < kGridRowsF32 ? m - r : kGridRowsF32))
      return rc;
  return 0;
}

// elements of a 16-byte chunk of a float dtype
int64_t chunkOf(int dtype) { return dtype == DLI_F32 ? 4 : 8; }

// wide: the 16-byte form, for aligned tensors of whole chunks (b too, when it repeats)
int binary(FloatKernels& kernels, FloatKernels& wide, const char* op, int dtype, const void* a,
           const void* b, void* out, int64_t total, int64_t width, void* stream) {
  DeviceKernel* k = kernels.pick(dtype);
  if (k == nullptr) return badDtype(op, dtype);
  if (total < 0 || width < 0) return badArg(op, "negative size");
  if (total == 0) return 0;
  if (width == 0) return badArg(op, "broadcast operand is empty");
  if (a == nullptr || b == nullptr || out == nullptr) return badArg(op, "NULL pointer");
  const int64_t c = chunkOf(dtype);
  if (total % c == 0 && width % c == 0 && width <= total && total / c < (int64_t{1} << 32) &&
      aligned16(a) && aligned16(b) && aligned16(out))
    return launch(*wide.pick(dtype), {strideBlocks(total / c)}, {256}, 0, stream, a, b, out,
                  total / c, width / c);
  return launch(*k, {strideBlocks(total)}, {256}, 0, stream, a, b, out, total, width);
}

int unary(FloatKernels& kernels, FloatKernels& wide, const char* op, int dtype, const void* x,
          void* out, int64_t total, void* stream) {
  DeviceKernel* k = kernels.pick(dtype);
  if (k == nullptr) return badDtype(op, dtype);
  if (total < 0) return badArg(op, "negative size");
  if (total == 0) return 0;
  if (x == nullptr || out == nullptr) return badArg(op, "NULL pointer");
  const int64_t c = chunkOf(dtype);
  if (total % c == 0 && aligned16(x) && aligned16(out))
    return launch(*wide.pick(dtype), {strideBlocks(total / c)}, {256}, 0, stream, x, out, total / c);
  return launch(*k, {strideBlocks(total)}, {256}, 0, stream, x, out, total);
}

// ---- packed-row attention (packed_attention.hip) ------------------------------------------------
// Rows (queries x heads of a KV group) per workgroup: 128, or 64 for units of at most 64 rows.
int64_t packedTile(int64_t rows) { return rows > 64 ? 128 : 64; }

// The same without key splits (contiguous keys): 64 also while that leaves CUs without a second
// workgroup, since a tile of 128 rows walks the same keys at almost twice the time of each. In us with
// 128 / 64 rows, 28 / 4 heads of 128: 16 x 16 8.8 / 6.4 (the row kernel 6.5), 2 x 64 x 64 9.0 / 6.5, 500 x
// 500 27.9 / 20.0, 16 queries over 4096 keys 174 / 124; 1000 x 1000 (438 tiles of 64 rows) 49.6 with 128.
int64_t denseTile(int64_t rows, int64_t units) {
  return (rows + 63) / 64 * units <= 256 ? 64 : packedTile(rows);
}

// fp32 attention of few keys and few query rows times keys stays on the row kernel: the packed kernel's
// tiles cost a short prompt what 64 keys cost. In us packed / row, 28 / 4 heads: head_dim 64 16 x 16 6.3 /
// 4.5, 40 x 40 (44800) 6.4 / 6.0, 48 x 48 (64512) 6.4 / 6.5, 8 x 16 x 16 (57344) 6.5 / 7.0; head_dim 128
// 16 x 16 9.8 / 6.0, 40 x 40 10.2 / 8.5, 8 x 16 x 16 10.1 / 10.7; 4 / 4 heads of 128 96 x 96 15.0 / 13.5,
// 16 x 128 14.7 / 15.9.
bool rowKernelF32(int64_t rows, int64_t keys) { return keys <= 96 && rows * keys <= 49152; }

// Key splits for `blocks` row tiles over all (sequence, KV head) pairs and a cache of T 64-key tiles:
// at most two workgroups per CU, and as many as the shorter walk (T / n tiles of 1 to 2.4 us) pays for
// the partial results (their traffic and merge grow with n): n^2 <= 3 T, or, where the row tiles
// alone occupy half of the CUs, T / 6. Measured in us, T / 2 splits (the rule before) and these:
// 3 queries of 28 / 4 heads of 128 over 4000 keys 25.3 / 21.3 (13 splits), 4 x 10 over 3000 30 / 25.2,
// 14 / 2 heads of 64 over 4000 22.5 / 17.8, over 1000 12.2 / 10.8; 2 x 300 queries of 28 / 4 heads
// (136 row tiles) over 64 keys 30.9 / 21.8 (unsplit), over 150 31.4 / 24.7, over 600 36.4 / 35.7.
// Up to 4 tiles the merge costs more than any split gives (unsplit / split by the root): 2 queries of 14 /
// 2 heads of 64 over 2 tiles 5.1 / 7.0, 4 tiles 7.0 / 8.4, 6 tiles 9.0 / 8.9; 2 x 100 of 28 / 4 heads of
// 128 over 2 tiles 11.4 / 14.7, 4 tiles 15.9 / 19.0, 6 tiles 20.5 / 20.9.
int64_t packedSplits(int64_t blocks, int64_t capacity) {
  const int64_t tiles = (capacity + dk::kPackedTileK - 1) / dk::kPackedTileK;
  const int64_t most = blocks > 0 && tiles > 4 ? 512 / blocks : 1;
  int64_t splits = 1;
  while (splits < most && splits < 64 &&
         (blocks >= 128 ? 6 * (splits + 1) <= tiles : (splits + 1) * (splits + 1) <= 3 * tiles))
    ++splits;
  return splits;
}

size_t packedPartialBytes(int64_t rows, int64_t head_dim, int64_t splits) {
  return static_cast<size_t>(rows * splits * (head_dim + 2)) * sizeof(float);
}

// The flash and packed kernels mask scores and take their maximum before the scale is multiplied in
// (one fma per probability), which needs a positive one: with another scale a key that a row does not
// see, at -inf, would come out as +inf or NaN. The row kernels scale q first and take any.
bool scaleAfterMask(float scale) { return scale > 0.f && std::isfinite(scale); }

// Forms that the packed kernels take (others run on the generic kernels).
bool packedForm(int dtype, int64_t batch, int64_t q_heads, int64_t kv_heads, int64_t seq_q,
                int64_t keys, float scale, const void* q, const void* k, const void* v,
                const void* out) {
  const int64_t limit = int64_t{1} << 30;
  return (dtype == DLI_BF16 || dtype == DLI_F32) && batch * kv_heads <= 65535 && keys > 0 && keys < limit &&
         seq_q < limit && seq_q * (q_heads / kv_heads) < limit && scaleAfterMask(scale) &&
         aligned16(q) && aligned16(k) && aligned16(v) && aligned16(out);
}

}  // namespace

// K splits of the tiled bf16 GEMM for decode-sized m: double while the 64 x 64 tiles times the
// splits stay within 256 workgroups and each part keeps at least 256 columns (at most 16 parts).
// Measured at 64 rows with weights that miss the caches: 3584 x 3584 best at 4 parts (13 us),
// 3584 x 18944 at 4 (33 us), 512 x 3584 at 7-8 (11 us), 18944 x 3584 unsplit (42 us); more
// parts only add fp32 partial traffic.
int64_t bf16Splits(int64_t m, int64_t n, int64_t k) {
  const int64_t tiles = ((m + 63) / 64) * ((n + 63) / 64);
  int64_t splits = 1;
  while (splits < 16 && tiles * splits * 2 <= 256 && k / (splits * 2) >= 256) splits *= 2;
  return splits;
}

// decode-sized bf16 linears that run faster on the tiled MFMA GEMM than on the skinny kernels
// (measured at m = 1, 8, 32, 64 on Qwen2-0.5B and -7B shapes: from m = 64 on every shape, from
// m = 32 on the wide ones, never at m <= 8)
bool tiledDecodeLinear(int64_t m, int64_t n) { return m > 32 || (m > 8 && n >= 8192); }

// Which kernels a 16-bit linear of m rows runs on: the skinny kernels (K over the 4 or the 16 waves
// of a workgroup, no second launch) or the tiled GEMM.
enum class Linear16 { kSkinny4, kSkinny16, kTiled };

// Skinny needs m <= 64 and K % 64 == 0. Its waves load x themselves, 16 rows a fragment, which
// costs more with every row and column of x; 16 waves of 16 weight rows up to one workgroup per CU
// (n <= 4096), else 4 waves of 32 rows. Measured in us (4 waves / 16 waves / tiled with its parts),
// n x k at m rows: 896 x 896 m = 1 4.3 / 3.3 / 8.6, m = 64 10.3 / 7.1 / 8.2; 896 x 4864 m = 8
// 13 / 8.3 / 8.7, m = 16 15.2 / 10.7 / 8.9; 4096 x 1024 m = 64 11.4 / 8.7 / 9.8; 3584 x 3584 m = 17
// 13.9 / 10.0 / 10.9, m = 32 16.5 / 12.6 / 11.4; 10 x 4096 m = 32 13.1 / 11.6 / 12.4; 4864 x 896
// m = 32 6.8 / 8.3 / 9.5, m = 50 10.0 / 12.1 / 9.9. From 8192 columns a weight streams from memory,
// where the tiled kernel is ahead as soon as more than 8 rows share it (a step of 9 rows with a head
// of 152064 x 3584: 615 us, 639 with the skinny kernel).
Linear16 linear16Route(int64_t m, int64_t n, int64_t k) {
  if (m > 64 || k % 64 != 0) return Linear16::kTiled;
  if (n > 4096)
    return m <= 8 || (n < 8192 && m * k <= 32768) ? Linear16::kSkinny4 : Linear16::kTiled;
  return m <= 8 || m * k <= 65536 || (n <= 64 && m <= 32) ? Linear16::kSkinny16
                                                          : Linear16::kTiled;
}

// Output tiles of the 16-bit GEMM: 128 x 128 from about 168 of them (at 896 columns, 2048 rows /
// 112 tiles ran faster in 64 x 64 tiles, 4096 rows / 224 tiles in 128 x 128 tiles); else 64 x 64,
// with two K groups per workgroup where the tiles leave CUs with one workgroup (in us, one group /
// two: 77 x 896 x 896 6.6 / 6.2, 1000 x 896 x 4864 19.9 / 18.7, 300 x 4864 x 896 (380 tiles) 9.2 /
// 9.4). One row tile over more column tiles than CUs streams its weights past the caches: a large
// weight that stays out of the memory-side cache leaves it to the rest of the layer (34 tokens
// through a layer of hidden 3584, ffn 18944: 205 us, 212 with cached loads).
TileForm16 tileForm16(int64_t m, int64_t n) {
  const bool few = ((m + 63) / 64) * ((n + 63) / 64) <= 256;
  if (m <= 64) return few ? TileForm16::k64Two : TileForm16::k64Stream;
  if (((m + 127) / 128) * ((n + 127) / 128) >= 168) return TileForm16::k128;
  return few ? TileForm16::k64Two : TileForm16::k64;
}

// Grid and threads of a tile form; false when the rows do not fit the grid.
bool tileLaunch16(TileForm16 form, int64_t m, int64_t n, Dim3* grid, Dim3* block) {
  const int64_t tile = form == TileForm16::k128 ? 128 : 64;
  const int64_t gx = (n + tile - 1) / tile, gy = (m + tile - 1) / tile;
  if (gy > kMaxGridY || gx > (int64_t{1} << 31)) return false;
  *grid = Dim3{static_cast<unsigned>(gx), static_cast<unsigned>(gy)};
  *block = Dim3{form == TileForm16::k64Two ? 512u : 256u};
  return true;
}

// K parts of a 16-bit linear on the tiled GEMM: parts of `per` columns (whole slices).
struct Parts16 {
  int64_t parts, per;
};
Parts16 parts16(int64_t m, int64_t k, int64_t splits) {
  const int64_t slice = m <= 64 ? 128 : 64;
  const int64_t per = ((k + splits - 1) / splits + slice - 1) / slice * slice;
  return Parts16{(k + per - 1) / per, per};
}
int64_t splits16(int64_t m, int64_t n, int64_t k) {
  if (m <= 64) {
    // two parts are not worth the second launch against two K groups in one workgroup
    // (64 x 4864 x 896: 9.6 us in two parts, 6.3 unsplit)
    const int64_t splits = bf16Splits(m, n, k);
    return splits <= 2 ? 1 : splits;
  }
  // A workgroup walks its K one slice per LDS round trip: few tiles over a long K are split until
  // about 224 workgroups walk at most 6 parts of at least 768 columns. Measured in us unsplit /
  // split: 77 x 896 x 4864 16.0 / 9.4 (6 parts), 200 rows 16.6 / 12.3, 300 rows 17.6 / 13.7 (3
  // parts); from 600 rows, and at K = 1024, the parts' fp32 traffic costs more than it gives
  // (600 x 896 x 4864 18.6 / 21.6).
  const int64_t tiles = ((m + 63) / 64) * ((n + 63) / 64);
  if (tiles > 96) return 1;
  int64_t splits = 224 / tiles;
  if (splits > k / 768) splits = k / 768;
  return splits < 1 ? 1 : (splits > 6 ? 6 : splits);
}

size_t tiled16Workspace(int64_t m, int64_t n, int64_t k) {
  const int64_t parts = parts16(m, k, splits16(m, n, k)).parts;
  return parts > 1 ? static_cast<size_t>(parts * m * n) * sizeof(float) : 0;
}

// out = T(x w^T + bias) (or fp32), optional ReLU, or with a residual (bf16) bf16(residual +
// bf16(x w^T + bias)), for bf16 and f16 operands with K % 8 == 0 and 16-byte aligned x and w on the
// tiled MFMA GEMM; K is split as far as the workspace holds the parts.
int tiled16(int dtype, const void* x, const void* w, const void* bias, const void* residual,
            void* out, int64_t m, int64_t n, int64_t k, int out_f32, int relu, void* workspace,
            size_t workspace_bytes, void* stream) {
  const bool h = dtype == DLI_F16;
  Parts16 p = parts16(m, k, splits16(m, n, k));
  while (p.parts > 1 && (workspace == nullptr ||
                         workspace_bytes < static_cast<size_t>(p.parts * m * n) * sizeof(float)))
    p = parts16(m, k, p.parts / 2);
  if (p.parts == 1) {
    const TileForm16 form = tileForm16(m, n);
    Dim3 grid, block;
    if (!tileLaunch16(form, m, n, &grid, &block)) return badArg("linear", "m too large");
    const int f = static_cast<int>(form);
    if (residual != nullptr)
      return launch(k_mfma_linres[f], grid, block, 0, stream, x, w, bias, residual, out, m, n, k);
    return launch((h ? k_mfma_f16 : k_mfma_bf16)[f], grid, block, 0, stream, x, w, bias, out, m, n,
                  k, out_f32, relu);
  }
  DeviceKernel& kern = m <= 64 ? (h ? k_mfma_f16_splitk : k_mfma_bf16_splitk)
                               : (h ? k_mfma_f16_rows : k_mfma_bf16_rows);
  if (int rc = launch(kern,
                      {static_cast<unsigned>((n + 63) / 64), static_cast<unsigned>((m + 63) / 64),
                       static_cast<unsigned>(p.parts)},
                      {256}, 0, stream, x, w, static_cast<float*>(workspace), m, n, k, p.per))
    return rc;
  return launch(h ? k_splitk_reduce_f16 : k_splitk_reduce_bf16, {strideBlocks((m * n + 3) / 4)},
                {256}, 0, stream, static_cast<const float*>(workspace), bias, residual, out, m, n,
                static_cast<int>(p.parts), out_f32, relu);
}

// The split GEMM alone: fp32 parts [parts, m, n] of x w^T in the workspace (K in
// whole 128-wide slices over at most bf16Splits(m, n, k) parts, as many as the workspace holds,
// at least one), for a caller's own reduce. *parts_out = the number of parts written.
int tiledBf16Parts(const void* x, const void* w, int64_t m, int64_t n, int64_t k,
                   void* workspace, size_t workspace_bytes, void* stream, int* parts_out) {
  int64_t splits = bf16Splits(m, n, k);
  const size_t part = static_cast<size_t>(m * n) * sizeof(float);
  while (splits > 1 && workspace_bytes < part * splits) splits /= 2;
  if (workspace == nullptr || workspace_bytes < part)
    return fail(DLI_HIP_EINVAL, "tiled split GEMM: workspace too small");
  const int64_t per = ((k + splits - 1) / splits + 127) / 128 * 128;
  const int64_t parts = (k + per - 1) / per;
  *parts_out = static_cast<int>(parts);
  return launch(k_mfma_bf16_splitk,
                {static_cast<unsigned>((n + 63) / 64), static_cast<unsigned>((m + 63) / 64),
                 static_cast<unsigned>(parts)},
                {256}, 0, stream, x, w, static_cast<float*>(workspace), m, n, k, per);
}


int decodeAttentionFast(int dtype, const void* q, const void* key_pool, const void* value_pool,
                        const int32_t* block_table, void* out, int64_t batch, int64_t q_heads,
                        int64_t kv_heads, int64_t seq_q, int64_t head_dim, int64_t block_size,
                        int64_t max_blocks, int64_t past, const void* positions,
                        int positions_dtype, float scale, int requested_splits, void* workspace,
                        size_t workspace_bytes, void* stream);
size_t decodeAttentionWorkspace(int64_t batch, int64_t q_heads, int64_t seq_q, int64_t head_dim,
                                int64_t max_tokens);
}  // namespace dli::hip

using namespace dli::hip;

extern "C" {

int dli_hip_add(int dtype, const void* a, const void* b, void* out, int64_t total, int64_t width,
                void* stream) {
  return binary(k_add, k_add16, "add", dtype, a, b, out, total, width, stream);
}

int dli_hip_mul(int dtype, const void* a, const void* b, void* out, int64_t total, int64_t width,
                void* stream) {
  return binary(k_mul, k_mul16, "mul", dtype, a, b, out, total, width, stream);
}

int dli_hip_silu(int dtype, const void* x, void* out, int64_t total, void* stream) {
  return unary(k_silu, k_silu16, "silu", dtype, x, out, total, stream);
}

int dli_hip_relu(int dtype, const void* x, void* out, int64_t total, void* stream) {
  return unary(k_relu, k_relu16, "relu", dtype, x, out, total, stream);
}

int dli_hip_rms_norm(int dtype, const void* x, const void* weight, void* out, int64_t rows,
                     int64_t hidden, float eps, void* stream) {
  DeviceKernel* k = k_rms_norm.pick(dtype);
  if (k == nullptr) return badDtype("rms_norm", dtype);
  if (rows < 0 || hidden <= 0) return badArg("rms_norm", "rows must be >= 0 and hidden > 0");
  if (rows == 0) return 0;
  // bf16 rows of up to 4096 elements in 16-byte chunks: one wave per row
  if (dtype == DLI_BF16 && hidden % 8 == 0 && hidden <= 4096 && aligned16(x) &&
      aligned16(weight) && aligned16(out)) {
    const int64_t groups = (rows + 3) / 4;
    const unsigned blocks = static_cast<unsigned>(groups < 65535 ? groups : 65535);
    DeviceKernel& kernel = hidden <= 1024   ? k_rms_norm_rows
                           : hidden <= 2048 ? k_rms_norm_mid_rows
                                            : k_rms_norm_wide_rows;
    return launch(kernel, {blocks}, {256}, 0, stream, x, weight, out, rows,
                  static_cast<int>(hidden), eps);
  }
  const unsigned blocks = static_cast<unsigned>(rows < 65535 ? rows : 65535);
  return launch(*k, {blocks}, {256}, 0, stream, x, weight, out, rows, hidden, eps);
}

int dli_hip_embedding(int dtype, int ids_dtype, const void* ids, const void* table, void* out,
                      int64_t tokens, int64_t hidden, int64_t vocab, void* stream) {
  DeviceKernel* k = k_embedding.pick(dtype);
  if (k == nullptr) return badDtype("embedding", dtype);
  if (!validIndexDtype(ids_dtype)) return badArg("embedding", "ids must be int64 or int32");
  if (tokens < 0 || hidden < 0 || vocab < 0) return badArg("embedding", "negative size");
  if (tokens == 0 || hidden == 0) return 0;
  const int ids64 = ids_dtype == DLI_I64 ? 1 : 0;
  const unsigned blocks = static_cast<unsigned>(tokens < 65535 ? tokens : 65535);
  return launch(*k, {blocks}, {256}, 0, stream, ids, ids64, table, out, tokens, hidden, vocab);
}

int dli_hip_softmax(int dtype, const void* x, void* out, int64_t rows, int64_t width,
                    void* stream) {
  DeviceKernel* k = k_softmax.pick(dtype);
  if (k == nullptr) return badDtype("softmax", dtype);
  if (rows < 0 || width <= 0) return badArg("softmax", "rows must be >= 0 and width > 0");
  if (rows == 0) return 0;
  const unsigned blocks = static_cast<unsigned>(rows < 65535 ? rows : 65535);
  return launch(*k, {blocks}, {256}, 0, stream, x, out, rows, width);
}

int dli_hip_transpose2d(int dtype, const void* x, void* out, int64_t rows, int64_t cols,
                        void* stream) {
  DeviceKernel* k = k_transpose.pick(dtype);
  if (k == nullptr) return badDtype("transpose", dtype);
  if (rows < 0 || cols < 0) return badArg("transpose", "negative size");
  if (rows == 0 || cols == 0) return 0;
  if ((rows + 31) / 32 > 65535) return badArg("transpose", "too many rows");
  return launch(*k, {blocksFor(cols, 32), blocksFor(rows, 32)}, {256}, 0, stream, x, out, rows,
                cols);
}

int dli_hip_permute_0213(int dtype, const void* x, void* out, int64_t n0, int64_t n1, int64_t n2,
                         int64_t n3, void* stream) {
  const char* op = "permute_0213";
  int64_t elem = 0;
  switch (dtype) {
    case DLI_F32: case DLI_I32: elem = 4; break;
    case DLI_BF16: case DLI_F16: elem = 2; break;
    case DLI_I64: elem = 8; break;
    default: return badDtype(op, dtype);
  }
  if (n0 < 0 || n1 < 0 || n2 < 0 || n3 < 0) return badArg(op, "negative size");
  if (n0 == 0 || n1 == 0 || n2 == 0 || n3 == 0) return 0;
  if (x == nullptr || out == nullptr) return badArg(op, "NULL pointer");
  const int64_t row_bytes = n3 * elem;
  const bool wide = row_bytes % 16 == 0 && (reinterpret_cast<uintptr_t>(x) & 15u) == 0 &&
                    (reinterpret_cast<uintptr_t>(out) & 15u) == 0;
  const int64_t row = wide ? row_bytes / 16 : row_bytes / 2;
  return launch(wide ? k_permute16 : k_permute2, {strideBlocks(n0 * n1 * n2 * row)}, {256}, 0,
                stream, x, out, n0, n1, n2, row);
}

int dli_hip_batch_norm2d(int dtype, const void* x, const void* weight, const void* bias,
                         const void* running_mean, const void* running_var, void* out,
                         int64_t total, int64_t channels, int64_t spatial, float eps,
                         void* stream) {
  DeviceKernel* k = k_bn.pick(dtype);
  if (k == nullptr) return badDtype("batch_norm2d", dtype);
  if (total < 0 || channels <= 0 || spatial <= 0)
    return badArg("batch_norm2d", "channels and spatial must be positive");
  if (total == 0) return 0;
  return launch(*k, {strideBlocks(total)}, {256}, 0, stream, x, weight, bias, running_mean,
                running_var, out, total, channels, spatial, eps);
}

int dli_hip_max_pool2d(int dtype, const void* x, void* out, int64_t n, int64_t c, int64_t h,
                       int64_t w, int64_t out_h, int64_t out_w, int64_t kernel_h,
                       int64_t kernel_w, int64_t stride_h, int64_t stride_w, int64_t pad_h,
                       int64_t pad_w, void* stream) {
  DeviceKernel* k = k_maxpool.pick(dtype);
  if (k == nullptr) return badDtype("max_pool2d", dtype);
  if (kernel_h <= 0 || kernel_w <= 0 || stride_h <= 0 || stride_w <= 0 || pad_h < 0 || pad_w < 0)
    return badArg("max_pool2d", "kernel and stride must be positive, padding non-negative");
  const int64_t total = n * c * out_h * out_w;
  if (n < 0 || c < 0 || out_h < 0 || out_w < 0) return badArg("max_pool2d", "negative size");
  if (total == 0) return 0;
  return launch(*k, {strideBlocks(total)}, {256}, 0, stream, x, out, n, c, h, w, out_h, out_w,
                kernel_h, kernel_w, stride_h, stride_w, pad_h, pad_w);
}

int dli_hip_conv2d(int dtype, const void* x, const void* weight, const void* bias, void* out,
                   int64_t n, int64_t in_c, int64_t h, int64_t w, int64_t out_c, int64_t kernel_h,
                   int64_t kernel_w, int64_t out_h, int64_t out_w, int64_t stride_h,
                   int64_t stride_w, int64_t pad_h, int64_t pad_w, void* stream) {
  return dli_hip_conv2d_act(dtype, x, weight, bias, out, n, in_c, h, w, out_c, kernel_h, kernel_w,
                            out_h, out_w, stride_h, stride_w, pad_h, pad_w, DLI_ACT_NONE, nullptr,
                            0, stream);
}

size_t dli_hip_conv2d_workspace(int dtype, int64_t n, int64_t in_c, int64_t out_c,
                                int64_t kernel_h, int64_t kernel_w, int64_t out_h, int64_t out_w) {
  if (dtype != DLI_F32 || n <= 0 || in_c <= 0 || out_c <= 0 || kernel_h <= 0 || kernel_w <= 0 ||
      out_h <= 0 || out_w <= 0)
    return 0;
  const int64_t pixels = n * out_h * out_w, patch = in_c * kernel_h * kernel_w;
  // (the image size is not known here; what it decides is met by images of gigabytes only)
  const bool vec = patch % 4 == 0 && kernel_h * kernel_w < 32;
  return partBytesF32(planF32(out_c, pixels, patch, vec, false, kMaxPartsF32), out_c, pixels);
}

int dli_hip_conv2d_act(int dtype, const void* x, const void* weight, const void* bias, void* out,
                       int64_t n, int64_t in_c, int64_t h, int64_t w, int64_t out_c,
                       int64_t kernel_h, int64_t kernel_w, int64_t out_h, int64_t out_w,
                       int64_t stride_h, int64_t stride_w, int64_t pad_h, int64_t pad_w,
                       int activation, void* workspace, size_t workspace_bytes, void* stream) {
  if (activation != DLI_ACT_NONE && activation != DLI_ACT_RELU)
    return badArg("conv2d", "unknown activation");
  if (stride_h <= 0 || stride_w <= 0 || pad_h < 0 || pad_w < 0)
    return badArg("conv2d", "stride must be positive, padding non-negative");
  if (n < 0 || in_c < 0 || out_c < 0 || out_h < 0 || out_w < 0 || h < 0 || w < 0 ||
      kernel_h < 0 || kernel_w < 0)
    return badArg("conv2d", "negative size");
  const int64_t total = n * out_c * out_h * out_w;
  if (total == 0) return 0;
  if (x == nullptr || weight == nullptr || out == nullptr) return badArg("conv2d", "NULL pointer");
  const int relu = activation == DLI_ACT_RELU ? 1 : 0;
  // fp32: implicit GEMM on MFMA, 32-bit index math (every element index below 2^31)
  const int64_t pixels = n * out_h * out_w, patch = in_c * kernel_h * kernel_w;
  const int64_t limit = int64_t{1} << 31;
  if (dtype == DLI_F32 && kernel_h < 65536 && kernel_w < 65536 && n * in_c * h * w < limit &&
      total < limit && out_c * patch < limit &&
      pixels < limit && (out_h - 1) * stride_h + kernel_h < limit &&
      (out_w - 1) * stride_w + kernel_w < limit) {
    auto i32 = [](int64_t v) { return static_cast<int>(v); };
    // a patch too short for MFMA tiles (an RGB input layer): direct, output-write bound
    if ((patch == 9 || patch == 27) && (out_c + dk::kSmallOc - 1) / dk::kSmallOc <= kMaxGridY) {
      dk::SmallConvTable tab{};
      tab.patch = i32(patch);
      for (int k = 0; k < tab.patch; ++k) {
        const int c = k / i32(kernel_h * kernel_w), ky = (k / i32(kernel_w)) % i32(kernel_h),
                  kx = k % i32(kernel_w);
        tab.offset[k] = (c * i32(h) + ky) * i32(w) + kx;
        tab.ky[k] = ky;
        tab.kx[k] = kx;
      }
      return launch(patch == 9 ? k_conv_small9 : k_conv_small27,
                    {static_cast<unsigned>((pixels + 255) / 256),
                     static_cast<unsigned>((out_c + dk::kSmallOc - 1) / dk::kSmallOc)},
                    {256}, 0, stream, x, weight, bias, out, i32(n), i32(in_c), i32(h), i32(w),
                    i32(out_c), i32(out_h), i32(out_w), i32(stride_h), i32(stride_w), i32(pad_h),
                    i32(pad_w), relu, tab);
    }
    const bool vec = convVec(n, in_c, h, w, patch, kernel_h * kernel_w, out_h * out_w) &&
                     aligned16(weight);
    const PlanF32 p = planF32(out_c, pixels, patch, vec, false,
                              partsHeldF32(workspace, workspace_bytes, out_c, pixels));
    if ((out_c + 63) / 64 <= kMaxGridY) {
      const int rc =
          launch(k_f32_conv[p.form],
                 {static_cast<unsigned>((pixels + 63) / 64), static_cast<unsigned>((out_c + 63) / 64),
                  static_cast<unsigned>(p.parts)},
                 {p.threads}, 0, stream, x, weight, bias, out, workspace, i32(n), i32(in_c), i32(h),
                 i32(w), i32(out_c), i32(kernel_h), i32(kernel_w), i32(out_h), i32(out_w),
                 i32(stride_h), i32(stride_w), i32(pad_h), i32(pad_w), i32(p.per), relu);
      if (rc != 0 || p.parts == 1) return rc;
      return launch(k_conv_splitk_reduce, {strideBlocks((out_c * pixels + 3) / 4)}, {256}, 0,
                    stream, workspace, bias, out, out_c, pixels, out_h * out_w,
                    static_cast<int>(p.parts), relu);
    }
  }
  DeviceKernel* k = k_conv2d.pick(dtype);
  if (k == nullptr) return badDtype("conv2d", dtype);
  int rc = launch(*k, {strideBlocks(total)}, {256}, 0, stream, x, weight, bias, out, n, in_c, h, w,
                  out_c, kernel_h, kernel_w, out_h, out_w, stride_h, stride_w, pad_h, pad_w);
  if (rc == 0 && relu) rc = unary(k_relu, k_relu16, "relu", dtype, out, out, total, stream);
  return rc;
}

int dli_hip_linear(int dtype, int out_dtype, const void* x, const void* w, const void* bias,
                   void* out, int64_t m, int64_t n, int64_t k, void* stream) {
  return dli_hip_linear_act(dtype, out_dtype, x, w, bias, out, m, n, k, DLI_ACT_NONE, nullptr, 0,
                            stream);
}

size_t dli_hip_linear_workspace(int dtype, int64_t m, int64_t n, int64_t k) {
  if (m <= 0 || n <= 0 || k <= 0) return 0;
  if (dtype == DLI_BF16 || dtype == DLI_F16) {  // the tiled GEMM's K parts
    if (k % 8 != 0 || linear16Route(m, n, k) != Linear16::kTiled) return 0;
    return tiled16Workspace(m, n, k);
  }
  if (dtype != DLI_F32) return 0;
  return partBytesF32(planF32(m, n, k, k % 4 == 0, true, kMaxPartsF32), m, n);
}

int dli_hip_linear_act(int dtype, int out_dtype, const void* x, const void* w, const void* bias,
                       void* out, int64_t m, int64_t n, int64_t k, int activation,
                       void* workspace, size_t workspace_bytes, void* stream) {
  if (activation != DLI_ACT_NONE && activation != DLI_ACT_RELU)
    return badArg("linear", "unknown activation");
  if (out_dtype != dtype && out_dtype != DLI_F32)
    return badArg("linear", "out_dtype must equal dtype or be float32");
  if (m < 0 || n < 0 || k < 0) return badArg("linear", "negative size");
  if (m == 0 || n == 0) return 0;
  if (x == nullptr || w == nullptr || out == nullptr) return badArg("linear", "NULL pointer");
  const int out_f32 = out_dtype == DLI_F32 ? 1 : 0;
  const int relu = activation == DLI_ACT_RELU ? 1 : 0;
  if (dtype == DLI_F32 && m <= kMaxRowsF32) {
    return byRowsF32(x, out, m, n, k, [&](const void* xr, void* outr, int64_t rows) {
      const bool vec = k > 0 && k % 4 == 0 && aligned16(xr) && aligned16(w);
      const PlanF32 p =
          planF32(rows, n, k, vec, true, partsHeldF32(workspace, workspace_bytes, rows, n));
      const int rc = launch(k_f32_linear[p.form],
                            {static_cast<unsigned>((n + 63) / 64),
                             static_cast<unsigned>((rows + p.tile_rows - 1) / p.tile_rows),
                             static_cast<unsigned>(p.parts)},
                            {p.threads}, 0, stream, xr, w, bias, outr, workspace, rows, n, k, p.per,
                            relu);
      if (rc != 0 || p.parts == 1) return rc;
      return launch(k_splitk_reduce, {strideBlocks((rows * n + 3) / 4)}, {256}, 0, stream,
                    workspace, bias, outr, rows, n, static_cast<int>(p.parts), relu);
    });
  }
  int rc;
  const bool h16 = dtype == DLI_BF16 || dtype == DLI_F16;
  const bool wide = h16 && k > 0 && k % 8 == 0 && aligned16(x) && aligned16(w);
  const Linear16 route = wide ? linear16Route(m, n, k) : Linear16::kTiled;
  // without the workspace for its K parts, the tiled GEMM of few rows is slower than the skinny
  // kernels up to 32 rows
  const bool no_parts = m <= 32 && k % 64 == 0 &&
                        workspace_bytes < dli_hip_linear_workspace(dtype, m, n, k);
  if (wide && (route != Linear16::kTiled || no_parts)) {
    const int w16 = route == Linear16::kSkinny16 ? 1 : 0;
    auto& kernels = (dtype == DLI_F16 ? k_skinny_f16 : k_skinny_bf16)[w16];
    rc = launch(kernels[m <= 16 ? 0 : (m <= 32 ? 1 : 2)], {blocksFor(n, w16 ? 16 : 32)},
                {w16 ? 1024u : 256u}, 0, stream, x, w, bias, out, m, n, k, out_f32);
  } else if (wide && (m + 63) / 64 <= kMaxGridY) {
    return tiled16(dtype, x, w, bias, nullptr, out, m, n, k, out_f32, relu, workspace,
                   workspace_bytes, stream);
  } else {
    DeviceKernel* kt = k_gemm.pick(dtype);
    if (kt == nullptr) return badDtype("linear", dtype);
    if ((m + 63) / 64 > kMaxGridY) return badArg("linear", "m too large");
    rc = launch(*kt, {blocksFor(n, 64), blocksFor(m, 64)}, {256}, 0, stream, x, w, bias, out, m,
                n, k, 1, out_f32);
  }
  if (rc == 0 && relu) rc = unary(k_relu, k_relu16, "relu", out_dtype, out, out, m * n, stream);
  return rc;
}

int dli_hip_matmul(int dtype, const void* a, const void* b, void* out, int64_t m, int64_t n,
                   int64_t k, void* stream) {
  if (m < 0 || n < 0 || k < 0) return badArg("matmul", "negative size");
  if (m == 0 || n == 0) return 0;
  if (a == nullptr || b == nullptr || out == nullptr) return badArg("matmul", "NULL pointer");
  if (dtype == DLI_F32 && m <= kMaxRowsF32) {
    return byRowsF32(a, out, m, n, k, [&](const void* ar, void* outr, int64_t rows) {
      const bool vec = k > 0 && k % 4 == 0 && aligned16(ar);
      const PlanF32 p = planF32(rows, n, k, vec, false, 1);
      return launch(k_f32_matmul[p.form],
                    {static_cast<unsigned>((n + 63) / 64), static_cast<unsigned>((rows + 63) / 64)},
                    {p.threads}, 0, stream, ar, b, outr, rows, n, k);
    });
  }
  DeviceKernel* kt = k_gemm.pick(dtype);
  if (kt == nullptr) return badDtype("matmul", dtype);
  if ((m + 63) / 64 > kMaxGridY) return badArg("matmul", "m too large");
  const void* no_bias = nullptr;
  return launch(*kt, {blocksFor(n, 64), blocksFor(m, 64)}, {256}, 0, stream, a, b, no_bias, out, m,
                n, k, 0, 0);
}

int dli_hip_rotary(int dtype, const void* q, const void* k, const float* cos_table,
                   const float* sin_table, void* out_q, void* out_k, int64_t batch,
                   int64_t q_heads, int64_t k_heads, int64_t seq, int64_t head_dim, int64_t pairs,
                   int64_t max_pos, int64_t start_pos, const void* positions,
                   int positions_dtype, void* stream) {
  DeviceKernel* kr = k_rotary.pick(dtype);
  if (kr == nullptr) return badDtype("rotary_embedding", dtype);
  if (head_dim <= 0 || head_dim % 2 != 0) return badArg("rotary_embedding", "head_dim must be even");
  if (pairs < 0 || 2 * pairs > head_dim) return badArg("rotary_embedding", "pairs > head_dim / 2");
  if (positions != nullptr && !validIndexDtype(positions_dtype))
    return badArg("rotary_embedding", "positions must be int64 or int32");
  if (batch < 0 || q_heads < 0 || k_heads < 0 || seq < 0) return badArg("rotary_embedding", "negative size");
  const int64_t work = batch * (q_heads > k_heads ? q_heads : k_heads) * seq * (head_dim / 2);
  if (work == 0) return 0;
  const int pos64 = positions_dtype == DLI_I64 ? 1 : 0;
  // whole rows of 16-byte chunks, 32-bit indices: 2000 x (28 + 4) heads x 128 bf16 13.5 us -> 8
  const int64_t c = chunkOf(dtype), limit = int64_t{1} << 30;
  if (2 * pairs == head_dim && head_dim % c == 0 && batch < limit && seq < limit &&
      head_dim < limit && (q_heads + k_heads) < limit &&
      batch * (q_heads + k_heads) < limit / seq && batch * (q_heads + k_heads) * seq < limit / head_dim &&
      aligned16(q) && aligned16(k) && aligned16(out_q) && aligned16(out_k) &&
      aligned16(cos_table) && aligned16(sin_table))
    return launch(*k_rotary16.pick(dtype),
                  {strideBlocks(batch * (q_heads + k_heads) * seq * (head_dim / c))}, {256}, 0,
                  stream, q, k, cos_table, sin_table, out_q, out_k, batch, q_heads, k_heads, seq,
                  head_dim, max_pos, start_pos, positions, pos64);
  return launch(*kr, {strideBlocks(work)}, {256}, 0, stream, q, k, cos_table, sin_table, out_q,
                out_k, batch, q_heads, k_heads, seq, head_dim, pairs, max_pos, start_pos, positions,
                pos64);
}

// attention with out as [B, Hq, Sq, D] (out_bshd 0) or [B, Sq, Hq, D] (1, the flash kernel's forms)
static int attentionImpl(int dtype, const void* q, const void* k, const void* v, void* out,
                  int64_t batch, int64_t q_heads, int64_t kv_heads, int64_t seq_q, int64_t seq_k,
                  int64_t head_dim, int causal, float scale, int out_bshd, void* stream) {
  DeviceKernel* ka = k_attention.pick(dtype);
  if (ka == nullptr) return badDtype("attention", dtype);
  if (head_dim <= 0 || head_dim > 256) return badArg("attention", "head_dim must be in [1, 256]");
  if (kv_heads <= 0 || q_heads % kv_heads != 0)
    return badArg("attention", "q_heads must be a multiple of kv_heads");
  if (batch < 0 || seq_q < 0 || seq_k < 0) return badArg("attention", "negative size");
  const int64_t rows = batch * q_heads * seq_q;
  if (rows == 0) return 0;
  if (q == nullptr || k == nullptr || v == nullptr || out == nullptr)
    return badArg("attention", "NULL pointer");
  // bf16 with head_dim 64 (prefill): flash-style MFMA kernel, 128 queries per workgroup (64 for
  // query sequences of at most 64)
  const bool flash = dtype == DLI_BF16 && head_dim == 64 && seq_k > 0 &&
                     batch * q_heads <= 65535 && seq_q < (int64_t{1} << 30) &&
                     seq_k < (int64_t{1} << 30) && aligned16(q) && aligned16(k) && aligned16(v) &&
                     aligned16(out);
  if (flash && scaleAfterMask(scale)) {
    const float log2e = 1.4426950408889634f;
    const int64_t tile_q = seq_q > 64 ? 128 : 64;
    return launch(tile_q == 128 ? k_flash_attention_q32 : k_flash_attention,
                  {static_cast<unsigned>((seq_q + tile_q - 1) / tile_q),
                   static_cast<unsigned>(batch * q_heads)},
                  {256}, 0, stream, q, k, v, out, q_heads, kv_heads, seq_q, seq_k, causal,
                  scale * log2e, out_bshd);
  }
  // bf16 with head_dim 128: the packed-row MFMA kernel (fewer than 16 queries over long keys stay
  // on the row kernel, whose waves split the heads; the packed kernel has no key splits here)
  // fp32 with head_dim 64 or 128: the same on the fp32 matrix instruction.
  const bool f32 = dtype == DLI_F32;
  if (!out_bshd && (head_dim == 128 || (f32 && head_dim == 64)) && seq_q >= 16 &&
      !(f32 && rowKernelF32(rows, seq_k)) &&
      packedForm(dtype, batch, q_heads, kv_heads, seq_q, seq_k, scale, q, k, v, out)) {
    dk::PackedAttentionArgs a{};
    a.q = q;
    a.k = k;
    a.v = v;
    a.out = out;
    a.q_heads = static_cast<int32_t>(q_heads);
    a.kv_heads = static_cast<int32_t>(kv_heads);
    a.seq_q = static_cast<int32_t>(seq_q);
    a.keys = static_cast<int32_t>(seq_k);
    a.causal = causal;
    a.splits = 1;
    a.scale_log2 = scale * 1.4426950408889634f;
    const int64_t unit_rows = seq_q * (q_heads / kv_heads);
    const int64_t tile = f32 ? 64 : denseTile(unit_rows, batch * kv_heads);
    DeviceKernel& kern = f32 ? (head_dim == 64 ? k_packed_f32_64 : k_packed_f32_128)
                             : (tile == 128 ? k_packed_dense128_r128 : k_packed_dense128);
    return launch(kern,
                  {blocksFor(unit_rows, tile), static_cast<unsigned>(batch * kv_heads)}, {256}, 0,
                  stream, a);
  }
  if (out_bshd && !flash)
    return badArg("attention", "a [B, S, H, D] output needs bf16, head_dim 64, seq_k > 0 and "
                               "16-byte aligned tensors (the flash kernel)");
  if (rows > 0x7fffffff) return badArg("attention", "too many query rows");
  return launch(*ka, {static_cast<unsigned>(rows)}, {64}, 0, stream, q, k, v, out, batch, q_heads,
                kv_heads, seq_q, seq_k, head_dim, causal, scale, out_bshd);
}

int dli_hip_attention(int dtype, const void* q, const void* k, const void* v, void* out,
                      int64_t batch, int64_t q_heads, int64_t kv_heads, int64_t seq_q,
                      int64_t seq_k, int64_t head_dim, int causal, float scale, void* stream) {
  return attentionImpl(dtype, q, k, v, out, batch, q_heads, kv_heads, seq_q, seq_k, head_dim,
                       causal, scale, 0, stream);
}

int dli_hip_attention_bshd(int dtype, const void* q, const void* k, const void* v, void* out,
                           int64_t batch, int64_t q_heads, int64_t kv_heads, int64_t seq_q,
                           int64_t seq_k, int64_t head_dim, int causal, float scale,
                           void* stream) {
  return attentionImpl(dtype, q, k, v, out, batch, q_heads, kv_heads, seq_q, seq_k, head_dim,
                       causal, scale, 1, stream);
}

int dli_hip_kv_append(int dtype, const void* key, const void* value, void* key_pool,
                      void* value_pool, const int32_t* block_table, int64_t batch, int64_t heads,
                      int64_t seq, int64_t head_dim, int64_t block_size, int64_t max_blocks,
                      int64_t start, const void* positions, int positions_dtype, void* stream) {
  DeviceKernel* ka = k_kv_append.pick(dtype);
  if (ka == nullptr) return badDtype("kv_append", dtype);
  if (block_size <= 0 || max_blocks <= 0) return badArg("kv_append", "empty cache geometry");
  if (positions != nullptr && !validIndexDtype(positions_dtype))
    return badArg("kv_append", "positions must be int64 or int32");
  if (batch < 0 || heads < 0 || seq < 0 || head_dim < 0) return badArg("kv_append", "negative size");
  const int64_t total = batch * heads * seq * head_dim;
  if (total == 0) return 0;
  const int pos64 = positions_dtype == DLI_I64 ? 1 : 0;
  // bf16 prompts (at least 16 new tokens) with 16-byte rows: 16 tokens of one head per
  // workgroup, values transposed in LDS (a decode step's one token stays on the element kernel:
  // 14 us against a few for the tiles at batch 64 x 4 heads)
  if (dtype == DLI_BF16 && seq >= 16 && head_dim % 8 == 0 && head_dim <= 256 &&
      batch * heads <= 65535 &&
      aligned16(key) && aligned16(value) && aligned16(key_pool)) {
    const int64_t chunks = (seq + 15) / 16;  // 16 tokens of one head per workgroup
    if (chunks <= 0x7fffffff)
      return launch(k_kv_append_tiles, {static_cast<unsigned>(chunks),
                                        static_cast<unsigned>(batch * heads)},
                    {256}, 0, stream, key, value, key_pool, value_pool, block_table, heads, seq,
                    static_cast<int>(head_dim), block_size, max_blocks, start, positions, pos64);
  }
  return launch(*ka, {strideBlocks(total)}, {256}, 0, stream, key, value, key_pool, value_pool,
                block_table, batch, heads, seq, head_dim, block_size, max_blocks, start, positions,
                pos64);
}

size_t dli_hip_paged_attention_workspace(int64_t batch, int64_t q_heads, int64_t seq_q,
                                         int64_t head_dim, int64_t max_tokens) {
  return decodeAttentionWorkspace(batch, q_heads, seq_q, head_dim, max_tokens);
}

// workspace: the decode kernels' (one query per sequence); partials: the packed kernels' key splits
static int pagedAttention(int dtype, const void* q, const void* key_pool, const void* value_pool,
                          const int32_t* block_table, void* out, int64_t batch, int64_t q_heads,
                          int64_t kv_heads, int64_t seq_q, int64_t head_dim, int64_t block_size,
                          int64_t max_blocks, int64_t past, const void* positions,
                          int positions_dtype, int causal, float scale, int splits,
                          void* workspace, size_t workspace_bytes, void* partials,
                          size_t partial_bytes, void* stream) {
  DeviceKernel* ka = k_paged_attention.pick(dtype);
  if (ka == nullptr) return badDtype("paged_attention", dtype);
  if (head_dim <= 0 || head_dim > 256) return badArg("paged_attention", "head_dim must be in [1, 256]");
  if (kv_heads <= 0 || q_heads % kv_heads != 0)
    return badArg("paged_attention", "q_heads must be a multiple of kv_heads");
  if (block_size <= 0 || max_blocks <= 0) return badArg("paged_attention", "empty cache geometry");
  if (positions != nullptr && !validIndexDtype(positions_dtype))
    return badArg("paged_attention", "positions must be int64 or int32");
  if (batch < 0 || seq_q < 0) return badArg("paged_attention", "negative size");
  if (splits < 0 || splits > kMaxDecodeSplits)
    return badArg("paged_attention", "splits must be in [0, 32]");
  const int64_t rows = batch * q_heads * seq_q;
  if (rows == 0) return 0;
  if (rows > 0x7fffffff) return badArg("paged_attention", "too many query rows");
  if (causal || seq_q == 1) {
    const int rc = decodeAttentionFast(dtype, q, key_pool, value_pool, block_table, out, batch,
                                       q_heads, kv_heads, seq_q, head_dim, block_size, max_blocks,
                                       past, positions, positions_dtype, scale, splits, workspace,
                                       workspace_bytes, stream);
    if (rc != 1) return rc;
  }
  const int pos64 = positions_dtype == DLI_I64 ? 1 : 0;
  // several queries per sequence: the packed-row MFMA kernels (64-key tiles inside cache blocks)
  if (dtype == DLI_BF16 && seq_q > 1 && (head_dim == 64 || head_dim == 128) &&
      block_size % dk::kPackedTileK == 0 && block_size < (int64_t{1} << 30) && max_blocks < (int64_t{1} << 30) &&
      packedForm(dtype, batch, q_heads, kv_heads, seq_q, max_blocks * block_size, scale, q, key_pool,
                 value_pool, out)) {
    const int64_t unit_rows = seq_q * (q_heads / kv_heads), tile = packedTile(unit_rows);
    const int64_t units = batch * kv_heads, blocks = (unit_rows + tile - 1) / tile;
    int64_t n = packedSplits(blocks * units, max_blocks * block_size);
    while (n > 1 &&
           (partials == nullptr || partial_bytes < packedPartialBytes(rows, head_dim, n)))
      --n;
    dk::PackedAttentionArgs a{};
    a.q = q;
    a.k = key_pool;
    a.v = value_pool;
    a.block_table = block_table;
    a.positions = positions;
    a.out = out;
    a.part_o = static_cast<float*>(partials);
    a.part_ml = n > 1 ? a.part_o + rows * n * head_dim : nullptr;
    a.past = past;
    a.max_blocks = max_blocks;
    a.pos64 = pos64;
    a.block_size = static_cast<int32_t>(block_size);
    a.q_heads = static_cast<int32_t>(q_heads);
    a.kv_heads = static_cast<int32_t>(kv_heads);
    a.seq_q = static_cast<int32_t>(seq_q);
    a.keys = static_cast<int32_t>(max_blocks * block_size);
    a.causal = causal;
    a.splits = static_cast<int32_t>(n);
    a.scale_log2 = scale * 1.4426950408889634f;
    const bool d64 = head_dim == 64, big = tile == 128;
    DeviceKernel& k = d64 ? (big ? k_packed_paged64_r128 : k_packed_paged64)
                          : (big ? k_packed_paged128_r128 : k_packed_paged128);
    if (int rc = launch(k, {static_cast<unsigned>(blocks), static_cast<unsigned>(units),
                            static_cast<unsigned>(n)},
                        {256}, 0, stream, a))
      return rc;
    if (n == 1) return 0;
    return launch(d64 ? k_packed_merge64 : k_packed_merge128,
                  {blocksFor(rows, 1024 / head_dim)}, {256}, 0, stream, a,
                  static_cast<int>(units));
  }
  return launch(*ka, {static_cast<unsigned>(rows)}, {64}, 0, stream, q, key_pool, value_pool,
                block_table, out, batch, q_heads, kv_heads, seq_q, head_dim, block_size, max_blocks,
                past, positions, pos64, causal, scale);
}

int dli_hip_paged_attention(int dtype, const void* q, const void* key_pool,
                            const void* value_pool, const int32_t* block_table, void* out,
                            int64_t batch, int64_t q_heads, int64_t kv_heads, int64_t seq_q,
                            int64_t head_dim, int64_t block_size, int64_t max_blocks, int64_t past,
                            const void* positions, int positions_dtype, int causal, float scale,
                            int splits, void* workspace, size_t workspace_bytes, void* stream) {
  return pagedAttention(dtype, q, key_pool, value_pool, block_table, out, batch, q_heads, kv_heads,
                        seq_q, head_dim, block_size, max_blocks, past, positions, positions_dtype,
                        causal, scale, splits, workspace, workspace_bytes, nullptr, 0, stream);
}

size_t dli_hip_chunk_attention_workspace(int dtype, int64_t batch, int64_t q_heads, int64_t seq_q,
                                         int64_t head_dim, int64_t max_tokens) {
  if (dtype != DLI_BF16 || batch <= 0 || q_heads <= 0 || seq_q <= 1 ||
      (head_dim != 64 && head_dim != 128))
    return 0;
  // fewer splits than this holds are used when the KV heads cut the rows into more tiles
  const int64_t rows = batch * q_heads * seq_q;
  const int64_t splits = packedSplits((rows + 127) / 128, max_tokens);
  return splits > 1 ? packedPartialBytes(rows, head_dim, splits) : 0;
}

int dli_hip_chunk_attention(int dtype, const void* q, const void* key_pool,
                            const void* value_pool, const int32_t* block_table, void* out,
                            int64_t batch, int64_t q_heads, int64_t kv_heads, int64_t seq_q,
                            int64_t head_dim, int64_t block_size, int64_t max_blocks, int64_t past,
                            const void* positions, int positions_dtype, int causal, float scale,
                            void* workspace, size_t workspace_bytes, void* stream) {
  if (seq_q == 1) return badArg("chunk_attention", "one query per sequence: paged_attention");
  return pagedAttention(dtype, q, key_pool, value_pool, block_table, out, batch, q_heads, kv_heads,
                        seq_q, head_dim, block_size, max_blocks, past, positions, positions_dtype,
                        causal, scale, 0, nullptr, 0, workspace, workspace_bytes, stream);
}

int dli_hip_argmax(int dtype, const void* x, int64_t* ids, int64_t rows, int64_t width,
                   void* stream) {
  DeviceKernel* ka = k_argmax.pick(dtype);
  if (ka == nullptr) return badDtype("argmax", dtype);
  if (rows < 0 || width <= 0) return badArg("argmax", "rows must be >= 0 and width > 0");
  if (rows == 0) return 0;
  const unsigned blocks = static_cast<unsigned>(rows < 65535 ? rows : 65535);
  // wide fp32 rows (logits over a vocabulary): the 16-byte-load kernel
  if (dtype == DLI_F32 && width % 4 == 0 && width >= 4096 &&
      (reinterpret_cast<uintptr_t>(x) & 15u) == 0)
    return launch(k_argmax_rows_v4, {blocks}, {1024}, 0, stream, x, ids, rows, width);
  return launch(*ka, {blocks}, {256}, 0, stream, x, ids, rows, width);
}

}  // extern "C"
