// Attention output projection + post-attention RMSNorm + residual (gfx950).
// Follows project_attention_out_post_attention
// (src/gemma4_flash_attention_decode.cu:34-129): a GEMV of the attention row
// (16 query heads x head_dim) against the column-major O weights
// ([3840][width]), the learned RMSNorm of the bf16 result
// (src/gemma4_rmsnorm.cu:28-85) and the residual add
// (src/gemma4_cuda_utils.cuh:105-122).
//
// The weights (31.5 MiB for width 4096, 63 MiB for 8192) are read once per
// launch; that stream is the roofline (HBM). They run on bf16 MFMA (exact
// products, fp32 sums), so a batch of decode rows costs little more than one
// row. The norm needs the whole 3840-wide row, so a second small kernel (one
// workgroup per row) applies it and the residual add.
#include "gemma4_attention_output.h"
#include "gemma4_device.hpp"
#include "lds_copy.hpp"
#include "prep_common.hpp"

namespace gemma4 {
namespace {

constexpr int kHidden = GEMMA4_ATTENTION_OUTPUT_HIDDEN;
constexpr int kNormThreads = 512;
constexpr int kHiddenPacks = kHidden / kPackElems;  // 480
static_assert(kHiddenPacks <= kNormThreads, "one pack per norm thread");

// Few rows (kFewRows): v_dot2 GEMV. A wave owns kCols hidden columns and holds
// all of their weights in registers (32 16-byte packs per lane, each load
// instruction reading 1 KiB of one column's contiguous weights), then runs
// each row against them: lane l dots packs l, l + 64, ... (exact bf16
// products, one rounding per pair) and a wave sum finishes each column.
constexpr int kRowWaves = 4;

template <int kWidth>
struct RowShape {
  static constexpr int kPacks = kWidth / (kPackElems * kWave);  // per lane per column
  static constexpr int kCols = 32 / kPacks;                     // 32 packs in flight per lane
  static constexpr int kGroups = kHidden / (kCols * kRowWaves);
  // The most rows that this kernel takes. Projection + tail with the weights
  // streamed from HBM, here and on the MFMA kernel: width 4096, 1 / 2 / 3 / 4
  // rows 9.4 / 10.2 / 10.9 / 11.6 us against - / 11.0 / 11.2 / 11.3; width
  // 8192, 1 / 2 / 4 / 6 rows 14.1 / 15.4 / 18.0 / 19.9 against 18.8 / 18.9 /
  // 19.0 / 19.0 (with the weights in the Infinity Cache the MFMA kernel is
  // level at one row, but a model's layers do not fit there).
  static constexpr int kFewRows = kWidth == 4096 ? 3 : 4;
  static_assert(kWidth % (kPackElems * kWave) == 0 && 32 % kPacks == 0, "width");
  static_assert(kHidden % (kCols * kRowWaves) == 0, "whole column groups");
};

template <int kWidth>
__global__ __launch_bounds__(kRowWaves *kWave) void o_projection_rows_kernel(
    const uint16_t *__restrict__ attn, const uint16_t *__restrict__ w,
    uint16_t *__restrict__ residual, int32_t rows) {
  using S = RowShape<kWidth>;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = wave_uniform(threadIdx.x / kWave);
  const int col0 = (blockIdx.x * kRowWaves + wave) * S::kCols;
  uint4 wp[S::kCols][S::kPacks];
#pragma unroll
  for (int c = 0; c < S::kCols; ++c)
#pragma unroll
    for (int i = 0; i < S::kPacks; ++i)
      wp[c][i] = load128_stream(w + (int64_t)(col0 + c) * kWidth + (i * kWave + lane) * kPackElems);
  for (int32_t r = 0; r < rows; ++r) {
    const uint16_t *a = attn + (int64_t)r * kWidth;
    uint4 ap[S::kPacks];
#pragma unroll
    for (int i = 0; i < S::kPacks; ++i) ap[i] = load128(a + (i * kWave + lane) * kPackElems);
    float sum[S::kCols];
#pragma unroll
    for (int c = 0; c < S::kCols; ++c) {
      float s = 0.0f;
#pragma unroll
      for (int i = 0; i < S::kPacks; ++i) {
        s = dot2_bf16(ap[i].x, wp[c][i].x, s);
        s = dot2_bf16(ap[i].y, wp[c][i].y, s);
        s = dot2_bf16(ap[i].z, wp[c][i].z, s);
        s = dot2_bf16(ap[i].w, wp[c][i].w, s);
      }
      sum[c] = wave_sum(s);
    }
    if (lane == 0) {
      uint16_t *out = residual + (int64_t)r * kHidden + col0;
      if constexpr (S::kCols == 4) {
        *reinterpret_cast<uint2 *>(out) =
            make_uint2(pack_bf16x2(sum[0], sum[1]), pack_bf16x2(sum[2], sum[3]));
      } else {
        *reinterpret_cast<uint32_t *>(out) = pack_bf16x2(sum[0], sum[1]);
      }
    }
  }
}

// Otherwise: D[row][col] = sum_k attn[row][k] * W[col][k] on
// v_mfma_f32_16x16x32_bf16. Workgroup: kColBlocks x 16 hidden columns and
// kRowBlocks x 16 rows; its four waves split k and work on their own until
// the partial sums meet in LDS. In a step lane l supplies A = attn[row l % 16]
// [k0 + 8 (l / 16) ..] and B = W[col l % 16][the same k], one 16-byte pack
// each, and the fp32 result holds column l % 16, rows 4 (l / 16) + 0..3.
// Loaded that way from memory, every group of 16 lanes touches 16 cache lines
// for 16 bytes each, and the CU's address path, not HBM, sets the time (16
// more rows of width 8192 cost 5.5 us, 20 bytes a clock and CU). So both
// operands come through LDS: 64 k (one 128-byte line) of 8 rows per copy
// instruction, into a ring of the wave's own; chunk c of row r at
// c ^ (r / 2 % 8), which keeps the operand reads free of bank conflicts.
// Projection + tail, before and now, weights from HBM: width 8192, 8 rows
// 21.2 -> 19.1 us, 24 28.1 -> 20.8, 64 44.9 -> 25.6, 128 78 -> 31.6; width
// 4096, 8 rows 12.9 -> 11.6, 64 25.1 -> 15.5, 128 39.8 -> 18.9. With four
// copies of the weights in turn, which the 256 MiB Infinity Cache still helps:
// width 8192, 24 rows 30.5 -> 15.1 (kernel 26.2 -> 13.0), 256 155 -> 37.
// Not taken: nontemporal weight copies. From HBM they gain 1-2 us up to 24
// rows (8192, 8 rows 17.1) and lose from 64 rows on; with weights that the
// Infinity Cache holds they lose 4 (24 rows 19.0 against 15.1). (The GEMV for
// few rows gains from HBM and loses nothing there.)
constexpr int kSplit = 4;  // waves per workgroup, one k slice each
constexpr int kChunkK = 64;
constexpr int kBlockUint4 = 16 * kChunkK / kPackElems;  // 16 rows of a chunk: 2 KiB
constexpr int kRingBytes = 36 * 1024;                   // per wave

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4_t mfma16(uint4 a, uint4 b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                 __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

template <int kWidth, int kRowBlocks, int kColBlocks>
__global__ __launch_bounds__(kSplit *kWave) void o_projection_kernel(
    const uint16_t *__restrict__ attn, const uint16_t *__restrict__ w,
    uint16_t *__restrict__ residual, int32_t rows, int32_t row_groups) {
  constexpr int kBlocks = kRowBlocks + kColBlocks;  // 2 KiB each in a ring entry
  constexpr int kRing = kRingBytes / (kBlocks * kBlockUint4 * 16) < 8
                            ? kRingBytes / (kBlocks * kBlockUint4 * 16) : 8;
  constexpr int kCopies = 2 * kBlocks;  // per entry
  constexpr int kChunks = kWidth / kSplit / kChunkK;
  static_assert(kRing >= 2 && kRing <= kChunks && (kRing - 1) * kCopies < 63, "ring");
  __shared__ __attribute__((aligned(1024))) uint4 s_ring[kSplit][kRing][kBlocks][kBlockUint4];
  static_assert(kRing * kBlocks * 2 >= kRowBlocks * kColBlocks, "partial sums fit the ring");
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = wave_uniform(threadIdx.x / kWave);
  // Workgroups of one column group are eight apart (one XCD), so that its
  // row groups share the weights in that L2.
  const int xcd = blockIdx.x % 8, rest = blockIdx.x / 8;
  const int col0 = (rest / row_groups * 8 + xcd) * 16 * kColBlocks;
  const int row0 = rest % row_groups * 16 * kRowBlocks;
  if (col0 >= kHidden) return;

  // Byte offsets of this lane's 16 bytes within a row block's chunk, for the
  // two copies of a block: rows lane / 8 and 8 + lane / 8. Rows past the last
  // repeat it; their results are not stored.
  uint32_t w_off[2], a_off[kRowBlocks][2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = 8 * i + lane / 8;
    const uint32_t chunk = (uint32_t)((lane % 8) ^ ((r >> 1) & 7)) * 16;
    w_off[i] = (uint32_t)r * kWidth * 2 + chunk;
#pragma unroll
    for (int b = 0; b < kRowBlocks; ++b)
      a_off[b][i] = (uint32_t)min(16 * b + r, rows - 1 - row0) * kWidth * 2 + chunk;
  }
  const uint64_t k_base = (uint64_t)wave * (kWidth / kSplit) * 2;
  const uint64_t w_base = reinterpret_cast<uint64_t>(w) + (uint64_t)col0 * kWidth * 2 + k_base;
  const uint64_t a_base = reinterpret_cast<uint64_t>(attn) + (uint64_t)row0 * kWidth * 2 + k_base;
  const uint32_t ring_lds = wave_uniform(lds_address(&s_ring[wave][0][0][0]));
  auto request = [&](int chunk, int entry) __attribute__((always_inline)) {
    const uint32_t lds = ring_lds + entry * (kBlocks * kBlockUint4 * 16);
    const uint64_t k = (uint64_t)chunk * kChunkK * 2;
#pragma unroll
    for (int b = 0; b < kColBlocks; ++b)
      copy_lanes2(w_base + k + (uint64_t)b * 16 * kWidth * 2, w_off[0],
                  w_base + k + (uint64_t)b * 16 * kWidth * 2, w_off[1], lds + b * kBlockUint4 * 16);
#pragma unroll
    for (int b = 0; b < kRowBlocks; ++b)
      copy_lanes2(a_base + k, a_off[b][0], a_base + k, a_off[b][1],
                  lds + (kColBlocks + b) * kBlockUint4 * 16);
  };

  // Few blocks leave registers for four sums each: shorter chains, a smaller
  // rounding error and no MFMA that waits for the one before it.
  constexpr int kSums = kRowBlocks * kColBlocks <= 2 ? 4 : 2;
  f32x4_t acc[kSums][kRowBlocks][kColBlocks];
#pragma unroll
  for (int i = 0; i < kSums; ++i)
#pragma unroll
    for (int b = 0; b < kRowBlocks; ++b)
#pragma unroll
      for (int c = 0; c < kColBlocks; ++c) acc[i][b][c] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < kRing; ++i) request(i, i);
  const int h = lane & 15, g = lane >> 4;
  int entry = 0;
  static_assert(kChunks % 2 == 0, "chunks go in pairs");
#pragma unroll 1
  for (int j0 = 0; j0 < kChunks; j0 += 2) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int j = j0 + i;
      if (j + kRing <= kChunks) {
        wait_vector<(kRing - 1) * kCopies>();  // the younger entries stay in flight
      } else {
        wait_vector<0>();
      }
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int slot = h * 8 + ((4 * t + g) ^ ((h >> 1) & 7));
        uint4 op[kBlocks];
#pragma unroll
        for (int b = 0; b < kBlocks; ++b) op[b] = s_ring[wave][entry][b][slot];
        f32x4_t(&sum)[kRowBlocks][kColBlocks] = acc[(2 * i + t) % kSums];
#pragma unroll
        for (int b = 0; b < kRowBlocks; ++b)
#pragma unroll
          for (int c = 0; c < kColBlocks; ++c)
            sum[b][c] = mfma16(op[kColBlocks + b], op[c], sum[b][c]);
      }
      wait_lds_reads();
      if (j + kRing < kChunks) request(j + kRing, entry);
      entry = entry + 1 == kRing ? 0 : entry + 1;
    }
  }

  // ---- partial sums of the k slices, over the wave's own ring
  f32x4_t *mine = reinterpret_cast<f32x4_t *>(&s_ring[wave][0][0][0]);
#pragma unroll
  for (int b = 0; b < kRowBlocks; ++b)
#pragma unroll
    for (int c = 0; c < kColBlocks; ++c) {
      f32x4_t sum = acc[0][b][c] + acc[1][b][c];
      if constexpr (kSums == 4) sum += acc[2][b][c] + acc[3][b][c];
      mine[(b * kColBlocks + c) * kWave + lane] = sum;
    }
  __syncthreads();
  for (int i = wave; i < kRowBlocks * kColBlocks; i += kSplit) {
    f32x4_t sum = reinterpret_cast<const f32x4_t *>(&s_ring[0][0][0][0])[i * kWave + lane];
#pragma unroll
    for (int k = 1; k < kSplit; ++k)
      sum += reinterpret_cast<const f32x4_t *>(&s_ring[k][0][0][0])[i * kWave + lane];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int32_t row = row0 + 16 * (i / kColBlocks) + 4 * g + e;
      if (row < rows)
        residual[(int64_t)row * kHidden + col0 + 16 * (i % kColBlocks) + h] =
            (uint16_t)f32_to_bf16_bits(sum[e]);
    }
  }
}

// One workgroup per row: thread t < 480 owns pack t of the hidden row.
__global__ __launch_bounds__(kNormThreads) void post_attention_norm_kernel(
    const uint16_t *__restrict__ residual, const uint16_t *__restrict__ weight,
    const uint16_t *__restrict__ x, uint16_t *__restrict__ normed, uint16_t *__restrict__ ffn) {
  __shared__ float wave_sums[kNormThreads / kWave];
  const int t = threadIdx.x;
  const int64_t off = (int64_t)blockIdx.x * kHidden + t * kPackElems;
  const bool owner = t < kHiddenPacks;
  float v[kPackElems] = {};
  if (owner) unpack8(load128(residual + off), v);
  float sq = 0.0f;
#pragma unroll
  for (int i = 0; i < kPackElems; ++i) sq = fmaf(v[i], v[i], sq);
  sq = wave_sum(sq);
  if ((t & (kWave - 1)) == 0) wave_sums[t / kWave] = sq;
  __syncthreads();
  float total = 0.0f;
#pragma unroll
  for (int i = 0; i < kNormThreads / kWave; ++i) total += wave_sums[i];
  if (!owner) return;
  const float scale = 1.0f / sqrtf(total / (float)kHidden + kRmsEps);
  float g[kPackElems], xi[kPackElems];
  unpack8(load128(weight + t * kPackElems), g);
  unpack8(load128(x + off), xi);
  float n[kPackElems], f[kPackElems];
#pragma unroll
  for (int i = 0; i < kPackElems; ++i) {
    n[i] = v[i] * scale * g[i];
    // The residual adds the bf16-rounded normed value.
    n[i] = __uint_as_float(f32_to_bf16_bits(n[i]) << 16);
    f[i] = xi[i] + n[i];
  }
  store128(normed + off, make_uint4(pack_bf16x2(n[0], n[1]), pack_bf16x2(n[2], n[3]),
                                    pack_bf16x2(n[4], n[5]), pack_bf16x2(n[6], n[7])));
  store128(ffn + off, make_uint4(pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3]),
                                 pack_bf16x2(f[4], f[5]), pack_bf16x2(f[6], f[7])));
}

template <int kWidth, int kRowBlocks, int kColBlocks>
hipError_t launch_blocks(const uint16_t *attn, const uint16_t *w, uint16_t *residual, int32_t rows,
                         hipStream_t stream) {
  const int row_groups = (rows + 16 * kRowBlocks - 1) / (16 * kRowBlocks);
  const int col_groups = kHidden / (16 * kColBlocks);
  hipLaunchKernelGGL((o_projection_kernel<kWidth, kRowBlocks, kColBlocks>),
                     dim3((col_groups + 7) / 8 * 8 * row_groups), dim3(kSplit * kWave), 0, stream,
                     attn, w, residual, rows, row_groups);
  return hipGetLastError();
}

// Row and column blocks per workgroup: 240 workgroups of up to 64 rows, so
// that every CU but 16 has one and the attention rows are read as seldom as
// that allows (column blocks = row groups). Up to 32 rows each workgroup
// takes them all; 33-64 rows as two groups of 32 (64 rows at width 8192:
// 21.5 us, as one group of 64 and half the columns 23.9), 128 as 2 x 64
// (29.7; 2 x 2 blocks 37.7), 192 as 3 x 64 (33.0; 4 x 2 blocks 50.4), 256 as
// 4 x 64 (37.2; 4 x 2 blocks 52.1).
template <int kWidth>
hipError_t launch_projection(const uint16_t *attn, const uint16_t *w, uint16_t *residual,
                             int32_t rows, hipStream_t stream) {
  using S = RowShape<kWidth>;
  // The MFMA kernel's copies into LDS take 16-byte aligned chunks; the GEMV's
  // loads may start anywhere.
  const bool aligned =
      ((reinterpret_cast<uintptr_t>(attn) | reinterpret_cast<uintptr_t>(w)) & 15) == 0;
  if (rows <= S::kFewRows || !aligned) {
    hipLaunchKernelGGL(o_projection_rows_kernel<kWidth>, dim3(S::kGroups), dim3(kRowWaves * kWave),
                       0, stream, attn, w, residual, rows);
    return hipGetLastError();
  }
  if (rows <= 16) return launch_blocks<kWidth, 1, 1>(attn, w, residual, rows, stream);
  if (rows <= 32) return launch_blocks<kWidth, 2, 1>(attn, w, residual, rows, stream);
  if (rows <= 64) return launch_blocks<kWidth, 2, 2>(attn, w, residual, rows, stream);
  if (rows <= 96) return launch_blocks<kWidth, 3, 2>(attn, w, residual, rows, stream);
  if (rows <= 128) return launch_blocks<kWidth, 4, 2>(attn, w, residual, rows, stream);
  if (rows <= 192) return launch_blocks<kWidth, 4, 3>(attn, w, residual, rows, stream);
  return launch_blocks<kWidth, 4, 4>(attn, w, residual, rows, stream);
}

}  // namespace
}  // namespace gemma4

extern "C" hipError_t gemma4_attention_o_projection_post_norm_bf16(
    gemma4_bf16 *residual_out, gemma4_bf16 *normed_out, gemma4_bf16 *ffn_residual,
    const gemma4_bf16 *attention_out, const gemma4_bf16 *o_proj_col_major,
    const gemma4_bf16 *post_norm_weight, const gemma4_bf16 *attention_x, int32_t rows,
    int32_t attention_width, hipStream_t stream) {
  using namespace gemma4;
  if (residual_out == nullptr || normed_out == nullptr || ffn_residual == nullptr ||
      attention_out == nullptr || o_proj_col_major == nullptr || post_norm_weight == nullptr ||
      attention_x == nullptr || rows < 0 || (attention_width != 4096 && attention_width != 8192)) {
    return hipErrorInvalidValue;
  }
  if (rows == 0) return hipSuccess;
  auto *res = reinterpret_cast<uint16_t *>(residual_out);
  const auto *attn = reinterpret_cast<const uint16_t *>(attention_out);
  const auto *w = reinterpret_cast<const uint16_t *>(o_proj_col_major);
  const hipError_t e = attention_width == 4096 ? launch_projection<4096>(attn, w, res, rows, stream)
                                               : launch_projection<8192>(attn, w, res, rows, stream);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(post_attention_norm_kernel, dim3(rows), dim3(kNormThreads), 0, stream, res,
                     reinterpret_cast<const uint16_t *>(post_norm_weight),
                     reinterpret_cast<const uint16_t *>(attention_x),
                     reinterpret_cast<uint16_t *>(normed_out),
                     reinterpret_cast<uint16_t *>(ffn_residual));
  return hipGetLastError();
}
