// Prefill self-attention launchers with Q/K/V preparation, gfx950: the drop-in
// for gemma4_flash_attention_{sliding,global}_fwd_bf16_norm_rope
// (src/gemma4_flash_attention.cuh:9-45, src/gemma4_flash_attention_prefill.cu:1110-1257).
// Each launcher runs two kernels on the caller's stream:
//   1. prefill_prep_kernel: per (token row, kv head) Q and K get learned
//      RMSNorm + split-half RoPE at the row's absolute position, V gets
//      scale-free RMSNorm (the 1x512 geometry derives V from the raw K), into
//      the caller's q/k/v_prepared buffers
//      (src/gemma4_flash_attention_prefill.cu:1023-1101);
//   2. causal attention over the prepared rows (seqlen_q == seqlen_k):
//      the 8x256 geometry reuses the chunk kernel (no prior context), the
//      1x512 geometry runs prefill_d512_kernel below.
//
// prefill_d512_short_kernel (sequences up to kD512ShortRows): 16 query heads
// share one 512-dim KV head. A wave owns
// one query row and all 16 heads (16 MFMA columns) on
// v_mfma_f32_16x16x32_bf16, computing S^T = K Q^T (16 keys x 16 heads per
// block, 16 k-steps of 32 dims) and O^T = V^T P^T (32 dim blocks of 16). In
// the 16x16 accumulator lane l holds head l % 16 and four keys (or dims)
// 4 (l/16) + i, so P^T feeds the second MFMA from registers when its 32-key
// contraction order is permuted to {4g..4g+3, 16+4g..16+4g+3} for lane
// group g, and V^T is read in that order by two ds_read_b64_tr_b16 per
// operand. O^T is 128 fp32 per lane (VGPR accumulator form, a build flag
// for this file), Q^T 64 registers held in AGPRs. A workgroup is four
// consecutive rows that share 32-key K/V tiles copied into two LDS stages
// with global_load_lds (tile t+1 in flight while tile t is computed; K chunk
// c of key k at c ^ (k & 15), V chunk c at c ^ ((k & 7) << 1), 16-byte
// chunks, so the operand reads are bank-conflict free). Scheduling: each
// score block issues its 16 K-fragment reads into AGPRs before its first
// MFMA (one counter wait per MFMA, two accumulator chains), and the P.V
// phase keeps its transposing V reads four MFMAs ahead. The lazy online
// softmax of the chunk kernel (maximum moved only when it grows by more than
// 8 in log2 units).
//
// prefill_d512_kernel (longer ones): the same tiles and operands on two waves
// per row. Each scores 16 of a tile's 32 keys and, for all four rows, weighs
// V in its own 64 dims, so that one V operand serves four MFMAs (32 instead of
// 128 KiB of V reads per tile and CU) and two waves per SIMD cover each
// other's LDS latency; maxima and probabilities travel through LDS. Three
// tiles are in work at once and one barrier separates iterations. What bounds
// it: the sum of many short LDS round trips, ~4000 clocks per 32-key iteration
// against 1024 of MFMA. 2048 / 1024 / 777 rows, prep included: 148.6 / 64.0 /
// 54.7 us against 163.2 / 74.0 / 61.1 on the short form; without the
// overlap of tiles 151.7 / 68.0 / 57.3. Back to back, 2048 rows: 155 -> 132.
#include "gemma4_device.hpp"
#include "lds_copy.hpp"
#include "prep_common.hpp"

#include "gemma4_flash_attention.h"

#include <math.h>
#include <type_traits>

namespace gemma4 {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef short i16x4_t __attribute__((ext_vector_type(4)));

struct PrefillPrepParams {
  uint16_t *q_prepared;  // [rows][16][D]
  uint16_t *k_prepared;  // [rows][Hk][D]
  uint16_t *v_prepared;
  const uint16_t *q;
  const uint16_t *k;
  const uint16_t *v;     // null for the 1x512 geometry (V from K)
  const uint16_t *q_norm_weight;
  const uint16_t *k_norm_weight;
  const float *cos;
  const float *sin;
  const int32_t *token_position;  // [rows]
};

// Workgroup (block of kPrepRows token rows, kv head), one wave per prepared
// head; a wave first loads its head of all kPrepRows rows, then prepares
// and stores them one by one, so the row loads overlap. A negative
// position skips the row (src/gemma4_flash_attention_prefill.cu:1049-1051).
// Two rows per workgroup: more, smaller workgroups measured faster for
// 2048 rows (launchers 8x256 / 1x512: 8 rows 67.5 / 164 us, 4 rows 64.5 /
// 157.3 us, 2 rows 63.5 / 157.4 us, 1 row 63.2 / 157.2 us, 16 rows 69.7 /
// 183.6 us).
constexpr int kPrepRows = 2;

template <int kHeads, int kDim, int kRotary, bool kHasV>
__global__ __launch_bounds__((prep_waves<kHeads, kHasV>() * kWave)) void prefill_prep_kernel(
    PrefillPrepParams p, int64_t rows) {
  constexpr int kGroup = kQueryHeads / kHeads;
  constexpr int kPer = kDim / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = wave_uniform(threadIdx.x / kWave);
  const int head = blockIdx.y;
  const int64_t row0 = (int64_t)blockIdx.x * kPrepRows;
  int32_t position[kPrepRows];
#pragma unroll
  for (int r = 0; r < kPrepRows; ++r)
    position[r] = row0 + r < rows ? wave_uniform(p.token_position[row0 + r]) : -1;
  float x[kPrepRows][kPer];
  // Loads the given tensor's head of every row of the block.
  auto load_rows = [&](const uint16_t *base, int heads_per_row, int h) {
#pragma unroll
    for (int r = 0; r < kPrepRows; ++r) {
      const int64_t rr = row0 + r < rows ? row0 + r : row0;
      load_head<kDim>(base + (rr * heads_per_row + h) * kDim, x[r], lane);
    }
  };
  if (wave < kGroup) {
    const int qh = head * kGroup + wave;
    load_rows(p.q, kQueryHeads, qh);
#pragma unroll
    for (int r = 0; r < kPrepRows; ++r) {
      if (position[r] < 0) continue;
      store_weighted_rope<kDim, kRotary>(
          p.q_prepared + ((row0 + r) * kQueryHeads + qh) * kDim, x[r], p.q_norm_weight,
          p.cos + (int64_t)position[r] * (kRotary / 2), p.sin + (int64_t)position[r] * (kRotary / 2),
          lane);
    }
    if (kHasV || wave != 0) return;
  }
  const bool k_wave = kHasV ? wave == kGroup : wave == 0;
  load_rows(k_wave ? p.k : p.v, kHeads, head);
#pragma unroll
  for (int r = 0; r < kPrepRows; ++r) {
    if (position[r] < 0) continue;
    const int64_t off = ((row0 + r) * kHeads + head) * kDim;
    if (k_wave) {
      store_weighted_rope<kDim, kRotary>(p.k_prepared + off, x[r], p.k_norm_weight,
                                         p.cos + (int64_t)position[r] * (kRotary / 2),
                                         p.sin + (int64_t)position[r] * (kRotary / 2), lane);
      if constexpr (!kHasV) store_scale_free<kDim>(p.v_prepared + off, x[r], lane);
    } else {
      store_scale_free<kDim>(p.v_prepared + off, x[r], lane);
    }
  }
}

// ---- 1x512 causal self-attention ---------------------------------------
// Up to this many rows the short form is faster: the long form fills its
// pipeline of three tiles first. Short / long, prep included, 1 / 2 / 4
// sequences: 260 rows 28.6 / 30.5, 32.3 / 34.0, 39.3 / 45.0 us; 400 36.3 / 37.4,
// 40.1 / 41.1, 59.8 / 62.5; 512 42.8 / 42.9, 45.9 / 45.5, 76.2 / 76.4; 700 52.4 /
// 51.6, 58.5 / 57.5, 102.6 / 105.2.
constexpr int kD512ShortRows = 512;
constexpr int kD512 = 512;
constexpr int kD512Rows = 4;          // query rows per workgroup, two waves each
constexpr int kD512Waves = 2 * kD512Rows;
constexpr int kD512Threads = kD512Waves * kWave;
constexpr int kD512ShortThreads = kD512Rows * kWave;  // the short form: a wave per row
constexpr int kD512VLead = 4;         // its P.V MFMAs the V reads run ahead
constexpr int kD512Tile = 32;         // keys per LDS tile
constexpr int kD512RowBytes = kD512 * 2;
constexpr int kD512Chunks = kD512RowBytes / 16;  // 16-byte chunks per row
constexpr float kD512Slack = 8.0f;
constexpr int kD512Blocks = kD512 / 16 / kD512Waves;  // 16-dim blocks of O^T per wave

struct D512Params {
  uint16_t *out;        // [B][L][16][512]
  const uint16_t *q;    // [B][L][16][512]
  const uint16_t *k;    // [B][L][1][512]
  const uint16_t *v;
  int32_t seq_len;
  float q_scale;        // softmax_scale * log2(e)
};

__device__ __forceinline__ f32x4_t mfma16(uint4 a, uint4 b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                 __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

typedef unsigned u32x4v_t __attribute__((ext_vector_type(4)));

// The 16 K-fragment reads of one 16-key score block into AGPRs, all in
// flight before the first MFMA. For lane key k (k & 15 = lane & 15) and lane
// group g, k-step s sits at chunk (4s + g) ^ (k & 15) of the key's row: bits
// 0-1 of the chunk are g ^ (k & 3), bits 2-3 are (s & 3) ^ ((k >> 2) & 3)
// and bits 4+ are s >> 2. So with base = the address of k-step 0, k-step s
// is at (base ^ (64 (s & 3))) + 256 (s >> 2): four XORed addresses, four
// immediate offsets each. Issue position p = 4 (s & 3) + (s >> 2).
template <int kImm>
__device__ __forceinline__ void d512_read_block(uint32_t k_addr, u32x4v_t (&kf)[16]) {
  uint32_t t0, t1;
  asm volatile(
      "s_waitcnt lgkmcnt(0)\n\t"
      "v_xor_b32 %[t0], 0, %[ka]\n\t"
      "ds_read_b128 %[f0], %[t0] offset:%[i0]\n\t"
      "ds_read_b128 %[f4], %[t0] offset:%[i1]\n\t"
      "ds_read_b128 %[f8], %[t0] offset:%[i2]\n\t"
      "ds_read_b128 %[f12], %[t0] offset:%[i3]\n\t"
      "v_xor_b32 %[t1], 64, %[ka]\n\t"
      "ds_read_b128 %[f1], %[t1] offset:%[i0]\n\t"
      "ds_read_b128 %[f5], %[t1] offset:%[i1]\n\t"
      "ds_read_b128 %[f9], %[t1] offset:%[i2]\n\t"
      "ds_read_b128 %[f13], %[t1] offset:%[i3]\n\t"
      "v_xor_b32 %[t0], 128, %[ka]\n\t"
      "ds_read_b128 %[f2], %[t0] offset:%[i0]\n\t"
      "ds_read_b128 %[f6], %[t0] offset:%[i1]\n\t"
      "ds_read_b128 %[f10], %[t0] offset:%[i2]\n\t"
      "ds_read_b128 %[f14], %[t0] offset:%[i3]\n\t"
      "v_xor_b32 %[t1], 192, %[ka]\n\t"
      "ds_read_b128 %[f3], %[t1] offset:%[i0]\n\t"
      "ds_read_b128 %[f7], %[t1] offset:%[i1]\n\t"
      "ds_read_b128 %[f11], %[t1] offset:%[i2]\n\t"
      "ds_read_b128 %[f15], %[t1] offset:%[i3]"
      : [t0] "=&v"(t0), [t1] "=&v"(t1),
        [f0] "=&a"(kf[0]), [f1] "=&a"(kf[1]), [f2] "=&a"(kf[2]), [f3] "=&a"(kf[3]), [f4]
        "=&a"(kf[4]), [f5] "=&a"(kf[5]), [f6] "=&a"(kf[6]), [f7] "=&a"(kf[7]), [f8]
        "=&a"(kf[8]), [f9] "=&a"(kf[9]), [f10] "=&a"(kf[10]), [f11] "=&a"(kf[11]), [f12]
        "=&a"(kf[12]), [f13] "=&a"(kf[13]), [f14] "=&a"(kf[14]), [f15] "=&a"(kf[15])
      : [ka] "v"(k_addr), [i0] "i"(kImm), [i1] "i"(kImm + 256), [i2] "i"(kImm + 512),
        [i3] "i"(kImm + 768));
}
// Issue position of k-step s in d512_read_block.
constexpr int d512BlockPos(int s) { return 4 * (s & 3) + (s >> 2); }
template <int kStep>
__device__ __forceinline__ void d512_block_ready(u32x4v_t &f) {
  asm volatile("s_waitcnt lgkmcnt(%[n])" : "+a"(f) : [n] "i"(15 - d512BlockPos(kStep)));
}
// Half of the 16 K-fragment reads of one 16-key score block into AGPRs, all
// eight in flight before their first MFMA. For lane key k (k & 15 = lane & 15)
// and lane group g, k-step s sits at chunk (4s + g) ^ (k & 15) of the key's
// row: bits 0-1 of the chunk are g ^ (k & 3), bits 2-3 are (s & 3) ^
// ((k >> 2) & 3) and bits 4+ are s >> 2. So with base = the address of k-step
// 0, k-step s is at (base ^ (64 (s & 3))) + 256 (s >> 2): two XORed addresses
// per half, four immediate offsets each. Fragment i of half kHalf is k-step
// 2 kHalf + i / 4 + 4 (i % 4).
template <int kHalf>
__device__ __forceinline__ void d512_read_kfrags(uint32_t k_addr, u32x4v_t (&kf)[8]) {
  uint32_t t0, t1;
  asm volatile(
      "s_waitcnt lgkmcnt(0)\n\t"
      "v_xor_b32 %[t0], %[x0], %[ka]\n\t"
      "ds_read_b128 %[f0], %[t0] offset:%[i0]\n\t"
      "ds_read_b128 %[f1], %[t0] offset:%[i1]\n\t"
      "ds_read_b128 %[f2], %[t0] offset:%[i2]\n\t"
      "ds_read_b128 %[f3], %[t0] offset:%[i3]\n\t"
      "v_xor_b32 %[t1], %[x1], %[ka]\n\t"
      "ds_read_b128 %[f4], %[t1] offset:%[i0]\n\t"
      "ds_read_b128 %[f5], %[t1] offset:%[i1]\n\t"
      "ds_read_b128 %[f6], %[t1] offset:%[i2]\n\t"
      "ds_read_b128 %[f7], %[t1] offset:%[i3]"
      : [t0] "=&v"(t0), [t1] "=&v"(t1), [f0] "=&a"(kf[0]), [f1] "=&a"(kf[1]), [f2] "=&a"(kf[2]),
        [f3] "=&a"(kf[3]), [f4] "=&a"(kf[4]), [f5] "=&a"(kf[5]), [f6] "=&a"(kf[6]), [f7]
        "=&a"(kf[7])
      : [ka] "v"(k_addr), [x0] "i"(128 * kHalf), [x1] "i"(128 * kHalf + 64), [i0] "i"(0),
        [i1] "i"(256), [i2] "i"(512), [i3] "i"(768));
}
template <int kPos>
__device__ __forceinline__ void d512_kfrag_ready(u32x4v_t &f) {
  asm volatile("s_waitcnt lgkmcnt(%[n])" : "+a"(f) : [n] "i"(7 - kPos));
}
template <int kBegin, int kEnd, class F>
__device__ __forceinline__ void d512_static_for(F &&f) {
  if constexpr (kBegin < kEnd) {
    f(std::integral_constant<int, kBegin>{});
    d512_static_for<kBegin + 1, kEnd>(f);
  }
}

__global__ __launch_bounds__(kD512Threads) void prefill_d512_kernel(D512Params p) {
  constexpr int KS = kD512 / 32;  // 32-dim k-steps of S^T
  // Two stages of K and V tiles (32 keys x 1 KiB each), and what the waves
  // trade, by the parity of the tile: each row's maxima over a wave's 16 keys,
  // the probabilities as B operands (one wave's keys in each half), the
  // rescale of the row's accumulators where its maximum moved; at the end the
  // rows' sums.
  struct Lds {
    uint4 k[2][kD512Tile * kD512Chunks];
    uint4 v[2][kD512Tile * kD512Chunks];
    uint2 p[2][kD512Rows][kWave][2];
    float max[2][kD512Rows][2][kQueryHeads];
    float alpha[2][kD512Rows][kQueryHeads];
    int32_t moved[2][kD512Rows];
    float sum[kD512Rows][2][kQueryHeads];
  };
  __shared__ __attribute__((aligned(1024))) Lds lds;

  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = wave_uniform(t >> 6);
  const int my_row = wave >> 1;  // row of the workgroup
  const int blk = wave & 1;      // its 16 keys of every tile
  const int head = lane & 15;    // MFMA column
  const int g = lane >> 4;       // lane group: keys / dims 4g..4g+3 of the accumulator
  const int b = blockIdx.y;
  const int L = p.seq_len;
  // Causal work grows with the row: the last rows are dispatched first, so
  // the workgroups of the first rows fill the CUs that free up early
  // (longest-first order; one workgroup per CU at a time).
  const int r0 = (gridDim.x - 1 - blockIdx.x) * kD512Rows;
  const int row = r0 + my_row;
  const int last_key = min(r0 + kD512Rows, L) - 1;  // last key any row of the workgroup sees

  // Q^T operand: lane holds Q[row][head][32 s + 8 g .. +8] for k-step s. A row
  // past the sequence computes the last one's scores and is not stored.
  uint4 qreg[KS];
  {
    const uint16_t *qrow =
        p.q + (((int64_t)b * L + min(row, L - 1)) * kQueryHeads + head) * kD512 + 8 * g;
#pragma unroll
    for (int s = 0; s < KS; ++s) qreg[s] = load128(qrow + 32 * s);
    // Q lives in AGPRs (an MFMA operand may be an AGPR); all loads are
    // issued before the first constraint forces a wait.
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      u32x4v_t t4 = {qreg[s].x, qreg[s].y, qreg[s].z, qreg[s].w};
      asm volatile("" : "+a"(t4));
      qreg[s] = make_uint4(t4.x, t4.y, t4.z, t4.w);
    }
  }

  float m_run = -INFINITY, l_run = 0.0f;  // of this wave's row
  f32x4_t acc[kD512Rows][kD512Blocks];    // every row's, this wave's dims
#pragma unroll
  for (int r = 0; r < kD512Rows; ++r)
#pragma unroll
    for (int d = 0; d < kD512Blocks; ++d) acc[r][d] = f32x4_t{};

  const uint64_t kseq = reinterpret_cast<uint64_t>(p.k + (int64_t)b * L * kD512);
  const uint64_t vseq = reinterpret_cast<uint64_t>(p.v + (int64_t)b * L * kD512);
  const int n_tiles = last_key / kD512Tile + 1;
  // Copy of a tile into a stage: wave w copies keys 4w .. 4w+3, one 1 KiB row
  // per copy; lane l fills LDS chunk l with the swizzled source chunk. Past
  // the sequence's end its last row is repeated (and masked). All but one XOR
  // per row is scalar: the registers are full.
  constexpr int kCopyRows = kD512Tile / kD512Waves;
  constexpr int kPairs = kCopyRows / 2;
  constexpr int kStageBytes = kD512Tile * kD512RowBytes;
  const uint32_t lane_bytes = lane * 16;
  const uint32_t k_dst = wave_uniform(lds_address(&lds.k[0][kCopyRows * wave * kD512Chunks]));
  const uint32_t v_dst = wave_uniform(lds_address(&lds.v[0][kCopyRows * wave * kD512Chunks]));
  auto row_base = [&](uint64_t seq, int kt, int key) __attribute__((always_inline)) {
    return seq + (uint64_t)(uint32_t)min(kt + key, L - 1) * kD512RowBytes;
  };
  auto copy_k = [&](int kt, int stage, int i) __attribute__((always_inline)) {
    const int key = kCopyRows * wave + 2 * i;
    copy_lanes2(row_base(kseq, kt, key), lane_bytes ^ (16 * (key & 15)),
                row_base(kseq, kt, key + 1), lane_bytes ^ (16 * ((key + 1) & 15)),
                k_dst + stage * kStageBytes + i * 2 * kD512RowBytes);
  };
  auto copy_v = [&](int kt, int stage, int i) __attribute__((always_inline)) {
    const int key = kCopyRows * wave + 2 * i;
    copy_lanes2(row_base(vseq, kt, key), lane_bytes ^ (32 * (key & 7)),
                row_base(vseq, kt, key + 1), lane_bytes ^ (32 * ((key + 1) & 7)),
                v_dst + stage * kStageBytes + i * 2 * kD512RowBytes);
  };
  const int k15 = lane & 15;
  const uint32_t k_base = lds_address(&lds.k[0][0]) + (16 * blk + k15) * kD512RowBytes +
                          16 * (g ^ (k15 & 3)) + 64 * ((k15 >> 2) & 3);
  // V^T operand of dim block d: lane i of group g reads rows k0 + j,
  // dims 16 d + 4 q (j = (lane % 16) / 4, q = lane % 4) with k0 = 4 g and
  // 16 + 4 g; chunk 2 (4 wave + d) + q / 2 of a row at c ^ 2 (row % 8).
  const int vj = (lane & 15) >> 2, vq = lane & 3;
  const int v_row = 4 * g + vj;  // and 16 + 4 g + vj, the same modulo 8
  const int v_lane = v_row * kD512RowBytes + (wave >> 1) * 256 + ((vq >> 1) << 4) + ((vq & 1) << 3);

  // Three tiles are in work at once, so that an iteration needs one barrier
  // and its parts do not wait for each other: scores of tile it, softmax of
  // tile it - 1 (whose maxima the barrier made known to both waves of a row),
  // P.V of tile it - 2. Tiles -1 and -2 have probability 0 and meet zeroed V
  // stages; past the last tile every key is masked.
#pragma unroll
  for (int i = 0; i < kPairs; ++i) copy_k(0, 0, i);
  for (int i = t; i < 2 * kD512Tile * kD512Chunks; i += kD512Threads)
    lds.v[0][i] = make_uint4(0, 0, 0, 0);
  lds.p[0][my_row][lane][blk] = make_uint2(0, 0);
  if (lane < kQueryHeads) lds.max[1][my_row][blk][lane] = -INFINITY;
  if (lane == 0) lds.moved[0][my_row] = 0;
  float sc[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};  // of tile it - 1

#pragma unroll 1
  for (int it = 0; it < n_tiles + 2; ++it) {
    const int S = it & 1;  // parity of tiles it and it - 2
    // Each wave waits for its own copies, the barrier for all: K of tile it,
    // V of tile it - 2; and every wave is done with iteration it - 1.
    wait_copies();
    lds_barrier();
    const float other_max = lds.max[S ^ 1][my_row][blk ^ 1][head];
    const float own_max = lds.max[S ^ 1][my_row][blk][head];
    int32_t moved[kD512Rows];
    uint4 pb[kD512Rows];
#pragma unroll
    for (int r = 0; r < kD512Rows; ++r) {
      moved[r] = lds.moved[S][r];
      pb[r] = *reinterpret_cast<const uint4 *>(&lds.p[S][r][lane][0]);
    }
    auto v_operand = [&](int d) __attribute__((always_inline)) {
      uint2 half_op[2];
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const char *addr = reinterpret_cast<const char *>(lds.v[S]) + v_lane +
                           16 * r * kD512RowBytes +
                           (((kD512Blocks * (wave & 1) + d) ^ (v_row & 7)) << 5);
        typedef __attribute__((address_space(3))) i16x4_t lds_i16x4;
        const i16x4_t tr = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_i16x4 *)(__attribute__((address_space(3))) const char *)(addr));
        half_op[r] = __builtin_bit_cast(uint2, tr);
      }
      return make_uint4(half_op[0].x, half_op[0].y, half_op[1].x, half_op[1].y);
    };
    // P.V of tile it - 2, in two halves around the scores (their operands do
    // not fit the registers together); one V operand serves the four rows.
    uint4 vt[2] = {v_operand(0), v_operand(1)};
#pragma unroll
    for (int r = 0; r < kD512Rows; ++r) {
      if (wave_uniform(moved[r]) == 0) continue;
      const float alpha = lds.alpha[S][r][head];
#pragma unroll
      for (int d = 0; d < kD512Blocks; ++d) acc[r][d] *= alpha;
    }
    // Scores of tile it, half of the k-steps at a time: the fragments arrive
    // under the P.V and the softmax. The copies of K of tile it + 1 and V of
    // tile it - 1 ride on the MFMAs (the last K tile is copied again, unread:
    // no branch around those).
    const int kt = it * kD512Tile;
    const int next_k = min(it + 1, n_tiles - 1) * kD512Tile;
    const int next_v = min(it - 1, n_tiles - 1) * kD512Tile;
    f32x4_t s2[2] = {f32x4_t{}, f32x4_t{}};
    auto score_half = [&](auto hc, u32x4v_t (&kf)[8]) __attribute__((always_inline)) {
      constexpr int kHalf = decltype(hc)::value;
      d512_static_for<0, 8>([&](auto pc) __attribute__((always_inline)) {
        constexpr int pos = decltype(pc)::value;
        constexpr int s = 2 * kHalf + pos / 4 + 4 * (pos % 4);
        d512_kfrag_ready<pos>(kf[pos]);
        s2[pos & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(bf16x8_t, kf[pos]), __builtin_bit_cast(bf16x8_t, qreg[s]),
            s2[pos & 1], 0, 0, 0);
        if constexpr (kHalf == 0 && pos % 4 == 1) {
          if (next_v >= 0) copy_v(next_v, S ^ 1, pos / 4);
        }
        if constexpr (kHalf == 1 && pos % 4 == 1) copy_k(next_k, S ^ 1, pos / 4);
        // Keep each fragment's wait right before its MFMA: without this
        // fence the scheduler issued all the waits first, one lgkmcnt(0) in
        // effect, and the reads no longer overlapped the MFMAs.
        __builtin_amdgcn_sched_barrier(0);
      });
    };
    u32x4v_t kf[8];
    d512_read_kfrags<0>(k_base + S * kStageBytes, kf);
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int r = 0; r < kD512Rows; ++r) acc[r][d] = mfma16(vt[d], pb[r], acc[r][d]);

    score_half(std::integral_constant<int, 0>{}, kf);
    d512_read_kfrags<1>(k_base + S * kStageBytes, kf);

    // Softmax of tile it - 1.
    const float tmax = fmaxf(own_max, other_max) * p.q_scale;
    const bool moves = __builtin_amdgcn_ballot_w64(tmax > m_run + kD512Slack) != 0;
    if (moves) {
      const float m_new = fmaxf(m_run, tmax);
      const float alpha = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_new);
      l_run *= alpha;
      m_run = m_new;
      if (lane < kQueryHeads) lds.alpha[S ^ 1][my_row][lane] = alpha;  // the same from both waves
    }
    const float m_use = m_run == -INFINITY ? 0.0f : m_run;
    float pr[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      pr[j] = __builtin_amdgcn_exp2f(fmaf(sc[j], p.q_scale, -m_use));
      l_run += pr[j];
    }
    lds.p[S ^ 1][my_row][lane][blk] =
        make_uint2(cvt_pk_bf16(pr[0], pr[1]), cvt_pk_bf16(pr[2], pr[3]));
    if (lane == 0) lds.moved[S ^ 1][my_row] = moves ? 1 : 0;

    score_half(std::integral_constant<int, 1>{}, kf);
    // Lane holds head `head`, keys 16 blk + 4 g + i.
#pragma unroll
    for (int d = 0; d < 2; ++d) vt[d] = v_operand(2 + d);
    const f32x4_t score = s2[0] + s2[1];
    float smax = -INFINITY;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      sc[j] = kt + 16 * blk + 4 * g + j <= row ? score[j] : -INFINITY;
      smax = fmaxf(smax, sc[j]);
    }
    smax = xor_max<16>(smax);
    smax = xor_max<32>(smax);
    if (lane < kQueryHeads) lds.max[S][my_row][blk][lane] = smax;
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int r = 0; r < kD512Rows; ++r) acc[r][2 + d] = mfma16(vt[d], pb[r], acc[r][2 + d]);
  }
  static_assert(kPairs == 2, "two pairs of copies per operand");

  wait_copies();  // no copy may still be writing LDS when the workgroup exits

  // Normalise and store: lane holds head `head`, dims
  // 16 (wave * kD512Blocks + d) + 4 g + i of every row.
  l_run = xor_sum<16>(l_run);
  l_run = xor_sum<32>(l_run);
  if (lane < kQueryHeads) lds.sum[my_row][blk][lane] = l_run;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kD512Rows; ++r) {
    if (r0 + r >= L) break;
    const float sum = lds.sum[r][0][head] + lds.sum[r][1][head];
    const float inv = sum > 0.0f ? 1.0f / sum : 0.0f;
    uint16_t *orow = p.out + (((int64_t)b * L + r0 + r) * kQueryHeads + head) * kD512 +
                     wave * kD512Blocks * 16 + 4 * g;
#pragma unroll
    for (int d = 0; d < kD512Blocks; ++d) {
      const f32x4_t o = acc[r][d] * inv;
      *reinterpret_cast<uint2 *>(orow + 16 * d) =
          make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
    }
  }
}

// The short form: one wave per row, no exchange between waves.
__global__ __launch_bounds__(kD512ShortThreads, 1) void prefill_d512_short_kernel(D512Params p) {
  constexpr int KS = kD512 / 32;  // 32-dim k-steps of S^T
  constexpr int DB = kD512 / 16;  // 16-dim blocks of O^T
  // Two stages of K and V tiles (32 keys x 1 KiB each).
  struct Lds {
    uint4 k[2][kD512Tile * kD512Chunks];
    uint4 v[2][kD512Tile * kD512Chunks];
  };
  __shared__ __attribute__((aligned(1024))) Lds lds;

  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = wave_uniform(t >> 6);
  const int head = lane & 15;   // MFMA column
  const int g = lane >> 4;      // lane group: keys / dims 4g..4g+3 of the accumulator
  const int b = blockIdx.y;
  const int L = p.seq_len;
  // Causal work grows with the row: the last rows are dispatched first, so
  // the workgroups of the first rows fill the CUs that free up early
  // (longest-first order; one workgroup per CU at a time).
  const int r0 = (gridDim.x - 1 - blockIdx.x) * kD512Rows;
  const int row = r0 + wave;
  const bool row_ok = row < L;
  const int last_key = min(r0 + kD512Rows, L) - 1;  // last key any row of the workgroup sees

  // Q^T operand: lane holds Q[row][head][32 s + 8 g .. +8] for k-step s.
  uint4 qreg[KS];
  {
    const uint16_t *qrow = p.q + (((int64_t)b * L + (row_ok ? row : 0)) * kQueryHeads + head) * kD512;
#pragma unroll
    for (int s = 0; s < KS; ++s)
      qreg[s] = row_ok ? load128(qrow + 32 * s + 8 * g) : make_uint4(0, 0, 0, 0);
    // Q lives in AGPRs (an MFMA operand may be an AGPR); all loads are
    // issued before the first constraint forces a wait.
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      u32x4v_t t4 = {qreg[s].x, qreg[s].y, qreg[s].z, qreg[s].w};
      asm volatile("" : "+a"(t4));
      qreg[s] = make_uint4(t4.x, t4.y, t4.z, t4.w);
    }
  }

  float m_run = -INFINITY, l_run = 0.0f;
  f32x4_t acc[DB];
#pragma unroll
  for (int d = 0; d < DB; ++d) acc[d] = f32x4_t{};

  const uint16_t *kseq = p.k + (int64_t)b * L * kD512;
  const uint16_t *vseq = p.v + (int64_t)b * L * kD512;
  const int n_tiles = last_key / kD512Tile + 1;
  // Copy of a tile into a stage: wave w copies keys 8w .. 8w+7, one 1 KiB
  // row per copy; lane l fills LDS chunk l with the swizzled source chunk.
  constexpr int kCopyRows = kD512Tile / (kD512ShortThreads / kWave);
  auto copy_tile = [&](int kt, int stage) {
#pragma unroll
    for (int i = 0; i < kCopyRows; ++i) {
      const int key = kCopyRows * wave + i;
      const int64_t src_row = (int64_t)min(kt + key, L - 1) * kD512;  // past the end: masked
      const uint32_t dk = lds_address(&lds.k[stage][key * kD512Chunks]);
      const uint32_t dv = lds_address(&lds.v[stage][key * kD512Chunks]);
      copy_row_pair(reinterpret_cast<uint64_t>(kseq + src_row + 8 * (lane ^ (key & 15))),
                    wave_uniform(dk));
      copy_row_pair(reinterpret_cast<uint64_t>(vseq + src_row + 8 * (lane ^ ((key & 7) << 1))),
                    wave_uniform(dv));
    }
  };
  const int k15 = lane & 15;
  const uint32_t k_base = lds_address(&lds.k[0][0]) + k15 * kD512RowBytes +
                          16 * (g ^ (k15 & 3)) + 64 * ((k15 >> 2) & 3);
  constexpr int kStageBytes = kD512Tile * kD512RowBytes;
  copy_tile(0, 0);
  for (int tile = 0; tile < n_tiles; ++tile) {
    const int kt = tile * kD512Tile;
    const int stage = tile & 1;
    // Tile `tile` copied (each wave waits for its own copies, the barrier for
    // all); every wave is done with tile-1, so the other stage is free.
    wait_copies();
    __syncthreads();
    if (tile + 1 < n_tiles) copy_tile(kt + kD512Tile, stage ^ 1);
    if (!row_ok || kt > row) continue;  // uniform per wave
    const uint4 *s_v = lds.v[stage];

    // Scores of the two 16-key blocks: lane holds head `head`, keys
    // 16 blk + 4 g + i.
    f32x4_t sblk[2];
    auto score_block = [&](auto st, auto bl) __attribute__((always_inline)) {
      constexpr int kImm =
          decltype(st)::value * kStageBytes + decltype(bl)::value * 16 * kD512RowBytes;
      u32x4v_t kf[16];
      d512_read_block<kImm>(k_base, kf);
      f32x4_t s2[2] = {f32x4_t{}, f32x4_t{}};
      d512_static_for<0, 16>([&](auto pc) __attribute__((always_inline)) {
        constexpr int pos = decltype(pc)::value;
        constexpr int s = 4 * (pos & 3) + (pos >> 2);  // k-step at issue position pos
        d512_block_ready<s>(kf[s]);
        s2[pos & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(bf16x8_t, kf[s]), __builtin_bit_cast(bf16x8_t, qreg[s]),
            s2[pos & 1], 0, 0, 0);
        // Keep each fragment's wait right before its MFMA: without this
        // fence the scheduler issued all sixteen waits first, one
        // lgkmcnt(0) in effect, and the reads no longer overlapped the
        // MFMAs.
        __builtin_amdgcn_sched_barrier(0);
      });
      return s2[0] + s2[1];
    };
    if (stage == 0) {
      sblk[0] = score_block(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{});
      sblk[1] = score_block(std::integral_constant<int, 0>{}, std::integral_constant<int, 1>{});
    } else {
      sblk[0] = score_block(std::integral_constant<int, 1>{}, std::integral_constant<int, 0>{});
      sblk[1] = score_block(std::integral_constant<int, 1>{}, std::integral_constant<int, 1>{});
    }
    float sc[8];
    float tmax = -INFINITY;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int kp = kt + 16 * (j / 4) + 4 * g + (j % 4);
      const float x = sblk[j / 4][j % 4];
      sc[j] = kp <= row ? x : -INFINITY;
      tmax = fmaxf(tmax, sc[j]);
    }
    tmax = xor_max<16>(tmax);
    tmax = xor_max<32>(tmax) * p.q_scale;
    if (__builtin_amdgcn_ballot_w64(tmax > m_run + kD512Slack) != 0) {
      const float m_new = fmaxf(m_run, tmax);
      const float alpha = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_new);
      l_run *= alpha;
#pragma unroll
      for (int d = 0; d < DB; ++d) acc[d] *= alpha;
      m_run = m_new;
    }
    const float m_use = m_run == -INFINITY ? 0.0f : m_run;
    uint32_t pw[4];
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
      const float p0 = __builtin_amdgcn_exp2f(fmaf(sc[j], p.q_scale, -m_use));
      const float p1 = __builtin_amdgcn_exp2f(fmaf(sc[j + 1], p.q_scale, -m_use));
      l_run += p0 + p1;
      pw[j / 2] = cvt_pk_bf16(p0, p1);
    }
    const uint4 pb = make_uint4(pw[0], pw[1], pw[2], pw[3]);
    // V^T operand of dim block d: lane i of group g reads rows k0 + j,
    // dims 16 d + 4 q (j = (lane % 16) / 4, q = lane % 4) with k0 = 4 g
    // and 16 + 4 g.
    const int vj = (lane & 15) >> 2;
    const int vq = lane & 3;
#pragma unroll
    for (int d = 0; d < DB; ++d) {
      uint2 half_op[2];
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const int vrow = 16 * r + 4 * g + vj;
        const int c = 2 * d + (vq >> 1);
        const char *addr = reinterpret_cast<const char *>(s_v) + vrow * kD512RowBytes +
                           ((c ^ ((vrow & 7) << 1)) << 4) + ((vq & 1) << 3);
        typedef __attribute__((address_space(3))) i16x4_t lds_i16x4;
        const i16x4_t tr = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_i16x4 *)(__attribute__((address_space(3))) const char *)(addr));
        half_op[r] = __builtin_bit_cast(uint2, tr);
      }
      acc[d] = mfma16(make_uint4(half_op[0].x, half_op[0].y, half_op[1].x, half_op[1].y), pb,
                      acc[d]);
    }
    // Keep the transposing V reads kD512VLead MFMAs ahead of their MFMA
    // (measured: 2 ahead 171 us, 4 ahead 164 us, 6 ahead 164.7 us for the
    // 2048-row launcher).
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * kD512VLead, 1);
#pragma unroll
    for (int i = 0; i < DB - kD512VLead; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 1);  // 1 MFMA
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);  // its successor's 2 reads
    }
    __builtin_amdgcn_sched_group_barrier(0x008, kD512VLead, 1);
  }

  wait_copies();  // no copy may still be writing LDS when the workgroup exits

  // Normalise and store: lane holds head `head`, dims 16 d + 4 g + i.
  l_run = xor_sum<16>(l_run);
  l_run = xor_sum<32>(l_run);
  if (!row_ok) return;
  const float inv = l_run > 0.0f ? 1.0f / l_run : 0.0f;
  uint16_t *orow = p.out + (((int64_t)b * L + row) * kQueryHeads + head) * kD512;
#pragma unroll
  for (int d = 0; d < DB; ++d) {
    uint2 o;
    o.x = pack_bf16x2(acc[d][0] * inv, acc[d][1] * inv);
    o.y = pack_bf16x2(acc[d][2] * inv, acc[d][3] * inv);
    *reinterpret_cast<uint2 *>(orow + 16 * d + 4 * g) = o;
  }
}

static_assert(kD512Tile % kD512Rows == 0, "a workgroup's rows see the same tiles");
static_assert(kD512Blocks == 4, "two waves' blocks are one period of V's swizzle");

bool prefill_args_ok(const void *out, const void *qp, const void *kp, const void *vp,
                     const void *q, const void *k, const void *position, int batch_size,
                     int seqlen_q, int seqlen_k) {
  // src/gemma4_flash_attention_prefill.cu:1131-1138, 1199-1205
  return batch_size > 0 && seqlen_q > 0 && seqlen_q == seqlen_k && out != nullptr &&
         qp != nullptr && kp != nullptr && vp != nullptr && q != nullptr && k != nullptr &&
         position != nullptr && (int64_t)batch_size * seqlen_q <= 0x7fffffff;
}

}  // namespace
}  // namespace gemma4

using namespace gemma4;

extern "C" hipError_t gemma4_flash_attention_sliding_fwd_bf16_norm_rope(
    gemma4_bf16 *d_out, gemma4_bf16 *d_q_prepared, gemma4_bf16 *d_k_prepared,
    gemma4_bf16 *d_v_prepared, const gemma4_bf16 *d_q, const gemma4_bf16 *d_k,
    const gemma4_bf16 *d_v, const gemma4_bf16 *d_q_norm_weight,
    const gemma4_bf16 *d_k_norm_weight, const float *d_cos, const float *d_sin,
    const int32_t *d_token_position, int batch_size, int seqlen_q, int seqlen_k, int window_size,
    float softmax_scale, hipStream_t stream) {
  if (!prefill_args_ok(d_out, d_q_prepared, d_k_prepared, d_v_prepared, d_q, d_k,
                       d_token_position, batch_size, seqlen_q, seqlen_k) ||
      window_size <= 0 || d_v == nullptr || d_q_norm_weight == nullptr ||
      d_k_norm_weight == nullptr || d_cos == nullptr || d_sin == nullptr) {
    return hipErrorInvalidValue;
  }
  PrefillPrepParams pp{};
  pp.q_prepared = reinterpret_cast<uint16_t *>(d_q_prepared);
  pp.k_prepared = reinterpret_cast<uint16_t *>(d_k_prepared);
  pp.v_prepared = reinterpret_cast<uint16_t *>(d_v_prepared);
  pp.q = reinterpret_cast<const uint16_t *>(d_q);
  pp.k = reinterpret_cast<const uint16_t *>(d_k);
  pp.v = reinterpret_cast<const uint16_t *>(d_v);
  pp.q_norm_weight = reinterpret_cast<const uint16_t *>(d_q_norm_weight);
  pp.k_norm_weight = reinterpret_cast<const uint16_t *>(d_k_norm_weight);
  pp.cos = d_cos;
  pp.sin = d_sin;
  pp.token_position = d_token_position;
  // 8x256 geometry: RoPE over the whole head, V projection present.
  const int64_t rows = (int64_t)batch_size * seqlen_q;
  hipLaunchKernelGGL((prefill_prep_kernel<8, 256, 256, true>),
                     dim3((rows + kPrepRows - 1) / kPrepRows, 8),
                     dim3(prep_waves<8, true>() * kWave), 0, stream, pp, rows);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
  // Attention over the prepared rows: the chunk kernel without a prior
  // context (only num_heads, head_dim and window_size of the config are read).
  Gemma4KvCacheConfig c{};
  c.num_layers = 1;
  c.num_heads = 8;
  c.head_dim = 256;
  c.window_size = window_size;
  return gemma4_flash_attention_prefill_chunk_paged_bf16(
      d_out, d_q_prepared, d_k_prepared, d_v_prepared, nullptr, nullptr, nullptr, nullptr, c, 0,
      batch_size, seqlen_q, softmax_scale, stream);
}

extern "C" hipError_t gemma4_flash_attention_global_fwd_bf16_norm_rope(
    gemma4_bf16 *d_out, gemma4_bf16 *d_q_prepared, gemma4_bf16 *d_k_prepared,
    gemma4_bf16 *d_v_prepared, const gemma4_bf16 *d_q, const gemma4_bf16 *d_k,
    const gemma4_bf16 *d_q_norm_weight, const gemma4_bf16 *d_k_norm_weight, const float *d_cos,
    const float *d_sin, const int32_t *d_token_position, int batch_size, int seqlen_q,
    int seqlen_k, float softmax_scale, hipStream_t stream) {
  if (!prefill_args_ok(d_out, d_q_prepared, d_k_prepared, d_v_prepared, d_q, d_k,
                       d_token_position, batch_size, seqlen_q, seqlen_k) ||
      d_q_norm_weight == nullptr || d_k_norm_weight == nullptr || d_cos == nullptr ||
      d_sin == nullptr || batch_size > 65535 || !(softmax_scale > 0.0f)) {
    return hipErrorInvalidValue;
  }
  PrefillPrepParams pp{};
  pp.q_prepared = reinterpret_cast<uint16_t *>(d_q_prepared);
  pp.k_prepared = reinterpret_cast<uint16_t *>(d_k_prepared);
  pp.v_prepared = reinterpret_cast<uint16_t *>(d_v_prepared);
  pp.q = reinterpret_cast<const uint16_t *>(d_q);
  pp.k = reinterpret_cast<const uint16_t *>(d_k);
  pp.v = nullptr;
  pp.q_norm_weight = reinterpret_cast<const uint16_t *>(d_q_norm_weight);
  pp.k_norm_weight = reinterpret_cast<const uint16_t *>(d_k_norm_weight);
  pp.cos = d_cos;
  pp.sin = d_sin;
  pp.token_position = d_token_position;
  // 1x512 geometry: RoPE over a quarter of the head, V from the raw K.
  const int64_t rows = (int64_t)batch_size * seqlen_q;
  hipLaunchKernelGGL((prefill_prep_kernel<1, 512, 128, false>),
                     dim3((rows + kPrepRows - 1) / kPrepRows, 1),
                     dim3(prep_waves<1, false>() * kWave), 0, stream, pp, rows);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
  D512Params ap{};
  ap.out = reinterpret_cast<uint16_t *>(d_out);
  ap.q = reinterpret_cast<const uint16_t *>(d_q_prepared);
  ap.k = reinterpret_cast<const uint16_t *>(d_k_prepared);
  ap.v = reinterpret_cast<const uint16_t *>(d_v_prepared);
  ap.seq_len = seqlen_q;
  ap.q_scale = softmax_scale * kLog2e;
  const dim3 grid((seqlen_q + kD512Rows - 1) / kD512Rows, batch_size);
  if (seqlen_q <= kD512ShortRows) {
    hipLaunchKernelGGL(prefill_d512_short_kernel, grid, dim3(kD512ShortThreads), 0, stream, ap);
  } else {
    hipLaunchKernelGGL(prefill_d512_kernel, grid, dim3(kD512Threads), 0, stream, ap);
  }
  return hipGetLastError();
}
