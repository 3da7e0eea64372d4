// Split phase of the paged decode attention for the 1 x 512 geometry (one KV
// head under all 16 query heads) on bf16 MFMA, gfx950, with the optional fused
// append and preparation. Replaces the same phases as decode_split_kernel
// (src/gemma4_flash_attention_decode.cu:691-878, 216-375) for that geometry;
// the combine launch is the one in decode_attention.hip.
//
// Sixteen query heads over one key are a dense 16-row contraction, 16 K
// multiply-adds per key: on v_dot2 that arithmetic, not the 2 KiB of K and V
// per key, set the time. On MFMA it is a tenth of the streaming time.
//
// Workgroup (split, batch) of kWaves waves; a step is 16 keys per wave.
//   S^T = K Q^T    v_mfma_f32_16x16x32_bf16, 16 k-steps of 32 dims, each wave
//                  its own 16 keys. Lane (g, h) = (l / 16, l % 16) supplies
//                  K[key h][32 s + 8 g ..] and Q[head h][32 s + 8 g ..] (held
//                  in registers), and receives head h's scores of keys
//                  4 g .. 4 g + 3.
//   softmax        the waves trade their heads' maxima through LDS, so all
//                  weigh the step's keys against one running maximum; the
//                  accumulators are rescaled only if a head's maximum moved.
//   O^T += V^T P^T the same MFMA, each wave its own 512 / kWaves dims over
//                  the step's keys of all waves, two waves' keys at a time:
//                  the four probabilities a lane holds are half a B operand
//                  as they stand and travel through LDS that way; V^T comes from the
//                  row-major tiles by ds_read_b64_tr_b16. Lane (g, h)
//                  accumulates dims 16 d + 4 g .. + 3 of head h. Splitting
//                  the dims and not the keys here leaves nothing to merge at
//                  the end: merging four waves' 512 x 16 accumulators through
//                  LDS took 3.6 us of a 12 us launch (8193 keys in splits of
//                  48).
// Measured (MI355X), before (v_dot2 kernel) and now: one sequence of 8193 keys
// in 171 splits of 48, launch 19.1 -> 8.7 us (in the kernel 6.2: 0.8 to the
// first words, 2.4 until K has arrived and q is prepared, 1.3 scores to P.V,
// 1 for the partial stores; with V requested before q's preparation instead
// of after it, 7.2); 24 sequences of 200-12001 keys, 302 MB, 199 -> 64 us.
// Waves and splits: a split of up to 64 keys is one step of four waves. Longer
// ones run on two waves in 69 KiB of LDS, so that a CU holds two workgroups
// and one streams while the other starts, scores or stores (24 sequences in
// splits of 128 / 512: 93 / 82 us against 112 / 86 on four waves). With split
// counters always four: they share out the sixteen heads that the last
// workgroup folds (8193 keys in 65 splits of 128: 65 us, on two waves 90;
// 20000 in 250 of 80: 186 / 274; 24 sequences in splits of 512: 88 / 94).
// K and V rows are copied into the wave's own 32 KiB of LDS with
// global_load_lds (1 KiB, one whole row, per instruction; chunk c of key k at
// c ^ k for K and c ^ 2 (k % 8) for V, so that the operand reads are free of
// bank conflicts). The K copies of the next step go out as soon as the scores
// of this one are done, its V copies after this step's P.V: 32 KiB per wave
// in flight for all but the arithmetic. The copies are inline asm that the
// compiler does not count; every wait on them is written out here, and the
// loop issues no other vector memory operation.
#include "decode_row.hpp"
#include "gemma4_device.hpp"
#include "lds_copy.hpp"

#include "gemma4_flash_attention.h"

#include <math.h>

namespace gemma4 {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef short i16x4_t __attribute__((ext_vector_type(4)));
typedef unsigned u32x4v_t __attribute__((ext_vector_type(4)));

constexpr int kDim = 512;
constexpr int kTileKeys = kD512TileKeys;
constexpr int kRowBytes = kDim * 2;
constexpr int kRowChunks = kRowBytes / 16;              // 64: one per lane
constexpr int kTileUint4 = kTileKeys * kRowChunks;      // 16 KiB of K (or V)
constexpr int kSteps = kDim / 32;                       // k-steps of S^T
constexpr int kDimBlocks = kDim / 16;                   // blocks of O^T
constexpr int kChunkTiles = kWave / kTileKeys;          // tiles per page lookup
constexpr int kRot = kDim / 4;                          // rotary dims of a global head

// Four whole rows (1 KiB each) into four consecutive LDS rows: 16 bytes per
// lane from base[i] + off[i]. Few scalar instructions per row matter here (a
// wave issues 32 rows before its first wait): M0 is saved once and stepped.
// The bases come from v_readlane: a vector instruction that wrote an SGPR
// needs five wait states before a memory instruction reads it, which the
// compiler does not see for inline asm (the s_nop 4).
__device__ __forceinline__ void copy_rows4(const uint64_t (&base)[4], const uint32_t (&off)[4],
                                           uint32_t lds_addr) {
  uint32_t m0_saved;
  asm volatile(
      "s_mov_b32 %[m0s], m0\n\t"
      "s_mov_b32 m0, %[lds]\n\t"
      "s_nop 4\n\t"
      "global_load_lds_dwordx4 %[o0], %[b0]\n\t"
      "s_add_u32 m0, m0, 1024\n\t"
      "s_nop 0\n\t"  // SALU write of M0 -> LDS DMA reading it: one wait state (gfx9)
      "global_load_lds_dwordx4 %[o1], %[b1]\n\t"
      "s_add_u32 m0, m0, 1024\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %[o2], %[b2]\n\t"
      "s_add_u32 m0, m0, 1024\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %[o3], %[b3]\n\t"
      "s_mov_b32 m0, %[m0s]"
      : [m0s] "=&s"(m0_saved)
      : [lds] "s"(lds_addr), [o0] "v"(off[0]), [o1] "v"(off[1]), [o2] "v"(off[2]),
        [o3] "v"(off[3]), [b0] "s"(base[0]), [b1] "s"(base[1]), [b2] "s"(base[2]),
        [b3] "s"(base[3])
      : "memory", "scc");
}
// Lane `from`'s value of a per-lane 64-bit address, wave-uniform.
__device__ __forceinline__ uint64_t lane_address(uint64_t v, int from) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, from);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), from);
  return ((uint64_t)hi << 32) | lo;
}

template <int kWaves>
__global__ __launch_bounds__(kWaves *kWave, 1) void decode_split_d512_kernel(DecodeParams p) {
  constexpr int kWaveBlocks = kDimBlocks / kWaves;  // 16-dim blocks of O^T per wave
  // Each wave's keys of the step: K, then V.
  __shared__ __attribute__((aligned(1024))) uint4 s_tile[kWaves][2 * kTileUint4];
  __shared__ uint4 s_p[kWaves][kWave];             // their probabilities, as B operands (high, low)
  __shared__ float s_max[kWaves][kQueryHeads];     // and maxima
  __shared__ int32_t s_pages[kWaves][kWave];  // page-table entries of the next lookup
  // q on its way from rows to operands (chunk c of head h at c ^ h): a place
  // of its own in the four-wave workgroup, so that the V copies need not wait
  // for it; the first V tile in the two-wave one, of which two then fit a CU.
  constexpr bool kOwnQ = kWaves == 4;
  __shared__ __attribute__((aligned(1024))) uint4 s_q_own[kOwnQ ? kTileUint4 : 1];
  uint4 *const s_q = kOwnQ ? s_q_own : &s_tile[0][kTileUint4];
  __shared__ __attribute__((aligned(16))) float s_rope[kWaves][2][kRot / 2];  // cos, sin
  __shared__ int32_t s_append[kWave];  // page-table entry of the appended key
  __shared__ float s_l[kWaves][kQueryHeads];
  __shared__ int32_t s_last;

  const int lane = threadIdx.x & (kWave - 1);
  const int wave = wave_uniform(threadIdx.x / kWave);
  const int h = lane & 15;  // key of the K operand, head of the others
  const int g = lane >> 4;
  const Gemma4KvCacheConfig &c = p.c;
  // The arguments come cold from memory: all are asked for here, in one round
  // trip. Left to the compiler, the later ones are read behind the cut below
  // (24 sequences of 1-1500 keys 17.57 us, 17.31 so; one of 100 9.32, 9.26).
  asm volatile("" ::"s"(p.out), "s"(p.q), "s"(p.cache_k), "s"(p.page_table), "s"(p.counters),
               "s"(p.new_k), "s"(p.q_norm_weight), "s"(p.sin), "s"(c.page_size), "s"(p.q_scale),
               "s"(p.gate), "s"(p.balanced));
  int32_t split = blockIdx.y, b = blockIdx.z;
  int32_t split_size = p.split_size;
  const bool balanced = kWaves == 2 && p.balanced != 0;
  if (balanced) {
    // Workgroup n serves the n-th split in sequence order.
    const BalancedCut cut = balanced_cut(p, lane_live_keys(p));
    int32_t upto = cut.splits;  // splits of sequences 0 .. lane
#pragma unroll
    for (int d = 1; d < kWave; d *= 2) {
      const int32_t below = __shfl_up(upto, d);
      upto += lane >= d ? below : 0;
    }
    const int32_t n = blockIdx.x;
    const uint64_t before = __builtin_amdgcn_ballot_w64(upto <= n);
    b = __builtin_popcountll(before);
    if (b >= p.batch) return;
    split = n - (b > 0 ? __builtin_amdgcn_readlane(upto, b - 1) : 0);
    split_size = cut.size;
  }

  // ---- the words and rows that depend on nothing but the arguments are
  // requested together: length, token position, gate, the page-table entries
  // of this wave's first keys (known before the length for a cache without a
  // window), and q.
  const int32_t *tok_src = p.token_position != nullptr ? p.token_position + b : p.seq_lengths + b;
  const int32_t *gate_src = p.gate != nullptr ? p.gate : p.seq_lengths + b;
  const int32_t seq_word = p.seq_lengths[b];
  const int32_t tok_word = *tok_src;
  const int32_t gate_word = *gate_src;
  // Each wave loads its share of the query heads, and all load the token's K
  // and V rows and the norm weights: lane = chunk of the row. V comes from the
  // raw K where there is no V projection (the same row is read twice then: a
  // register copy would wait for the load).
  constexpr int kWaveHeads = kQueryHeads / kWaves;
  const bool prep = p.q_norm_weight != nullptr;
  uint4 q_row[kWaveHeads];
#pragma unroll
  for (int i = 0; i < kWaveHeads; ++i)
    q_row[i] = load128(p.q + ((int64_t)b * kQueryHeads + wave * kWaveHeads + i) * kDim +
                       lane * kPackElems);
  uint4 token_k = make_uint4(0, 0, 0, 0), token_v = token_k, wq = token_k, wk = token_k;
  if (p.token_position != nullptr) {
    const int64_t off = (int64_t)b * kDim + lane * kPackElems;
    token_k = load128(p.new_k + off);
    token_v = load128((p.new_v != nullptr ? p.new_v : p.new_k) + off);
  }
  if (prep) {
    wq = load128(p.q_norm_weight + lane * kPackElems);
    wk = load128(p.k_norm_weight + lane * kPackElems);
  }
  const int32_t pt_row = b * c.max_pages_per_seq;
  // 64-bit: a split past the live ones may lie beyond int32 keys; the entry
  // stays inside the sequence's row.
  const int64_t key0 =
      (int64_t)split * split_size + ((lane / kTileKeys) * kWaves + wave) * kTileKeys + h;
  const int32_t early_key = (int32_t)min(key0, (int64_t)0x7fffffff);
  const int32_t early_page = p.page_table[pt_row + (early_key / c.page_size) % c.max_pages_per_seq];

  const int32_t seq_len = wave_uniform(seq_word);
  const int32_t token_pos = p.token_position != nullptr ? wave_uniform(tok_word) : -1;
  int32_t first = c.window_size > 0 ? seq_len - c.window_size : 0;
  first = first < 0 ? 0 : first;
  // The plan's splits bound the keys, however the launch cuts them.
  const int32_t capacity =
      (int32_t)min((int64_t)p.split_size * p.num_splits, (int64_t)0x7fffffff);
  const int32_t key_count = min(seq_len > first ? seq_len - first : 0, capacity);
  const int32_t live_splits = (key_count + split_size - 1) / split_size;
  const bool direct = p.num_splits == 1;
  const bool combines = kWaves == 4 && p.counters != nullptr;  // see launch_split_d512

  if (p.gate != nullptr && wave_uniform(gate_word) != 0) {
    // A failed step: no append; a direct launch zeroes its rows (the combine
    // kernel zeroes them otherwise).
    if (direct && split == 0) {
      uint16_t *rows = p.out + (int64_t)b * kQueryHeads * kDim;
      for (int e = threadIdx.x; e < kQueryHeads * kRowChunks; e += kWaves * kWave)
        store128(rows + e * kPackElems, make_uint4(0, 0, 0, 0));
    }
    return;
  }

  // ---- the token's append: one split of the sequence owns it (split 0 when
  // the position is not among the live keys). Its attention takes the key
  // from the token's own rows (prepared in registers where they are raw), and
  // its first wave stores them at the end.
  const bool prep_token = prep && token_pos >= 0;
  bool owns = false;
  int32_t new_pos = -1;
  if (p.token_position != nullptr) {
    // The reference's skip rules (append_row); an unmapped page shows in the
    // key's own lookup.
    const bool droppable = token_pos < 0 || b >= c.batch_size ||
                           (c.window_size == 0 && token_pos / c.page_size >= c.max_pages_per_seq);
    const bool in_live = token_pos >= first && token_pos < seq_len;
    owns = !droppable && split == (in_live ? (token_pos - first) / split_size : 0);
    if (owns && in_live) new_pos = token_pos;
  }
  auto store_rows = [&](int32_t physical, uint4 k, uint4 v) __attribute__((always_inline)) {
    if (physical < 0 || physical >= c.num_pages) return;
    const int64_t row =
        ((int64_t)p.layer * c.num_pages + physical) * c.page_size + token_pos % c.page_size;
    store128(p.cache_k + row * kDim + lane * kPackElems, k);
    store128(p.cache_v + row * kDim + lane * kPackElems, v);
  };
  auto token_entry = [&]() -> const int32_t * {
    return p.page_table + pt_row + (token_pos / c.page_size) % c.max_pages_per_seq;
  };

  if (split >= live_splits) {
    if (key_count == 0 && split == 0 && (direct || combines)) {
      // No live key: the row is defined as zeros (src/...decode.cu:733-743).
      uint16_t *rows = p.out + (int64_t)b * kQueryHeads * kDim;
      for (int e = threadIdx.x; e < kQueryHeads * kRowChunks; e += kWaves * kWave)
        store128(rows + e * kPackElems, make_uint4(0, 0, 0, 0));
    }
    if (owns && wave == 0) {
      if (prep) {
        const float *cos_row = p.cos + (int64_t)token_pos * (kRot / 2);
        const float *sin_row = p.sin + (int64_t)token_pos * (kRot / 2);
        token_k = prep_pack<kWave, kRot>(token_k, p.k_norm_weight, cos_row, sin_row, lane);
        token_v = prep_pack<kWave, kRot>(token_v, nullptr, cos_row, sin_row, lane);
      }
      store_rows(*token_entry(), token_k, token_v);
    }
    return;
  }

  // ---- steps; the last ones of the split may leave waves without a key
  const int32_t begin = first + split * split_size;
  const int32_t end = min(first + key_count, begin + split_size);
  const int32_t n_tiles = (end - begin + kTileKeys - 1) / kTileKeys;
  const int32_t n_steps = (n_tiles + kWaves - 1) / kWaves;
  // Key of lane (tile within the lookup, h) of lookup m, at most end - 1.
  auto lookup_key = [&](int32_t m) -> int32_t {
    const uint32_t key =
        (uint32_t)begin + (uint32_t)(((m * kChunkTiles + lane / kTileKeys) * kWaves + wave) * kTileKeys + h);
    return (int32_t)min(key, (uint32_t)end);
  };
  auto page_entry = [&](int32_t m) -> const int32_t * {
    const int32_t key = min(lookup_key(m), end - 1);
    return p.page_table + pt_row + (key / c.page_size) % c.max_pages_per_seq;
  };
  // Cache row of the lane's key: kRowInvalid past the split or on an unmapped
  // page, kRowNewToken for the appended one.
  auto key_row_of = [&](int32_t m, int32_t physical) -> int32_t {
    const int32_t key = lookup_key(m);
    const bool ok = key < end && physical >= 0 && physical < c.num_pages;
    const int32_t row = (p.layer * c.num_pages + physical) * c.page_size + key % c.page_size;
    return !ok ? kRowInvalid : (key == new_pos ? kRowNewToken : row);
  };

  float m_run = -INFINITY, l_run = 0.0f;
  f32x4_t acc[kWaveBlocks];
#pragma unroll
  for (int d = 0; d < kWaveBlocks; ++d) acc[d] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

  const int32_t page0 = c.window_size == 0 ? early_page : *page_entry(0);
  int32_t row_word = key_row_of(0, page0);

  const uint64_t kcache = reinterpret_cast<uint64_t>(p.cache_k);
  const uint64_t vcache = reinterpret_cast<uint64_t>(p.cache_v);
  uint4 *const k_tile = &s_tile[wave][0];
  uint4 *const v_tile = &s_tile[wave][kTileUint4];
  const uint32_t k_lds = wave_uniform(lds_address(k_tile));
  const uint32_t v_lds = wave_uniform(lds_address(v_tile));
  // Row addresses of the lookup's keys, one per lane, and four rows of step
  // j from them. Every copy of a live tile goes out, so the counts in the
  // waits hold: an unreadable key and the appended one copy cache row 0; the
  // first is masked, the other's row is then written from registers.
  uint64_t k_addr, v_addr;
  auto address_rows = [&]() __attribute__((always_inline)) {
    const uint64_t off = (uint64_t)(uint32_t)max(row_word, 0) * kRowBytes;
    k_addr = kcache + off;
    v_addr = vcache + off;
  };
  auto copy_k4 = [&](int32_t j, int i0) __attribute__((always_inline)) {
    const int at = (j % kChunkTiles) * kTileKeys + i0;
    uint64_t base[4];
    uint32_t off[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      base[i] = lane_address(k_addr, at + i);
      off[i] = (uint32_t)(lane ^ (i0 + i)) * 16;
    }
    copy_rows4(base, off, k_lds + i0 * kRowBytes);
  };
  auto copy_v4 = [&](int32_t j, int i0) __attribute__((always_inline)) {
    const int at = (j % kChunkTiles) * kTileKeys + i0;
    uint64_t base[4];
    uint32_t off[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      base[i] = lane_address(v_addr, at + i);
      off[i] = (uint32_t)(lane ^ (((i0 + i) & 7) << 1)) * 16;
    }
    copy_rows4(base, off, v_lds + i0 * kRowBytes);
  };
  const uint32_t pages_lds = wave_uniform(lds_address(&s_pages[wave][0]));
  auto copy_pages = [&](int32_t m) __attribute__((always_inline)) {
    copy_dwords(page_entry(m), pages_lds);
  };
  auto live_in = [&](int32_t j) { return j * kWaves + wave < n_tiles; };

  // Every register load has landed before the first copy: a wait of the
  // compiler's own on one of them would wait for the copies too.
  auto landed = [](uint4 &x) __attribute__((always_inline)) {
    u32x4v_t t = {x.x, x.y, x.z, x.w};
    asm volatile("" : "+v"(t));
    x = make_uint4(t.x, t.y, t.z, t.w);
  };
  asm volatile("" : "+v"(row_word));
  address_rows();
#pragma unroll
  for (int i = 0; i < kWaveHeads; ++i) landed(q_row[i]);
  landed(token_k);
  landed(token_v);
  landed(wq);
  landed(wk);
  wait_vector<0>();
  if (prep_token) {
    copy_dwords(p.cos + (int64_t)token_pos * (kRot / 2) + lane,
                wave_uniform(lds_address(&s_rope[wave][0][0])));
    copy_dwords(p.sin + (int64_t)token_pos * (kRot / 2) + lane,
                wave_uniform(lds_address(&s_rope[wave][1][0])));
  }
  if (owns && wave == 0) copy_dwords(token_entry(), wave_uniform(lds_address(&s_append[0])));
  const bool live0 = live_in(0);
  if (live0) {
#pragma unroll
    for (int i = 0; i < kTileKeys; i += 4) copy_k4(0, i);
  }
  if (prep_token) {  // while the first K rows are in flight
    // cos and sin: everything before the tile's copies, if it has any.
    if (live0) {
      wait_vector<kTileKeys>();
    } else {
      wait_vector<0>();
    }
    PrepInputs pin{};
    const int d0 = lane * kPackElems;
    if (d0 < kRot) {
      const int pair = d0 < kRot / 2 ? d0 : d0 - kRot / 2;
      const float4 *cr = reinterpret_cast<const float4 *>(&s_rope[wave][0][pair]);
      const float4 *sr = reinterpret_cast<const float4 *>(&s_rope[wave][1][pair]);
      pin.c0 = cr[0]; pin.c1 = cr[1]; pin.s0 = sr[0]; pin.s1 = sr[1];
    }
    pin.w = wq;
#pragma unroll
    for (int i = 0; i < kWaveHeads; ++i)
      q_row[i] = prep_math<kWave, kRot>(q_row[i], true, pin, lane);
    if (owns) {
      pin.w = wk;
      token_k = prep_math<kWave, kRot>(token_k, true, pin, lane);
      token_v = prep_math<kWave, kRot>(token_v, false, pin, lane);
    }
  }
#pragma unroll
  for (int i = 0; i < kWaveHeads; ++i) {
    const int head = wave * kWaveHeads + i;
    s_q[head * kRowChunks + (lane ^ head)] = q_row[i];
  }
  if (kOwnQ && live0) {
#pragma unroll
    for (int i = 0; i < kTileKeys; i += 4) copy_v4(0, i);
  }
  lds_barrier();
  uint4 q[kSteps];
#pragma unroll
  for (int s = 0; s < kSteps; ++s) q[s] = s_q[h * kRowChunks + ((4 * s + g) ^ h)];
  if constexpr (!kOwnQ) {
    lds_barrier();  // every wave has its operands: the V tile is free
    if (live0) {
#pragma unroll
      for (int i = 0; i < kTileKeys; i += 4) copy_v4(0, i);
    }
  }
  if (n_steps > kChunkTiles) copy_pages(1);

  // V^T operand: lane group g reads rows 4 g + vj, dims 16 d + 4 vq.
  const int vj = (lane & 15) >> 2, vq = lane & 3;
  const int vrow = 4 * g + vj;
  const int v_off = vrow * kRowBytes + ((vq >> 1) << 4) + ((vq & 1) << 3);

  // An unreadable key's V row is zero (its probability is 0 as well, but the
  // bytes in its place may be anything), and so is a whole idle tile.
  auto zero_v = [&](uint32_t valid) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kTileKeys; ++i)
      if (((valid >> i) & 1u) == 0) v_tile[i * kRowChunks + lane] = make_uint4(0, 0, 0, 0);
  };

#pragma unroll 1
  for (int32_t j = 0; j < n_steps; ++j) {
    const bool live = live_in(j);
    const int at = (j % kChunkTiles) * kTileKeys;
    const uint32_t mine = live ? 0xFFFFu : 0u;
    const uint32_t valid =
        (uint32_t)(__builtin_amdgcn_ballot_w64(row_word != kRowInvalid) >> at) & mine;
    const uint32_t fresh =
        (uint32_t)(__builtin_amdgcn_ballot_w64(row_word == kRowNewToken) >> at) & mine;
    f32x4_t score = {0.0f, 0.0f, 0.0f, 0.0f};
    if (live) {
      wait_vector<kTileKeys>();  // K of this step (its V copies are younger)
      if (fresh != 0) {
        const int i = __builtin_ctz(fresh);
        k_tile[i * kRowChunks + (lane ^ i)] = token_k;
        wave_lds_sync();
      }
      f32x4_t s_acc[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) s_acc[i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int s = 0; s < kSteps; ++s) {
        const uint4 kf = k_tile[h * kRowChunks + ((4 * s + g) ^ h)];
        s_acc[s & 3] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(bf16x8_t, kf), __builtin_bit_cast(bf16x8_t, q[s]), s_acc[s & 3], 0,
            0, 0);
      }
      score = (s_acc[0] + s_acc[1]) + (s_acc[2] + s_acc[3]);
      // The K reads run eight MFMAs ahead (the compiler's own order waits
      // for each read right before its MFMA).
      __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
#pragma unroll
      for (int i = 0; i < kSteps - 8; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
      wait_lds_reads();
    }
    const bool more = j + 1 < n_steps;
    const bool live_next = more && live_in(j + 1);
    if (live_next) {
      if ((j + 1) % kChunkTiles == 0) {
        // Copied during this lookup's first step, long complete.
        row_word = key_row_of((j + 1) / kChunkTiles, s_pages[wave][lane]);
        address_rows();
      }
#pragma unroll
      for (int i = 0; i < kTileKeys; i += 4) copy_k4(j + 1, i);
    }

    float sc[4];
    float tmax = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      sc[i] = ((valid >> (4 * g + i)) & 1u) ? score[i] * p.q_scale : -INFINITY;
      tmax = fmaxf(tmax, sc[i]);
    }
    tmax = xor_max<16>(tmax);
    tmax = xor_max<32>(tmax);
    if (lane < kQueryHeads) s_max[wave][lane] = tmax;
    if (!live) zero_v(0);  // an idle wave's tile, if the step has one
    lds_barrier();
    float m_new = m_run;
#pragma unroll
    for (int k = 0; k < kWaves; ++k) m_new = fmaxf(m_new, s_max[k][h]);
    if (__builtin_amdgcn_ballot_w64(m_new > m_run) != 0) {
      const float alpha = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_new);
      l_run *= alpha;
#pragma unroll
      for (int d = 0; d < kWaveBlocks; ++d) acc[d] *= alpha;
      m_run = m_new;
    }
    const float m_use = m_run == -INFINITY ? 0.0f : m_run;
    float pr[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      pr[i] = __builtin_amdgcn_exp2f(sc[i] - m_use);
      l_run += pr[i];
    }
    // A probability is the sum of two bf16, 16 bits of it: one bf16 alone left
    // the outputs further from the 64-bit result than shorter splits did
    // (whose largest weights are 1), and the matrix units have the room. Both
    // parts are positive (the first is cut, not rounded, and the rest is
    // 2^-126 at least): with a negative or zero second part an infinite V
    // would turn into NaN.
    auto upper = [](float a, float b) __attribute__((always_inline)) {
      return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
    };
    const uint32_t hi01 = upper(pr[0], pr[1]), hi23 = upper(pr[2], pr[3]);
    const float hi[4] = {bf16_lo(hi01), bf16_hi(hi01), bf16_lo(hi23), bf16_hi(hi23)};
    float lo[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) lo[i] = fmaxf(pr[i] - hi[i], fminf(pr[i], 0x1p-126f));
    s_p[wave][lane] =
        make_uint4(hi01, hi23, cvt_pk_bf16(lo[0], lo[1]), cvt_pk_bf16(lo[2], lo[3]));

    if (live_next) {
      wait_vector<kTileKeys>();  // V of this step (the next K copies are younger)
    } else {
      wait_vector<0>();
    }
    if (live && valid != 0xFFFFu) zero_v(valid);
    if (fresh != 0) {
      const int i = __builtin_ctz(fresh);
      v_tile[i * kRowChunks + (lane ^ ((i & 7) << 1))] = token_v;
    }
    lds_barrier();
    // Two waves' keys per MFMA: contraction index 8 g + e is key 4 g + e of
    // the first for e < 4, key 4 g + e - 4 of the second otherwise.
    const int live_tiles = min(n_tiles - j * kWaves, kWaves);
#pragma unroll
    for (int k = 0; k < kWaves; k += 2) {
      if (k >= live_tiles) break;
      const uint4 p0 = s_p[k][lane], p1 = s_p[k + 1][lane];
      const uint4 p_hi = make_uint4(p0.x, p0.y, p1.x, p1.y);
      const uint4 p_lo = make_uint4(p0.z, p0.w, p1.z, p1.w);
      const char *v_base[2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
        v_base[i] = reinterpret_cast<const char *>(&s_tile[k + i][kTileUint4]) + v_off +
                    wave * kWaveBlocks * 32;
      auto weigh = [&](const uint4 &vt, const uint4 &pb, f32x4_t &a) __attribute__((always_inline)) {
        a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, vt),
                                                    __builtin_bit_cast(bf16x8_t, pb), a, 0, 0, 0);
      };
      uint4 vt[kWaveBlocks];
#pragma unroll
      for (int d = 0; d < kWaveBlocks; ++d) {
        // Block wave * kWaveBlocks + d; kWaveBlocks is a multiple of 8.
        typedef __attribute__((address_space(3))) i16x4_t lds_i16x4;
        const int off = (((d & 7) ^ (vrow & 7)) << 5) + (d >> 3) * 256;
        uint2 half[2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
          half[i] = __builtin_bit_cast(
              uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                         (lds_i16x4 *)(__attribute__((address_space(3))) const char *)(v_base[i] + off)));
        vt[d] = make_uint4(half[0].x, half[0].y, half[1].x, half[1].y);
        weigh(vt[d], p_hi, acc[d]);
        if (d > 0) weigh(vt[d - 1], p_lo, acc[d - 1]);
      }
      weigh(vt[kWaveBlocks - 1], p_lo, acc[kWaveBlocks - 1]);
      // V reads four blocks ahead of their MFMAs.
      __builtin_amdgcn_sched_group_barrier(0x100, 2 + 8, 1);
#pragma unroll
      for (int d = 0; d < kWaveBlocks - 4; ++d) {
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 1);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 8, 1);
    }
    if (more) {
      lds_barrier();  // every wave has read this step's V and probabilities
      if (live_next) {
#pragma unroll
        for (int i = 0; i < kTileKeys; i += 4) copy_v4(j + 1, i);
      }
      if ((j + 1) % kChunkTiles == 0 && j + 1 + kChunkTiles < n_steps)
        copy_pages((j + 1) / kChunkTiles + 1);
    }
  }
  l_run = xor_sum<16>(l_run);
  l_run = xor_sum<32>(l_run);
  if (lane < kQueryHeads) s_l[wave][lane] = l_run;
  __syncthreads();
  l_run = 0.0f;
#pragma unroll
  for (int k = 0; k < kWaves; ++k) l_run += s_l[k][h];

  // ---- emit: lane holds dims 16 (wave * kWaveBlocks + d) + 4 g .. + 3 of head h
  const bool whole_row = direct || (combines && live_splits == 1);
  const int64_t row = (int64_t)b * kQueryHeads + h;
  const int dim0 = wave * kWaveBlocks * 16 + 4 * g;
  if (whole_row) {
    const float inv = l_run > 0.0f ? 1.0f / l_run : 0.0f;
#pragma unroll
    for (int d = 0; d < kWaveBlocks; ++d)
      *reinterpret_cast<uint2 *>(p.out + row * kDim + dim0 + 16 * d) =
          make_uint2(pack_bf16x2(acc[d][0] * inv, acc[d][1] * inv),
                     pack_bf16x2(acc[d][2] * inv, acc[d][3] * inv));
  } else {
    const int64_t pidx = row * p.num_splits + split;
    const float m_nat = m_run == -INFINITY ? -INFINITY : m_run * kLn2;
    if (combines) {
      // Device-coherent (sc1) stores: the combining workgroup may run on
      // another XCD, whose L2 does not see this XCD's write-back lines.
      if (threadIdx.x < kQueryHeads) {
        coherent_store(p.partial_m + pidx, m_nat);
        coherent_store(p.partial_l + pidx, l_run);
      }
      // Rows of head h of this sequence: h * num_splits * 2 KiB past head 0's.
      const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(
          p.partial_acc + ((int64_t)b * kQueryHeads * p.num_splits + split) * kDim, 0, 0x7fffffff,
          0x00020000);
      const int32_t off = (h * p.num_splits * kDim + dim0) * 4;
#pragma unroll
      for (int d = 0; d < kWaveBlocks; ++d)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[d]), rsrc,
                                               off + 64 * d, 0, kCoherentAux);
    } else {
      if (threadIdx.x < kQueryHeads) {
        p.partial_m[pidx] = m_nat;
        p.partial_l[pidx] = l_run;
      }
      float *dst = p.partial_acc + pidx * kDim + dim0;
#pragma unroll
      for (int d = 0; d < kWaveBlocks; ++d) *reinterpret_cast<f32x4_t *>(dst + 16 * d) = acc[d];
    }
  }
  if (owns && wave == 0) store_rows(wave_uniform(s_append[0]), token_k, token_v);
  if (whole_row || !combines) return;

  // ---- in-kernel combine by the sequence's last split workgroup, as in
  // decode_split_kernel.
  wait_stores_complete();
  __syncthreads();
  if (threadIdx.x == 0) {
    int32_t *counter = p.counters + b;
    const int32_t arrived =
        __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const bool last = arrived == live_splits - 1;
    if (last) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = last ? 1 : 0;
  }
  __syncthreads();
  if (s_last == 0) return;
#pragma unroll 1
  for (int head = wave; head < kQueryHeads; head += kWaves)
    combine_row_group<1, kDim, kWave, 1>(p, b, head, live_splits, 0, lane);
}

template <int kWaves>
hipError_t launch(const DecodeParams &p, int32_t batch_count, hipStream_t stream) {
  const dim3 grid = p.balanced != 0 ? dim3(p.balanced) : dim3(1, p.num_splits, batch_count);
  hipLaunchKernelGGL(decode_split_d512_kernel<kWaves>, grid, dim3(kWaves * kWave), 0, stream, p);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_split_d512(const DecodeParams &p, int32_t batch_count, hipStream_t stream) {
  const bool four = p.counters != nullptr || (p.balanced == 0 && p.split_size <= kD512OneStep);
  return four ? launch<4>(p, batch_count, stream) : launch<2>(p, batch_count, stream);
}

}  // namespace gemma4
