// Row-level pieces shared by the two split kernels (8 x 256 in
// decode_attention.hip, 1 x 512 in decode_d512.hip): the in-kernel combine of
// a row's split partials and the per-row RMSNorm + RoPE preparation.
#pragma once

#include "decode_common.hpp"
#include "prep_common.hpp"

namespace gemma4 {

// Log-sum-exp combine of `splits` partials for GW consecutive query heads
// starting at q_head0 of batch b, by one wave of the last-arriving split
// workgroup, reading the other workgroups' partials with coherent loads that
// are issued in independent batches (one memory round trip per batch).
// Lane (r, cpack) owns dims [8*cpack, 8*cpack+8) and takes the splits
// s == r (mod RPL); the RPL row groups are summed at the end. Same
// arithmetic as decode_combine_kernel.
template <int GW, int D, int LPR, int RPL>
__device__ __forceinline__ void combine_row_group(const DecodeParams &p, int32_t b,
                                                  int32_t q_head0, int32_t splits,
                                                  int r, int cpack) {
  constexpr int kBatch = 8;
  const int lane = __lane_id();
#pragma unroll 1
  for (int g = 0; g < GW; ++g) {
    const int64_t row = (int64_t)b * kQueryHeads + q_head0 + g;
    const auto pm = coherent_view(p.partial_m + row * p.num_splits, splits);
    const auto pl = coherent_view(p.partial_l + row * p.num_splits, splits);
    const auto pa = coherent_view(p.partial_acc + row * p.num_splits * D, splits * D);
    float big_m = -INFINITY;
    for (int32_t s0 = 0; s0 < splits; s0 += kWave * 4) {
      float mv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int32_t s = s0 + i * kWave + lane;
        mv[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(pm, s * 4, 0, kCoherentAux));
        mv[i] = s < splits ? mv[i] : -INFINITY;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) big_m = fmaxf(big_m, mv[i]);
    }
    big_m = reduce_max_from<1>(big_m);
    float big_l = 0.0f;
    float sum[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int32_t s0 = r; s0 < splits; s0 += kBatch * RPL) {
      float ms[kBatch], ls[kBatch];
      u32x4 lo[kBatch], hi[kBatch];
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        const int32_t s = s0 + i * RPL;  // past `splits`: reads 0, weight 0
        ms[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(pm, s * 4, 0, kCoherentAux));
        ls[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(pl, s * 4, 0, kCoherentAux));
        const int32_t off = (s * D + cpack * 8) * 4;
        lo[i] = __builtin_amdgcn_raw_buffer_load_b128(pa, off, 0, kCoherentAux);
        hi[i] = __builtin_amdgcn_raw_buffer_load_b128(pa, off + 16, 0, kCoherentAux);
      }
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        const float w = ls[i] > 0.0f ? __builtin_amdgcn_exp2f((ms[i] - big_m) * kLog2e) : 0.0f;
        big_l = fmaf(ls[i] > 0.0f ? ls[i] : 0.0f, w, big_l);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          sum[j] = fmaf(__uint_as_float(lo[i][j]), w, sum[j]);
          sum[4 + j] = fmaf(__uint_as_float(hi[i][j]), w, sum[4 + j]);
        }
      }
    }
    big_l = sum_rows<LPR>(big_l);
#pragma unroll
    for (int j = 0; j < 8; ++j) sum[j] = sum_rows<LPR>(sum[j]);
    if (r == 0) {
      const float inv = (splits > 0 && big_l > 0.0f) ? 1.0f / big_l : 0.0f;
      uint4 o;
      o.x = pack_bf16x2(sum[0] * inv, sum[1] * inv);
      o.y = pack_bf16x2(sum[2] * inv, sum[3] * inv);
      o.z = pack_bf16x2(sum[4] * inv, sum[5] * inv);
      o.w = pack_bf16x2(sum[6] * inv, sum[7] * inv);
      store128(p.out + row * D + cpack * kPackElems, o);
    }
  }
}

// RMSNorm (learned weight, or scale-free with weight == null) and split-half
// RoPE over the first kRot dims of one head held in this kernel's layout:
// lane c of a row holds dims [8c, 8c + 8) of the D = 8 * LPR dims, so the sum
// of squares is a reduction over the LPR lanes of the row and the rotary
// partner of dim d (d + kRot/2 or d - kRot/2) sits kRot/16 lanes away.
// Follows src/gemma4_flash_attention_decode.cu:233-283 and
// src/gemma4_rope.cu:8-20; the result is rounded to bf16 as the reference
// stores prepared rows.
template <int LPR, int kRot>
__device__ __forceinline__ uint4 prep_pack(uint4 raw, const uint16_t *weight,
                                           const float *cos_row, const float *sin_row,
                                           int cpack) {
  float x[8];
  unpack8(raw, x);
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) ss = fmaf(x[i], x[i], ss);
  ss += lane_xor<1>(ss);
  ss += lane_xor<2>(ss);
  ss += lane_xor<4>(ss);
  ss += lane_xor<8>(ss);
  ss = xor_sum<16>(ss);
  if constexpr (LPR == 64) ss = xor_sum<32>(ss);
  const float scale = 1.0f / sqrtf(ss / (float)(LPR * kPackElems) + kRmsEps);
  float y[8];
  if (weight == nullptr) {
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = x[i] * scale;
  } else {
    float w[8];
    unpack8(load128(weight + cpack * kPackElems), w);
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = x[i] * scale * w[i];
    constexpr int kHalf = kRot / 2;
    float partner[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) partner[i] = lane_xor<kHalf / kPackElems>(y[i]);
    const int d0 = cpack * kPackElems;
    if (d0 < kRot) {
      const int pair = d0 < kHalf ? d0 : d0 - kHalf;
      const float sign = d0 < kHalf ? -1.0f : 1.0f;
#pragma unroll
      for (int i = 0; i < 8; ++i) y[i] = fmaf(sign * partner[i], sin_row[pair + i], y[i] * cos_row[pair + i]);
    }
  }
  return make_uint4(pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3]), pack_bf16x2(y[4], y[5]),
                    pack_bf16x2(y[6], y[7]));
}

// The inputs prep_pack reads besides the row, loaded ahead of the math: the
// lane's 8 weights (packed bf16) and cos / sin of its rotary pair.
struct PrepInputs {
  uint4 w;
  float4 c0, c1, s0, s1;
};
template <int LPR, int kRot>
__device__ __forceinline__ PrepInputs prep_inputs(const uint16_t *weight, const float *cos_row,
                                                  const float *sin_row, int cpack) {
  PrepInputs in;
  in.w = weight != nullptr ? load128(weight + cpack * kPackElems) : make_uint4(0, 0, 0, 0);
  const int d0 = cpack * kPackElems;
  const int pair = d0 < kRot / 2 ? d0 : d0 - kRot / 2;
  const bool rot = weight != nullptr && d0 < kRot;
  // Scalar loads: the tables come through the C-ABI with no alignment promise.
  const float *cr = rot ? cos_row + pair : nullptr;
  const float *sr = rot ? sin_row + pair : nullptr;
  in.c0 = rot ? make_float4(cr[0], cr[1], cr[2], cr[3]) : make_float4(0.f, 0.f, 0.f, 0.f);
  in.c1 = rot ? make_float4(cr[4], cr[5], cr[6], cr[7]) : make_float4(0.f, 0.f, 0.f, 0.f);
  in.s0 = rot ? make_float4(sr[0], sr[1], sr[2], sr[3]) : make_float4(0.f, 0.f, 0.f, 0.f);
  in.s1 = rot ? make_float4(sr[4], sr[5], sr[6], sr[7]) : make_float4(0.f, 0.f, 0.f, 0.f);
  return in;
}
// prep_pack's arithmetic on preloaded inputs (weighted: learned RMSNorm +
// RoPE; otherwise the scale-free RMSNorm), the same operations in the same
// order.
template <int LPR, int kRot>
__device__ __forceinline__ uint4 prep_math(uint4 raw, bool weighted, const PrepInputs &in,
                                           int cpack) {
  float x[8];
  unpack8(raw, x);
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) ss = fmaf(x[i], x[i], ss);
  ss += lane_xor<1>(ss);
  ss += lane_xor<2>(ss);
  ss += lane_xor<4>(ss);
  ss += lane_xor<8>(ss);
  ss = xor_sum<16>(ss);
  if constexpr (LPR == 64) ss = xor_sum<32>(ss);
  const float scale = 1.0f / sqrtf(ss / (float)(LPR * kPackElems) + kRmsEps);
  float y[8];
  if (!weighted) {
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = x[i] * scale;
  } else {
    float w[8];
    unpack8(in.w, w);
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = x[i] * scale * w[i];
    constexpr int kHalf = kRot / 2;
    float partner[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) partner[i] = lane_xor<kHalf / kPackElems>(y[i]);
    const int d0 = cpack * kPackElems;
    if (d0 < kRot) {
      const float sign = d0 < kHalf ? -1.0f : 1.0f;
      const float c[8] = {in.c0.x, in.c0.y, in.c0.z, in.c0.w, in.c1.x, in.c1.y, in.c1.z, in.c1.w};
      const float sn[8] = {in.s0.x, in.s0.y, in.s0.z, in.s0.w, in.s1.x, in.s1.y, in.s1.z, in.s1.w};
#pragma unroll
      for (int i = 0; i < 8; ++i) y[i] = fmaf(sign * partner[i], sn[i], y[i] * c[i]);
    }
  }
  return make_uint4(cvt_pk_bf16(y[0], y[1]), cvt_pk_bf16(y[2], y[3]), cvt_pk_bf16(y[4], y[5]),
                    cvt_pk_bf16(y[6], y[7]));
}

}  // namespace gemma4
