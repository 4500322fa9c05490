// Paged gather + unpack of a cache segment to bf16, bit-exact with the reference's _unpack_segment /
// _unpack_segment_i8 (int4_prefill.py:25-68): out = bf16(fp32(code - zp) * scale) or bf16(fp32(int8) * scale),
// one fp32 rounding and one bf16 rounding, both to nearest even.
//
// Memory-bound: each thread turns kUnits dwords of codes (8 nibbles or 4 int8 each) into 16 or 8 output bytes each. Threads
// of a wave cover consecutive dwords of a row, so both the code reads and the bf16 writes are coalesced, and a thread's
// loads are all issued before any is used: with one dword per thread and its block id, code and store in series, the
// launch was four rounds of that latency (and its index arithmetic 64-bit divisions). 16384 tokens of 4 heads of 256 (42
// MB): 9.9-10.9 us = 3.9-4.2 TB/s against 12.1-13.6.
#include "qp_common.h"

namespace qp {

struct UnpackParams {
  const uint8_t *codes;
  int64_t cs0, cs1, cs2;  // bytes
  const uint32_t *words;
  int64_t ws0, ws1, ws2;  // words
  const int32_t *block_row;
  uint16_t *out;
  int64_t os0, os1;       // elements
  int32_t start, block_size, num_kv_heads;
  uint32_t total;  // dwords of codes, below 2^31
  // divisions by the dwords of a row, the KV heads and the block size (magic and shift; unused for a divisor of 1)
  uint32_t dw, dw_magic, dw_shift, nkv_magic, nkv_shift, bs_magic, bs_shift;
};

constexpr int kUnits = 4;  // dwords of codes per thread

__device__ __forceinline__ uint32_t div_by(uint32_t x, uint32_t d, uint32_t magic, uint32_t shift) {
  return d == 1 ? x : (uint32_t)fast_div((int)x, magic, shift);
}

template <int FMT, bool VEC>
__global__ __launch_bounds__(256) void unpack_kernel(const UnpackParams p) {
  uint32_t code[kUnits], word[kUnits];
  uint16_t *o[kUnits];
  const uint32_t first = blockIdx.x * (kUnits * 256) + threadIdx.x;
#pragma unroll
  for (int k = 0; k < kUnits; ++k) {
    const uint32_t idx = first + 256 * k;
    if (idx >= p.total) break;
    const uint32_t row = div_by(idx, p.dw, p.dw_magic, p.dw_shift), d = idx - row * p.dw;
    const uint32_t t = div_by(row, p.num_kv_heads, p.nkv_magic, p.nkv_shift), h = row - t * p.num_kv_heads;
    const uint32_t pos = p.start + t;
    const uint32_t bidx = div_by(pos, p.block_size, p.bs_magic, p.bs_shift), slot = pos - bidx * p.block_size;
    const int64_t blk = p.block_row[bidx];
    code[k] = *reinterpret_cast<const uint32_t *>(p.codes + blk * p.cs0 + slot * p.cs1 + h * p.cs2 + 4 * d);
    word[k] = p.words[blk * p.ws0 + slot * p.ws1 + h * p.ws2];
    o[k] = p.out + t * p.os0 + h * p.os1 + (FMT == QP_CODES_INT4 ? 8 : 4) * d;
  }
#pragma unroll
  for (int k = 0; k < kUnits; ++k) {
    if (first + 256 * k >= p.total) break;
    if constexpr (FMT == QP_CODES_INT4) {
      const float zp = (float)(word[k] & 0xFu);
      const float scale = __uint_as_float(word[k] & 0xFFFFFFF0u);
      uint32_t w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float a = ((float)((code[k] >> (8 * i)) & 0xFu) - zp) * scale;      // channel 8d + 2i
        const float b = ((float)((code[k] >> (8 * i + 4)) & 0xFu) - zp) * scale;  // channel 8d + 2i + 1
        w[i] = pack_bf16x2(a, b);
      }
      if constexpr (VEC) {
        *reinterpret_cast<u32x4_t *>(o[k]) = u32x4_t{w[0], w[1], w[2], w[3]};
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) reinterpret_cast<uint32_t *>(o[k])[i] = w[i];
      }
    } else {
      const float scale = __uint_as_float(word[k]);
      uint32_t w[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const float a = (float)(int8_t)(code[k] >> (16 * i)) * scale;
        const float b = (float)(int8_t)(code[k] >> (16 * i + 8)) * scale;
        w[i] = pack_bf16x2(a, b);
      }
      if constexpr (VEC) {
        *reinterpret_cast<u32x2_t *>(o[k]) = u32x2_t{w[0], w[1]};
      } else {
        reinterpret_cast<uint32_t *>(o[k])[0] = w[0];
        reinterpret_cast<uint32_t *>(o[k])[1] = w[1];
      }
    }
  }
}

}  // namespace qp

using namespace qp;

extern "C" int qp_unpack_segment(const qp_cache_half *half, int32_t block_size, int32_t num_kv_heads,
                                 int32_t head_size, const int32_t *block_row, int32_t start, int32_t length,
                                 void *out, const int64_t out_stride[2], qp_stream_t stream) {
  QP_REQUIRE(half && block_row && out && out_stride, "qp_unpack_segment: null argument");
  QP_REQUIRE(half->codes && half->words, "qp_unpack_segment: null cache pointer");
  QP_REQUIRE(half->format == QP_CODES_INT4 || half->format == QP_CODES_INT8, "qp_unpack_segment: unknown code format");
  QP_REQUIRE(block_size > 0 && num_kv_heads > 0 && start >= 0 && length >= 0, "qp_unpack_segment: bad sizes");
  QP_REQUIRE(head_size > 0 && head_size % 8 == 0, "qp_unpack_segment: head size must be a multiple of 8");
  for (int i = 0; i < 3; ++i)
    QP_REQUIRE(half->code_stride[i] % 4 == 0, "qp_unpack_segment: code strides must be multiples of 4 bytes");
  QP_REQUIRE(((uintptr_t)half->codes & 3) == 0 && ((uintptr_t)half->words & 3) == 0,
             "qp_unpack_segment: cache views must be 4-byte aligned");
  QP_REQUIRE(out_stride[0] % 2 == 0 && out_stride[1] % 2 == 0 && ((uintptr_t)out & 3) == 0,
             "qp_unpack_segment: output rows must be 4-byte aligned");
  if (length == 0) return QP_OK;
  UnpackParams p;
  p.codes = static_cast<const uint8_t *>(half->codes);
  p.cs0 = half->code_stride[0];
  p.cs1 = half->code_stride[1];
  p.cs2 = half->code_stride[2];
  p.words = static_cast<const uint32_t *>(half->words);
  p.ws0 = half->word_stride[0];
  p.ws1 = half->word_stride[1];
  p.ws2 = half->word_stride[2];
  p.block_row = block_row;
  p.os0 = out_stride[0];
  p.os1 = out_stride[1];
  p.block_size = block_size;
  p.num_kv_heads = num_kv_heads;
  p.dw = half->format == QP_CODES_INT4 ? head_size / 8 : head_size / 4;
  p.dw_magic = p.dw_shift = p.nkv_magic = p.nkv_shift = p.bs_magic = p.bs_shift = 0;
  if (p.dw > 1) div_magic(p.dw, &p.dw_magic, &p.dw_shift);
  if (num_kv_heads > 1) div_magic((uint32_t)num_kv_heads, &p.nkv_magic, &p.nkv_shift);
  if (block_size > 1) div_magic((uint32_t)block_size, &p.bs_magic, &p.bs_shift);
  const bool vec = half->format == QP_CODES_INT4
                       ? (out_stride[0] % 8 == 0 && out_stride[1] % 8 == 0 && ((uintptr_t)out & 15) == 0)
                       : (out_stride[0] % 4 == 0 && out_stride[1] % 4 == 0 && ((uintptr_t)out & 7) == 0);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  // launches of at most 2^30 dwords of codes (one, unless the output is past 16 GiB, or 8 GiB of int8 keys)
  const int64_t per_token = (int64_t)num_kv_heads * p.dw;
  QP_SUPPORTED(per_token < (int64_t(1) << 30), "qp_unpack_segment: rows of a token too large");
  const int64_t most = (int64_t(1) << 30) / per_token;
  for (int64_t t0 = 0; t0 < length; t0 += most) {
    p.start = (int32_t)(start + t0);
    p.out = static_cast<uint16_t *>(out) + t0 * out_stride[0];
    p.total = (uint32_t)((length - t0 < most ? length - t0 : most) * per_token);
    const unsigned blocks = (p.total + kUnits * 256 - 1) / (kUnits * 256);
    if (half->format == QP_CODES_INT4) {
      if (vec) unpack_kernel<QP_CODES_INT4, true><<<blocks, 256, 0, s>>>(p);
      else unpack_kernel<QP_CODES_INT4, false><<<blocks, 256, 0, s>>>(p);
    } else {
      if (vec) unpack_kernel<QP_CODES_INT8, true><<<blocks, 256, 0, s>>>(p);
      else unpack_kernel<QP_CODES_INT8, false><<<blocks, 256, 0, s>>>(p);
    }
  }
  return launch_status();
}
