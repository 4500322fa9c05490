// Quantise-and-store of new keys / values into the paged int4 or k8v4 cache, and the randomized Hadamard
// rotation of rows.
//
// Store semantics follow `_store_k8v4` (k8v4_ops.py:11-63), whose value half states it matches vLLM's int4 store:
//   int8 key:  scale = max(absmax / 127, 1e-6); code = clamp(round(k / scale), -127, 127); word = fp32 scale
//   int4 half: scale = max((max - min) / 15, 1e-6); zp = clamp(round(-min / scale), 0, 15);
//              code = clamp(round(fma(x, 1 / scale, zp)), 0, 15); word = (bits(scale) & ~0xF) | zp
// with round = half away from zero through an fp32 `x +/- 0.5` and truncation (k8v4_ops.py:5-8). Token i goes to
// slot slot_mapping[i]; negative slots are skipped (k8v4_ops.py:25-27). With signs, key and value are first rotated
// (x -> x D H, Sylvester H, +/-1 diagonal D) in fp32 and rounded to bf16, as `single_rht(x.float()).to(x.dtype)`
// (k8v4_kv.py:71-72).
//
// A lane owns 8 consecutive channels, so a row is held by 8 to 64 lanes and a workgroup stores 4 to 32 consecutive tokens
// of one KV head (adjacent cells where slots are). Three stages of the Walsh-Hadamard transform are then local to a
// lane and the others, like the reductions, are DPP moves and row swaps on the VALU; a lane loads its 16 bytes of a row
// at once and stores its int4 codes as one dword. With one wave per (token, head), 2 channels per lane, LDS permutes for
// every exchange and 64-bit divisions for the slot, 4096 tokens of 8 heads of 128 (21 MB) took 22 us;
// this takes 11.2-11.6, set by the VALU work of the rotation and the quantiser's divisions as much as by memory.
#include "qp_common.h"

namespace qp {

struct StoreParams {
  const uint16_t *key;
  int64_t kst0, kst1;
  const uint16_t *value;
  int64_t vst0, vst1;
  const int64_t *slots;
  uint8_t *kcodes;
  int64_t ks0, ks1, ks2;
  uint32_t *kwords;
  int64_t kws0, kws1, kws2;
  uint8_t *vcodes;
  int64_t vs0, vs1, vs2;
  uint32_t *vwords;
  int64_t vws0, vws1, vws2;
  int32_t num_tokens, block_size;
  uint32_t bs_magic, bs_shift;  // slot / block_size == fast_div(slot, ...) for slots below 2^31 and block_size > 1
  const float *signs;
};

__device__ __forceinline__ float round_half_away(float x) { return x >= 0.f ? truncf(x + 0.5f) : truncf(x - 0.5f); }

constexpr int kStoreThreads = 256;

// Maximum over the LANES lanes of a row, every lane receiving it (a group's lanes agree after each step, so mirrors serve
// as exchanges).
template <int LANES>
__device__ __forceinline__ float row_max(float v) {
  v = fmaxf(v, dpp<0xB1>(v));
  v = fmaxf(v, dpp<0x4E>(v));
  v = fmaxf(v, dpp<0x141>(v));
  if constexpr (LANES >= 16) v = fmaxf(v, dpp<0x140>(v));  // row_mirror
  if constexpr (LANES >= 32) {
    const uint32_t b = __float_as_uint(v);
    const auto r = __builtin_amdgcn_permlane16_swap(b, b, false, false);
    v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  }
  if constexpr (LANES >= 64) {
    const uint32_t b = __float_as_uint(v);
    const auto r = __builtin_amdgcn_permlane32_swap(b, b, false, false);
    v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  }
  return v;
}

// The lane's 8 channels of a row as bf16 pairs.
template <bool VEC>
__device__ __forceinline__ u32x4_t load_bf16x8(const uint16_t *row) {
  if constexpr (VEC) {
    return *reinterpret_cast<const u32x4_t *>(row);
  } else {
    u32x4_t v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = (uint32_t)row[2 * i] | ((uint32_t)row[2 * i + 1] << 16);
    return v;
  }
}

// fp32 channels of the row, rotated and rounded to bf16 when ROT: (x D) H, butterflies over channel bits in ascending
// order as rht_kernel runs them.
template <int LANES, bool ROT>
__device__ __forceinline__ void store_row(float (&x)[8], u32x4_t v, const float (&signs)[8], int lane) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    x[2 * i] = bf16_lo(v[i]);
    x[2 * i + 1] = bf16_hi(v[i]);
  }
  if constexpr (ROT) {
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] *= signs[i];
    fwht_groups<8, LANES>(x, lane);
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = __uint_as_float((uint32_t)f32_to_bf16_bits(x[i]) << 16);
  }
}

// N code dwords of the lane to its place in the row.
template <bool VEC, int N>
__device__ __forceinline__ void put_codes(uint8_t *dst, const uint32_t (&w)[N]) {
  if constexpr (VEC) {
#pragma unroll
    for (int i = 0; i < N; ++i) reinterpret_cast<uint32_t *>(dst)[i] = w[i];
  } else {
#pragma unroll
    for (int i = 0; i < 4 * N; ++i) dst[i] = (uint8_t)(w[i / 4] >> (8 * (i % 4)));
  }
}

// Asymmetric int4 of a row: stores the lane's 8 codes as 4 bytes, returns the word.
template <int LANES, bool VEC>
__device__ __forceinline__ uint32_t quant_int4(const float (&x)[8], uint8_t *codes_row, int lane) {
  float lo = x[0], hi = x[0];
#pragma unroll
  for (int i = 1; i < 8; ++i) {
    lo = fminf(lo, x[i]);
    hi = fmaxf(hi, x[i]);
  }
  lo = -row_max<LANES>(-lo);
  hi = row_max<LANES>(hi);
  const float scale = fmaxf((hi - lo) / 15.0f, 1e-6f);
  const float zp = fminf(fmaxf(round_half_away(-lo / scale), 0.f), 15.f);
  const float inv = 1.0f / scale;
  uint32_t w[1] = {0};
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    // clamp(round_half_away(y), 0, 15): a negative y rounds to 0 at most, so only y + 0.5 of the others is truncated
    const float y = fmaf(x[i], inv, zp);
    w[0] |= (uint32_t)fminf(fmaxf(y, 0.f) + 0.5f, 15.f) << (4 * i);
  }
  put_codes<VEC>(codes_row + 4 * lane, w);
  return (__float_as_uint(scale) & 0xFFFFFFF0u) | (uint32_t)zp;
}

template <int LANES, bool VEC>
__device__ __forceinline__ uint32_t quant_int8(const float (&x)[8], uint8_t *codes_row, int lane) {
  float a = fabsf(x[0]);
#pragma unroll
  for (int i = 1; i < 8; ++i) a = fmaxf(a, fabsf(x[i]));
  a = row_max<LANES>(a);
  const float scale = fmaxf(a / 127.0f, 1e-6f);
  uint32_t w[2] = {0, 0};
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float q = fminf(fmaxf(round_half_away(x[i] / scale), -127.f), 127.f);
    w[i / 4] |= (uint32_t)(uint8_t)(int8_t)q << (8 * (i % 4));
  }
  put_codes<VEC>(codes_row + 8 * lane, w);
  return __float_as_uint(scale);
}

// VEC: rows of 16-byte aligned bf16 and 4-byte aligned codes (the host checks); else element by element.
template <int HS, int KFMT, bool VEC, bool ROT>
__global__ __launch_bounds__(kStoreThreads) void store_kernel(const StoreParams p) {
  constexpr int LANES = HS / 8;
  const int lane = threadIdx.x % LANES, h = blockIdx.y;
  const int64_t tok = (int64_t)blockIdx.x * (kStoreThreads / LANES) + threadIdx.x / LANES;
  if (tok >= p.num_tokens) return;
  const u32x4_t kv = load_bf16x8<VEC>(p.key + tok * p.kst0 + h * p.kst1 + 8 * lane);
  const u32x4_t vv = load_bf16x8<VEC>(p.value + tok * p.vst0 + h * p.vst1 + 8 * lane);
  const int64_t slot = p.slots[tok];
  float signs[8];
  if constexpr (ROT) {
#pragma unroll
    for (int i = 0; i < 8; ++i) signs[i] = p.signs[8 * lane + i];
  }
  if (slot < 0) return;
  int64_t blk, off;
  if ((slot >> 31) == 0 && p.block_size > 1) {
    blk = fast_div((int)slot, p.bs_magic, p.bs_shift);
    off = slot - blk * p.block_size;
  } else {
    blk = slot / p.block_size;
    off = slot % p.block_size;
  }
  float x[8];
  store_row<LANES, ROT>(x, kv, signs, lane);
  uint8_t *krow = p.kcodes + blk * p.ks0 + off * p.ks1 + h * p.ks2;
  const uint32_t kw =
      KFMT == QP_CODES_INT4 ? quant_int4<LANES, VEC>(x, krow, lane) : quant_int8<LANES, VEC>(x, krow, lane);
  store_row<LANES, ROT>(x, vv, signs, lane);
  uint8_t *vrow = p.vcodes + blk * p.vs0 + off * p.vs1 + h * p.vs2;
  const uint32_t vw = quant_int4<LANES, VEC>(x, vrow, lane);
  if (lane == 0) {
    p.kwords[blk * p.kws0 + off * p.kws1 + h * p.kws2] = kw;
    p.vwords[blk * p.vws0 + off * p.vws1 + h * p.vws2] = vw;
  }
}

// ------------------------------------------------------------------------------------------------ rotation

struct RhtParams {
  const void *in;
  int64_t in_stride;
  void *out;
  int64_t out_stride;
  int64_t rows;
  const float *signs;
  float out_scale;
  int32_t in_bf16, out_bf16, inverse;
};

// One wave per row: forward x -> (x D) H, inverse x -> (x H) D, times out_scale.
template <int E>
__global__ __launch_bounds__(256) void rht_kernel(const RhtParams p) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= p.rows) return;
  float x[E];
#pragma unroll
  for (int i = 0; i < E; ++i) {
    const int64_t at = row * p.in_stride + lane * E + i;
    x[i] = p.in_bf16 ? __uint_as_float((uint32_t) static_cast<const uint16_t *>(p.in)[at] << 16)
                     : static_cast<const float *>(p.in)[at];
  }
  if (!p.inverse) {
#pragma unroll
    for (int i = 0; i < E; ++i) x[i] *= p.signs[lane * E + i];
  }
  fwht_wave<E>(x, lane);
#pragma unroll
  for (int i = 0; i < E; ++i) {
    float y = p.inverse ? x[i] * p.signs[lane * E + i] : x[i];
    y *= p.out_scale;
    const int64_t at = row * p.out_stride + lane * E + i;
    if (p.out_bf16) static_cast<uint16_t *>(p.out)[at] = f32_to_bf16_bits(y);
    else static_cast<float *>(p.out)[at] = y;
  }
}

}  // namespace qp

using namespace qp;

namespace {

template <int HS, int KFMT>
void launch_store_format(const StoreParams &p, dim3 grid, bool vec, hipStream_t s) {
  if (p.signs) {
    if (vec) store_kernel<HS, KFMT, true, true><<<grid, kStoreThreads, 0, s>>>(p);
    else store_kernel<HS, KFMT, false, true><<<grid, kStoreThreads, 0, s>>>(p);
  } else {
    if (vec) store_kernel<HS, KFMT, true, false><<<grid, kStoreThreads, 0, s>>>(p);
    else store_kernel<HS, KFMT, false, false><<<grid, kStoreThreads, 0, s>>>(p);
  }
}

template <int HS>
void launch_store(const StoreParams &p, int kfmt, int num_kv_heads, bool vec, hipStream_t s) {
  constexpr int kTokens = kStoreThreads / (HS / 8);  // per workgroup
  const dim3 grid((p.num_tokens + (int64_t)kTokens - 1) / kTokens, num_kv_heads);
  if (kfmt == QP_CODES_INT4) launch_store_format<HS, QP_CODES_INT4>(p, grid, vec, s);
  else launch_store_format<HS, QP_CODES_INT8>(p, grid, vec, s);
}

template <int E>
void launch_rht(const RhtParams &p, hipStream_t s) {
  const unsigned blocks = (unsigned)((p.rows + 3) / 4);
  rht_kernel<E><<<blocks, 256, 0, s>>>(p);
}

}  // namespace

extern "C" int qp_store(const qp_paged_cache *cache, const qp_store_args *a, qp_stream_t stream) {
  QP_REQUIRE(cache && a && a->key && a->value && a->slot_mapping, "qp_store: null argument");
  QP_REQUIRE(cache->key.codes && cache->key.words && cache->value.codes && cache->value.words,
             "qp_store: null cache view");
  const int hs = cache->head_size;
  QP_SUPPORTED(hs == 64 || hs == 128 || hs == 256 || hs == 512, "qp_store: head size must be 64, 128, 256 or 512");
  QP_REQUIRE(cache->key.format == QP_CODES_INT4 || cache->key.format == QP_CODES_INT8, "qp_store: bad key format");
  QP_REQUIRE(cache->value.format == QP_CODES_INT4, "qp_store: values must be int4");
  QP_REQUIRE(cache->block_size > 0 && cache->num_kv_heads > 0 && a->num_tokens >= 0, "qp_store: bad sizes");
  if (a->num_tokens == 0) return QP_OK;
  StoreParams p;
  p.key = static_cast<const uint16_t *>(a->key);
  p.kst0 = a->key_stride[0];
  p.kst1 = a->key_stride[1];
  p.value = static_cast<const uint16_t *>(a->value);
  p.vst0 = a->value_stride[0];
  p.vst1 = a->value_stride[1];
  p.slots = a->slot_mapping;
  p.kcodes = static_cast<uint8_t *>(const_cast<void *>(cache->key.codes));
  p.ks0 = cache->key.code_stride[0];
  p.ks1 = cache->key.code_stride[1];
  p.ks2 = cache->key.code_stride[2];
  p.kwords = static_cast<uint32_t *>(const_cast<void *>(cache->key.words));
  p.kws0 = cache->key.word_stride[0];
  p.kws1 = cache->key.word_stride[1];
  p.kws2 = cache->key.word_stride[2];
  p.vcodes = static_cast<uint8_t *>(const_cast<void *>(cache->value.codes));
  p.vs0 = cache->value.code_stride[0];
  p.vs1 = cache->value.code_stride[1];
  p.vs2 = cache->value.code_stride[2];
  p.vwords = static_cast<uint32_t *>(const_cast<void *>(cache->value.words));
  p.vws0 = cache->value.word_stride[0];
  p.vws1 = cache->value.word_stride[1];
  p.vws2 = cache->value.word_stride[2];
  p.num_tokens = a->num_tokens;
  p.block_size = cache->block_size;
  p.bs_magic = p.bs_shift = 0;
  if (p.block_size > 1) div_magic((uint32_t)p.block_size, &p.bs_magic, &p.bs_shift);
  p.signs = a->rht_signs;
  // vector accesses where every row allows them; views of any alignment go element by element
  bool vec = aligned(p.key, 16) && aligned(p.value, 16) && aligned(p.kcodes, 4) && aligned(p.vcodes, 4);
  for (int i = 0; i < 2; ++i) vec = vec && a->key_stride[i] % 8 == 0 && a->value_stride[i] % 8 == 0;
  for (int i = 0; i < 3; ++i) vec = vec && cache->key.code_stride[i] % 4 == 0 && cache->value.code_stride[i] % 4 == 0;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int nkv = cache->num_kv_heads;
  switch (hs) {
    case 64: launch_store<64>(p, cache->key.format, nkv, vec, s); break;
    case 128: launch_store<128>(p, cache->key.format, nkv, vec, s); break;
    case 256: launch_store<256>(p, cache->key.format, nkv, vec, s); break;
    default: launch_store<512>(p, cache->key.format, nkv, vec, s); break;
  }
  return launch_status();
}

extern "C" int qp_rht(const void *in, int32_t in_dtype, int64_t in_row_stride, void *out, int32_t out_dtype,
                      int64_t out_row_stride, int64_t rows, int32_t head_size, const float *signs, int32_t inverse,
                      float out_scale, qp_stream_t stream) {
  QP_REQUIRE(in && out && signs, "qp_rht: null argument");
  QP_REQUIRE((in_dtype == QP_DTYPE_BF16 || in_dtype == QP_DTYPE_F32) &&
                 (out_dtype == QP_DTYPE_BF16 || out_dtype == QP_DTYPE_F32),
             "qp_rht: dtype must be bf16 or fp32");
  QP_SUPPORTED(head_size == 64 || head_size == 128 || head_size == 256 || head_size == 512 || head_size == 1024,
               "qp_rht: head size must be a power of two in 64..1024");
  QP_REQUIRE(rows >= 0, "qp_rht: bad row count");
  if (rows == 0) return QP_OK;
  RhtParams p;
  p.in = in;
  p.in_stride = in_row_stride;
  p.out = out;
  p.out_stride = out_row_stride;
  p.rows = rows;
  p.signs = signs;
  p.out_scale = out_scale;
  p.in_bf16 = in_dtype == QP_DTYPE_BF16;
  p.out_bf16 = out_dtype == QP_DTYPE_BF16;
  p.inverse = inverse;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  switch (head_size) {
    case 64: launch_rht<1>(p, s); break;
    case 128: launch_rht<2>(p, s); break;
    case 256: launch_rht<4>(p, s); break;
    case 512: launch_rht<8>(p, s); break;
    default: launch_rht<16>(p, s); break;
  }
  return launch_status();
}
