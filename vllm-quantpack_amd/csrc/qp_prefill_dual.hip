// Chunked-prefill attention over the paged int4 / k8v4 KV cache at heads 64 and 128, with two waves per SIMD.
//
// Reference semantics: as prefill_kernel (qp_prefill.hip), whose arithmetic this kernel keeps: bf16 query and
// exact-integer code operands, fp32 accumulation, S = (q . (128 + k) - sum(q) (128 + zp_k)) s_k scale (int8 keys:
// 128 sum(q)), P_v16 = bf16(P s_v) feeding the PV product and the zero-point sum (int4_kv.py:90-94), l in fp32 from the
// unrounded P (at head 128 below 8 query heads per KV head: the sum of P_v16 / s_v, FOLD below), causal within each
// sequence's query chunk (replacing int4_prefill.py:203-232).
//
// MI355X design. At these head sizes 32 rows' O^T accumulators, zero-point tile included, take at most 80 registers, so
// a wave's tile loop fits 256 (at head 128 some instances spill up to 10 around it; the build refuses spill code in it)
// and two waves fit a SIMD: one wave's softmax and unpack run beside the other's MFMAs. A workgroup of
// 8 waves owns 256 consecutive (token, query head) rows of one sequence and KV head (any GQA width fills them) and one
// key split; a tile of 64 keys is unpacked once for all rows, with one barrier per tile.
//   * 32x32x16 MFMAs: with two waves per SIMD (a loop of MFMAs with N independent FMAs after each, both waves running it)
//     the SIMD takes about max(32, 11 + 4 N) cycles per 32x32x16 MFMA and max(16, 9 + 4 N) per 16x16x32 one, and this
//     kernel has 6.2 VALU instructions per 32x32x16 MFMA at head 128 folded and 7.9 otherwise, so the larger shape hides
//     most of them.
//   * The tile's packed pages are copied HBM -> LDS four tiles ahead (global_load_lds_dwordx4, one or two copies per
//     wave). Past the end of the split the last run is copied again, so no iteration has an end case.
//   * A tile is worked through in 32-key sub-tiles u: the MFMAs of S^T = K Q^T of sub-tile u + 1 and of O^T += V^T P^T of
//     u - 1 alternate (each S^T MFMA waits for the one before it, about 64 cycles, so the other's fill the gap), beside
//     the softmax of u, whose S^T registers packed to bf16 are the B operand of the next sub-tile's PV. The K unpack of
//     tile i + 2 and the V unpack of tile i + 1 are spread over them; the per-key scalars of tile i + 2 are made by one
//     wave, another each tile, as every wave would otherwise repeat about 30 VALU.
//   * The running maximum never changes within a pass, so a tile is one basic block without a branch (kDualBias below).
// The K rows in LDS are padded by one 16-byte unit and the V^T rows' units XOR-swizzled, so that the operand reads and
// the unpack's stores hit every bank once. V^T row r < HS / 2 holds channel 2 r and row r + HS / 2 channel 2 r + 1 (the
// two nibbles of a code byte): a thread's stores then go to two runs of whole rows, and a lane's accumulators hold 8
// consecutive output channels.
//
// What bounds it, and what it measured (64 q / 8 KV heads of 128, 2048 tokens over 16384 cached keys, int4): 1.25-1.29 ms
// = 909-935 TFLOP/s (1.46 ms on the slowest box) against 1.96 ms on 32x32x16 MFMAs with one wave per SIMD; MFMAs busy 46 %
// of the cycles at about 2.1 GHz (2.3 GHz under the head-256 kernel: this one draws more power), the LDS active 53 %. The
// following were measured on the folded form (1.21 ms): without the softmax 1.04 ms, without the unpack 1.10 ms, without
// both, the copies and the operand re-reads 0.79 ms. The order of the steps hardly matters: reads two sub-tiles ahead,
// fences between the steps, raised wave priorities and the build's scheduler are all within 2 %. 16x16x32 MFMAs with the
// phases in turn took 1.27 ms, the two halves of the waves half a tile apart behind a barrier per half 1.45 ms. 8 prompts
// of 128..2048 tokens, 32 q / 8 KV heads: 146 against 265 us on four 16-row tiles per wave; head 64 (32 q / 8 KV heads,
// 512 tokens over 4096, int8 keys): 48-49 against 94 us as query slices.
#include "qp_prefill.h"

#include <type_traits>

namespace qp {

constexpr int kDualWaves = 8;
constexpr int kDualThreads = kDualWaves * 64;
constexpr int kDualRows = kDualWaves * 32;  // (token, query head) rows per workgroup
constexpr float kDualBias = 56.f;      // log2 units between a row's maximum m and its first sub-tile's maximum
constexpr float kDualHeadroom = 64.f;  // largest score - m taken without a second pass

template <int HS, int KFMT>
struct DualShape {
  static constexpr int kHS = HS;
  static constexpr int kKeys = 64;                   // keys per tile
  static constexpr int kSubs = kKeys / 32;
  static constexpr int kKeyBytes = KFMT == QP_CODES_INT4 ? HS / 2 : HS;
  static constexpr int kCell = kKeyBytes + 4 + HS / 2 + 4;
  static constexpr int kRuns = kKeys / 16;
  static constexpr int kRunUnits = kCell;            // 16-byte units of one 16-cell page run
  static constexpr int kSlot = kKeys * kCell;
  static constexpr int kKU = HS / 8;                 // 16-byte units of a K row
  static constexpr int kKdRow = 16 * kKU + 16;       // bf16 K row, padded: 16 rows of one unit are in distinct banks
  static constexpr int kKd = kKeys * kKdRow;
  static constexpr int kVs = HS * 64;                // V^T rows of a sub-tile (32 keys, four units)
  static constexpr int kVt = kSubs * kVs;
  // per-key scalars: a, e, s_v (FOLD: b; fp32 [kKeys] each), then per sub-tile four bf16 rows of 32 keys in V^T key order.
  // Row 0, 16 + zp_v, is every row of the zero-point tile's A operand, so that every lane gets its query row's sum. With
  // FOLD rows 0..2 are that tile's first three, rows 1 and 2 the two halves of 1 / s_v; nothing fills row 3, and the
  // results of the tile's other rows are not used.
  static constexpr int kSc = kKeys * 20;
  static constexpr int kSlots = 4, kKbufs = 3, kVbufs = 3, kScs = 4;
  static constexpr int kOffK = kSlots * kSlot;
  static constexpr int kOffV = kOffK + kKbufs * kKd;
  static constexpr int kOffS = kOffV + kVbufs * kVt;
  static constexpr int kLds = kOffS + kScs * kSc;
  static constexpr int kUnits = HS / 64;             // K units and V units of a thread
  static_assert(kKeys * kKU == kUnits * kDualThreads && (HS / 2) * (kKeys / 4) == kUnits * kDualThreads, "units");
  static_assert(kSlot % 16 == 0 && kKd % 16 == 0 && kVt % 16 == 0 && kSc % 16 == 0 && kLds <= 160 * 1024, "LDS");
  // HBM -> LDS copies of a tile: the runs' full 64-unit copies, then their tails; copy q goes to wave q % 8 as its
  // (q / 8)-th (past the last, a wave copies one of the last copies again, the same bytes to the same place, so that
  // every wave waits on kMax copies per tile)
  static constexpr int kFull = kRunUnits / 64, kTail = kRunUnits % 64;
  static constexpr int kFullCopies = kRuns * kFull;
  static constexpr int kCopies = kFullCopies + kRuns;
  static constexpr int kMax = kUnits;
  static_assert(kTail > 0 && kCopies <= kMax * kDualWaves && 2 * kCopies >= kMax * kDualWaves, "copies per wave");
  // position of 16-byte unit c in V^T row r: any 16 rows of one unit are in distinct banks
  static constexpr __host__ __device__ int v_swz(int r, int c) { return c ^ ((r >> 2) & 3); }
  // unit of a K row's chunk of 8 channels: lane half h reads channels HS / 2 h .. in steps of 8
  static constexpr __host__ __device__ int k_unit(int chunk) { return 2 * (chunk % (kKU / 2)) + chunk / (kKU / 2); }
  // unit and byte in it of key kk (0..31) in a V^T row: MFMA step kk / 16, lane half h's 8 slots are keys 4 h .. 4 h + 3
  // and 8 + 4 h .. of the 16
  static constexpr __host__ __device__ int v_unit(int kk) { return 2 * (kk >> 4) + ((kk >> 2) & 1); }
  static constexpr __host__ __device__ int v_byte(int kk) { return 2 * ((kk & 3) + 4 * ((kk >> 3) & 1)); }
};

__device__ __forceinline__ f32x16_t mfma32x32x16(bf16x8_t a, bf16x8_t b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// Maximum over the two lanes l, l ^ 32, both receiving it.
__device__ __forceinline__ float halves_max(float v) {
  const uint32_t b = __float_as_uint(v);
  const auto q = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  return fmaxf(__uint_as_float(q[0]), __uint_as_float(q[1]));
}

// Butterflies of the Walsh-Hadamard transform on local index bits lo .. hi - 1 (powers of two).
template <int E>
__device__ __forceinline__ void dual_butterfly(float (&x)[E], int lo, int hi) {
#pragma unroll
  for (int span = lo; span < hi; span <<= 1)
#pragma unroll
    for (int i = 0; i < E; ++i)
      if (!(i & span)) {
        const float u = x[i], v = x[i + span];
        x[i] = u + v;
        x[i + span] = u - v;
      }
}

// The butterfly between lanes l and l ^ 32 (the channel bit that the lane half stands for).
template <int E>
__device__ __forceinline__ void dual_butterfly_halves(float (&x)[E], int h) {
#pragma unroll
  for (int i = 0; i < E; ++i) {
    const float v = __shfl_xor(x[i], 32, 64);
    x[i] = h ? v - x[i] : x[i] + v;
  }
}

// log2 of the XCDs that share a (KV head, split) pair's row blocks: 8 over the largest power of two in the pairs.
__host__ __device__ __forceinline__ uint32_t dual_share(uint32_t pairs) {
  return (pairs & 7) == 0 ? 0 : (pairs & 3) == 0 ? 1 : (pairs & 1) == 0 ? 2 : 3;
}

// FOLD: the value scales are folded into the scores (the QK accumulators start at b = log2(s_v) / a, so one exp2 gives
// P s_v) and l comes out of the zero-point tile's MFMA, as in the head-256 tile kernel; it normalises by the rounded
// weights, and a key whose value scale is 0 drops out of it. Otherwise l is summed in fp32 from the unrounded P, two VALU
// instructions more per score. A shape has the form of the kernel that served it before this one, so that its sums keep
// their bits (dual_folds: the tile kernel folds, the query slices and 32x32x16 MFMAs with one wave per SIMD did not). Both
// forms, on one box, and how far they are off the 64-bit result: 8 prompts of up to 2048 tokens, 32 q / 8 KV heads of 128: 155 us and 2.7e-3 folded, 160 us and 3.0e-3 otherwise;
// 2048 tokens over 16384 keys, 64 q / 8 KV heads: 1409 us and 3.7e-3, 1463 us and 3.8e-3; 512 tokens over 4096, 32 q / 8
// KV heads of 64: 48.4 us and 3.5e-3, 51.2 us and 3.6e-3.
template <int HS, int KFMT, bool SPAN, bool FOLD>
__global__ __launch_bounds__(kDualThreads) void prefill_dual_kernel(const PrefillParams p) {
  using Sh = DualShape<HS, KFMT>;
  constexpr int KT = Sh::kKeys;
  constexpr int kSubs = Sh::kSubs;
  constexpr int kCs = HS / 16;     // 16-channel QK steps
  constexpr int kCt = HS / 32;     // channel tiles; tile kCt is the zero-point tile
  __shared__ __attribute__((aligned(1024))) uint8_t smem[Sh::kLds];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = uniform(tid >> 6);
  const int col = lane & 31, h = lane >> 5;
  // Workgroups go to the 8 XCDs in turn: 2^share of them (dual_share; gridDim.x is a multiple) take the same (KV head,
  // split) pairs, one after the other, and of a pair's row blocks every 2^share-th, so that the blocks that share keys
  // share as few L2s as balance allows. Later blocks, which see more keys, come first. (With a contiguous eighth of all
  // blocks per XCD, two XCDs that shared a KV head had its longer and its shorter blocks: 12 prompts of up to 2048 tokens,
  // 28 q / 4 KV heads of 128: 177 us against 199; 6 of up to 1200: 52.6 against 55.4.)
  const uint32_t lin = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
  const uint32_t pairs = gridDim.y * gridDim.z;
  const uint32_t share = dual_share(pairs), per = gridDim.x >> share;
  const uint32_t xcd = lin & 7, turn = (lin >> 3) / per;
  const uint32_t pair = (xcd >> share) * ((pairs << share) >> 3) + turn;
  const int rank = (int)((((lin >> 3) - turn * per) << share) + (xcd & ((1u << share) - 1)));
  const int kvh = (int)(pair % gridDim.y);
  const int split = (int)(pair / gridDim.y);
  const int G = p.num_q_heads / p.num_kv_heads;
  const int blk = (int)gridDim.x - 1 - rank;
  // row block -> sequence: sequence s's rows (cu_q[s] G .. cu_q[s + 1] G) own blocks [cu_q[s] G / kRows + s, ...)
  int lo = 0, hi = p.num_seqs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if ((int)(((int64_t)p.cu_q[mid] * G) / kDualRows) + mid <= blk) lo = mid;
    else hi = mid - 1;
  }
  const int seq = lo;
  const int q0 = p.cu_q[seq], qlen = p.cu_q[seq + 1] - q0;
  const int nrows = qlen * G;
  const int r0 = (blk - (int)(((int64_t)q0 * G) / kDualRows) - seq) * kDualRows;  // first local row of the block
  if (r0 < 0 || r0 >= nrows) return;
  if (p.skip_seq && p.skip_seq[seq] >= 0) return;
  const int n = p.used_k[seq];
  const int t_first = r0 / G, t_last = (min(nrows, r0 + kDualRows) - 1) / G;
  const int first_pos = n - qlen + t_first;
  const int kend = max(0, min(n, n - qlen + t_last + 1));  // keys any row of the block can see
  // key split: the split-KV segment rule shared with qp_merge_segments
  const int S = p.num_splits;
  const int seg = segment_keys(n, S, p.min_keys);
  const int kb = split * seg;
  const int ke = uniform(min(kend, kb + seg));
  if (S > 1 && kb >= n) return;  // inactive segment: the merge does not read it

  // ---- the wave's 32 rows: lane row col -> local row rr = (token rr / G, query head rr % G)
  const bool active = r0 + 32 * w < nrows;
  const int rr = r0 + 32 * w + col;
  const bool valid = rr < nrows;
  const int tok = valid ? rr / G : 0, jh = valid ? rr % G : 0;
  const int row_pos = valid ? n - qlen + tok : kPfNoRow;  // (< 0: a context shorter than the chunk)
  bf16x8_t qop[kCs];
  float qsum, m = -INFINITY, l = 0.f;  // l: of the lane's keys, until the epilogue
  {
    // channels HS / 2 h .. of the row (rotated when asked, then rounded to bf16 once, as a separate rotation pass would)
    const uint16_t *src = p.q + (int64_t)(q0 + tok) * p.qs0 + (int64_t)(kvh * G + jh) * p.qs1 + HS / 2 * h;
    uint32_t qw[HS / 4];
#pragma unroll
    for (int i = 0; i < HS / 16; ++i) {
      const u32x4_t v = valid ? *reinterpret_cast<const u32x4_t *>(src + 8 * i) : u32x4_t{0u, 0u, 0u, 0u};
#pragma unroll
      for (int j = 0; j < 4; ++j) qw[4 * i + j] = v[j];
    }
    if (p.qsigns) {
      float x[HS / 2];
#pragma unroll
      for (int i = 0; i < HS / 4; ++i) {
        x[2 * i] = bf16_lo(qw[i]) * p.qsigns[HS / 2 * h + 2 * i];
        x[2 * i + 1] = bf16_hi(qw[i]) * p.qsigns[HS / 2 * h + 2 * i + 1];
      }
      dual_butterfly(x, 1, HS / 2);
      dual_butterfly_halves(x, h);
#pragma unroll
      for (int i = 0; i < HS / 4; ++i) qw[i] = pack_bf16x2(x[2 * i], x[2 * i + 1]);
    }
    float qs = 0.f;  // the row's query sum: the 128 offset of the key operands (and the int4 zero point) folds into it
#pragma unroll
    for (int cs = 0; cs < kCs; ++cs) {
      const u32x4_t x = u32x4_t{qw[4 * cs], qw[4 * cs + 1], qw[4 * cs + 2], qw[4 * cs + 3]};
      qs += bf16_lo(x[0]) + bf16_hi(x[0]) + bf16_lo(x[1]) + bf16_hi(x[1]) + bf16_lo(x[2]) + bf16_hi(x[2]) +
            bf16_lo(x[3]) + bf16_hi(x[3]);
      if constexpr (KFMT == QP_CODES_INT4) {  // K operand order per 8 channels: (c0, c4, c1, c5, c2, c6, c3, c7)
        u32x4_t y;
        y[0] = (x[0] & 0xFFFFu) | (x[2] << 16);
        y[1] = (x[0] >> 16) | (x[2] & 0xFFFF0000u);
        y[2] = (x[1] & 0xFFFFu) | (x[3] << 16);
        y[3] = (x[1] >> 16) | (x[3] & 0xFFFF0000u);
        qop[cs] = as_bf16x8(y);
      } else {
        qop[cs] = as_bf16x8(x);
      }
    }
    qsum = qs + shfl_xor_f(qs, 32);
    if constexpr (KFMT != QP_CODES_INT4) qsum *= 128.f;
  }
  // O^T tiles: lane l holds row l % 32, V^T rows 32 ct + 8 (i / 4) + 4 h + i % 4
  f32x16_t acc[kCt + 1];
#pragma unroll
  for (int ct = 0; ct <= kCt; ++ct)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[ct][i] = 0.f;  // (a split without keys)

  const int ntiles = ke > kb ? (ke - kb + KT - 1) / KT : 0;
  if (ntiles > 0) {
    const int32_t *trow = p.table + (int64_t)seq * p.table_stride;
    const __attribute__((address_space(4))) int32_t *ctab = (const __attribute__((address_space(4))) int32_t *)trow;
    const int nplain = max(0, min(first_pos + 1, ke) - kb) / KT;  // tiles whose keys are visible to every row
    auto tile_key = [&](int t) { return kb + t * KT; };
    auto pk_of = [&](int t) { return smem + (t & (Sh::kSlots - 1)) * Sh::kSlot; };
    // K and V buffer t % 3, for t = it .. it + 2 of the running tile it (ph = it % 3)
    int ph = 0;
    auto kd_of = [&](int k) { return smem + Sh::kOffK + (ph + k < 3 ? ph + k : ph + k - 3) * Sh::kKd; };
    auto vt_of = [&](int k) { return smem + Sh::kOffV + (ph + k < 3 ? ph + k : ph + k - 3) * Sh::kVt; };
    auto sc_of = [&](int t) { return smem + Sh::kOffS + (t & (Sh::kScs - 1)) * Sh::kSc; };

    // ---- the wave's copies of a tile: copy i covers run c_run[i] from unit c_unit[i] on, c_lanes[i] lanes
    int c_run[Sh::kMax], c_unit[Sh::kMax], c_lanes[Sh::kMax];
#pragma unroll
    for (int i = 0; i < Sh::kMax; ++i) {
      const int at = w + kDualWaves * i;
      const int q = at < Sh::kCopies ? at : 2 * Sh::kCopies - 1 - at;
      c_run[i] = q < Sh::kFullCopies ? q / Sh::kFull : q - Sh::kFullCopies;
      c_unit[i] = q < Sh::kFullCopies ? 64 * (q % Sh::kFull) : 64 * Sh::kFull;
      c_lanes[i] = q < Sh::kFullCopies ? 64 : Sh::kTail;
    }
    const uint32_t lds0 = lds_addr(smem);
    const uint8_t *hbase = p.kcodes + (int64_t)kvh * p.ks2;
    const uint32_t ks0 = (uint32_t)p.ks0;
    const int last_run = (ke - 1) & ~15;  // (the split starts at a multiple of 32 keys)
    int bid[Sh::kMax], soff[Sh::kMax];    // block and byte offset in it of the runs of the next tile to copy
    auto locate = [&](int t) {            // (a run past the last takes the last again)
#pragma unroll
      for (int i = 0; i < Sh::kMax; ++i) {
        const int key = uniform(min(tile_key(t) + 16 * c_run[i], last_run));
        const int b = uniform(fast_div(key, p.bs_magic, p.bs_shift));
        soff[i] = (key - b * p.block_size) * Sh::kCell;
        bid[i] = ctab[b];
      }
    };
    auto copy = [&](int t) {
#pragma unroll
      for (int i = 0; i < Sh::kMax; ++i)
        if (lane < c_lanes[i])
          dma16_saddr<false>(hbase + (uint64_t)(uint32_t)bid[i] * ks0 + (uint32_t)soff[i], 16 * (c_unit[i] + lane),
                             lds0 + (uint32_t)((t & (Sh::kSlots - 1)) * Sh::kSlot +
                                               16 * (c_run[i] * Sh::kRunUnits + c_unit[i])));
    };
    auto fetch = [&](int t) {
      if constexpr (SPAN) {
        locate(t);
        copy(t);
      } else {
        pf_gather<Sh, KT, kDualThreads>(p, trow, tile_key(t), ke, kvh, pk_of(t));
      }
    };

    // ---- the thread's units of the unpack (i = 0, and 1 at head 128): 8 channels of one key's K row; two channels of 4
    // keys of V (keys 4 vq .. of sub-tile vs + i, code byte vc)
    const int ku_key = tid / Sh::kKU, ku_c = tid % Sh::kKU;
    constexpr int kKuStep = kDualThreads / Sh::kKU;  // keys between the two K units
    const int ku_src = ku_key * Sh::kCell + (Sh::kKeyBytes / Sh::kKU) * ku_c;
    const int ku_dst = ku_key * Sh::kKdRow + 16 * Sh::k_unit(ku_c);
    const int vq = tid & 7, vc = (tid >> 3) % (HS / 2), vs = (tid >> 3) / (HS / 2);
    const int vu_src = (32 * vs + 4 * vq) * Sh::kCell + Sh::kKeyBytes + 4 + (vc & ~3);
    const uint32_t vu_sel = 0x0C040C00u + 0x00010001u * (vc & 3);  // code byte vc of two keys' dwords, one per half
    auto v_dst = [&](int r) {
      return vs * Sh::kVs + 64 * r + 16 * Sh::v_swz(r, Sh::v_unit(4 * vq)) + Sh::v_byte(4 * vq);
    };
    const int vu_dst0 = v_dst(vc), vu_dst1 = v_dst(vc + HS / 2);
    u32x2_t kx;
    uint32_t vx[4];
    auto k_load = [&](const uint8_t *pk, int i) {
      const uint8_t *src = pk + ku_src + i * kKuStep * Sh::kCell;
      if constexpr (KFMT == QP_CODES_INT4) kx[0] = *reinterpret_cast<const uint32_t *>(src);
      else kx = *reinterpret_cast<const u32x2_t *>(src);
    };
    auto k_store = [&](uint8_t *kd, int i) {
      u32x4_t y;
      if constexpr (KFMT == QP_CODES_INT4) {
        const uint32_t x4 = kx[0] >> 4;
        y = u32x4_t{nib_pair(kx[0]), nib_pair(x4), nib_pair(kx[0] >> 8), nib_pair(x4 >> 8)};
      } else {
        const u32x2_t a = i8_quad_bf16(kx[0]), b = i8_quad_bf16(kx[1]);
        y = u32x4_t{a[0], a[1], b[0], b[1]};
      }
      *reinterpret_cast<u32x4_t *>(kd + ku_dst + i * kKuStep * Sh::kKdRow) = y;
    };
    auto v_load = [&](const uint8_t *pk, int i) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        vx[k] = *reinterpret_cast<const uint32_t *>(pk + vu_src + (32 * i + k) * Sh::kCell);
    };
    auto v_store = [&](uint8_t *vt, int i) {
      const uint32_t p01 = __builtin_amdgcn_perm(vx[1], vx[0], vu_sel), p23 = __builtin_amdgcn_perm(vx[3], vx[2], vu_sel);
      uint8_t *dst = vt + i * Sh::kVs;
      *reinterpret_cast<u32x2_t *>(dst + vu_dst0) = u32x2_t{nib_pair16(p01, 0), nib_pair16(p23, 0)};
      *reinterpret_cast<u32x2_t *>(dst + vu_dst1) = u32x2_t{nib_pair16(p01, 1), nib_pair16(p23, 1)};
    };
    // the per-key scalars of tile t, by wave w0 (lane kk takes key kk)
    auto scalars = [&](int t, int w0) {
      if (w != w0) return;
      const int kk = lane;
      const uint8_t *pk = pk_of(t);
      uint8_t *sc = sc_of(t);
      const bool ok = tile_key(t) + kk < ke;
      const uint32_t kw = *reinterpret_cast<const uint32_t *>(pk + kk * Sh::kCell + Sh::kKeyBytes);
      const uint32_t vw = *reinterpret_cast<const uint32_t *>(pk + kk * Sh::kCell + Sh::kCell - 4);
      float a, e, x;  // x: b, or s_v
      uint16_t rhi = 0, rlo = 0;
      if constexpr (FOLD) {
        pf_key_scalars<KFMT>(kw, vw, p.scale_log2, ok, a, e, x, rhi, rlo);
      } else {
        a = ok ? __uint_as_float(KFMT == QP_CODES_INT4 ? kw & 0xFFFFFFF0u : kw) * p.scale_log2 : 0.f;
        e = a * (float)(128u + (kw & 0xFu));
        x = ok ? __uint_as_float(vw & 0xFFFFFFF0u) : 0.f;
      }
      float *kf = reinterpret_cast<float *>(sc);
      kf[kk] = a;
      if constexpr (KFMT == QP_CODES_INT4) kf[KT + kk] = e;
      kf[2 * KT + kk] = x;
      uint8_t *z = sc + 12 * KT + 256 * (kk >> 5) + 16 * Sh::v_unit(kk & 31) + Sh::v_byte(kk & 31);
      *reinterpret_cast<uint16_t *>(z) = ok ? (uint16_t)(0x4180u | ((vw & 0xFu) << 3)) : 0;
      if constexpr (FOLD) {
        *reinterpret_cast<uint16_t *>(z + 64) = rhi;
        *reinterpret_cast<uint16_t *>(z + 128) = rlo;
      }
    };

    // ---- operand addresses (a swizzle depends on col alone: 32 rows are a multiple of its period)
    auto k_op = [&](const uint8_t *kd, int u, int cs) {
      return *reinterpret_cast<const bf16x8_t *>(
          kd + (32 * u + col) * Sh::kKdRow + 16 * h + 32 * cs);
    };
    // scalar array k (0 a, 1 e, 2 s_v or b) of the lane's keys 8 q + 4 h .. of sub-tile u
    auto scalar4 = [&](const uint8_t *sc, int k, int u, int q) {
      return *reinterpret_cast<const f32x4_t *>(sc + 4 * (k * KT + 32 * u + 8 * q + 4 * h));
    };
    // what a key's score loses per unit of qsum: e = a (128 + zp) for int4 keys; for int8 keys 128 a, the 128 being in
    // qsum already
    auto offset4 = [&](const f32x4_t &a4, const uint8_t *sc, int u, int q) {
      if constexpr (KFMT == QP_CODES_INT4) return scalar4(sc, 1, u, q);
      else return a4;
    };
    // S^T of a sub-tile starts from the keys' biases b = log2(s_v) / a, or from 0
    auto start = [&](f32x16_t &s, const uint8_t *sc, int u) {
      if constexpr (!FOLD) {
        s = f32x16_t{};
        return;
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4_t b = scalar4(sc, 2, u, q);
#pragma unroll
        for (int j = 0; j < 4; ++j) s[4 * q + j] = b[j];
      }
    };

    f32x16_t s;
    float rmax;  // largest score - m of the lane's keys
    // P of the sub-tile before the running one, and its V^T rows and zero-point rows (at first: zeros on the first ones)
    u32x4_t pop[2];
    const uint8_t *pv, *pz;
    constexpr int kP = 2 * (kCt + 1);  // PV steps of a sub-tile: channel tile c % (kCt + 1), key step c / (kCt + 1)
    auto v_op = [&](int c) {
      const int ct = c % (kCt + 1), ks = c / (kCt + 1);
      return *reinterpret_cast<const bf16x8_t *>(
          ct == kCt ? pz + (FOLD ? 64 * (col & 3) : 0) + 16 * (2 * ks + h)
                    : pv + 64 * (32 * ct + col) + 16 * Sh::v_swz(col, 2 * ks + h));
    };

    // One tile. ROWS: the wave has rows (else it only copies and unpacks); MASK: some key is past some row or the split.
    auto tile = [&](int it, auto rows_tag, auto mask_tag) {
      constexpr bool ROWS = decltype(rows_tag)::value, MASK = decltype(mask_tag)::value;
      if constexpr (SPAN) wait_vmcnt<Sh::kMax>();
      __syncthreads();  // tile it + 2 landed; K(it + 1), V(it) unpacked; K(it - 1)'s, V(it - 2)'s, slot it's readers done
      if constexpr (SPAN) {
        copy(it + Sh::kSlots);
        locate(it + Sh::kSlots + 1);
      } else {
        fetch(it + Sh::kSlots);
      }
      const uint8_t *sc = sc_of(it), *vt = vt_of(0);
#pragma unroll
      for (int u = 0; u < kSubs; ++u) {
        const int k0 = tile_key(it) + 32 * u;
        if (MASK && u > 0 && k0 >= ke) break;  // (the split's last tile: nothing is left to unpack either)
        const bool last = u == kSubs - 1;
        const uint8_t *kd1 = kd_of(last ? 1 : 0), *sc1 = last ? sc_of(it + 1) : sc;
        const int u1 = last ? 0 : u + 1;
        // at head 128 each sub-tile unpacks a K and a V unit, at head 64 the first K and the second V
        const bool unpack_k = Sh::kUnits == kSubs || u == 0, unpack_v = Sh::kUnits == kSubs || u == 1;
        const int ui = Sh::kUnits == kSubs ? u : 0;
        if (unpack_k) k_load(pk_of(it + 2), ui);
        if (unpack_v) v_load(pk_of(it + 1), ui);
        if constexpr (ROWS) {
          constexpr int kPre = 2, kAll = kCs + kP;
          f32x16_t sn;
          bf16x8_t kbuf[kPre], vbuf[kPre];
          float t[16];
          f32x4_t sv4;
          u32x4_t pn[2];
#pragma unroll
          for (int c = 0; c < kPre; ++c) {
            kbuf[c] = k_op(kd1, u1, c);
            vbuf[c] = v_op(c);
          }
          start(sn, sc1, u1);
          auto scores = [&](int q) {
            const f32x4_t a4 = scalar4(sc, 0, u, q), e4 = offset4(a4, sc, u, q);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const float c = fmaf(qsum, e4[j], m);
              t[4 * q + j] = fmaf(s[4 * q + j], a4[j], -c);
              if constexpr (MASK) {
                const int key = k0 + 8 * q + 4 * h + j;
                if (key > row_pos || key >= ke) t[4 * q + j] = -INFINITY;
              }
            }
            rmax = fmaxf(fmaxf(rmax, t[4 * q]), t[4 * q + 1]);
            rmax = fmaxf(fmaxf(rmax, t[4 * q + 2]), t[4 * q + 3]);
          };
          auto probs = [&](int i) {  // P s_v of two keys (FOLD: the scores carry log2(s_v), and the PV MFMA sums l)
            const float p0 = __builtin_amdgcn_exp2f(t[2 * i]), p1 = __builtin_amdgcn_exp2f(t[2 * i + 1]);
            if constexpr (FOLD) {
              pn[i >> 2][i & 3] = pack_bf16x2(p0, p1);
            } else {
              if (i % 2 == 0) sv4 = scalar4(sc, 2, u, i / 2);
              l += p0 + p1;
              pn[i >> 2][i & 3] = pack_bf16x2(p0 * sv4[2 * (i & 1)], p1 * sv4[2 * (i & 1) + 1]);
            }
          };
          constexpr int kCheck = kAll / 2 - 1;  // the last step beside which scores are made
#pragma unroll
          for (int c = 0; c < kAll; ++c) {
            if (c < 2 * kCs && c % 2 == 0) {
              const int q = c / 2;
              const bf16x8_t kop = kbuf[q % kPre];
              if (q + kPre < kCs) kbuf[q % kPre] = k_op(kd1, u1, q + kPre);
              sn = mfma32x32x16(kop, qop[q], sn);
            } else {
              const int v = c < 2 * kCs ? c / 2 : c - kCs, ct = v % (kCt + 1), ks = v / (kCt + 1);
              const bf16x8_t vop = vbuf[v % kPre];
              if (v + kPre < kP) vbuf[v % kPre] = v_op(v + kPre);
              acc[ct] = mfma32x32x16(vop, as_bf16x8(pop[ks]), acc[ct]);
            }
            if (c <= kCheck) {
#pragma unroll
              for (int q = 0; q < 4; ++q)
                if (q * (kCheck + 1) / 4 == c) scores(q);
            } else {
#pragma unroll
              for (int i = 0; i < 8; ++i)
                if (kCheck + 1 + i * (kAll - kCheck - 1) / 8 == c) probs(i);
            }
            if (unpack_k && c == kCheck) k_store(kd_of(2), ui);
            if (unpack_v && c == kCheck + 2) v_store(vt_of(1), ui);
          }
          s = sn;
          pop[0] = pn[0];
          pop[1] = pn[1];
          // (made here: the compiler would sink the exponentials and their sum past the tile's last branch)
          asm volatile("" : "+v"(pop[0]), "+v"(pop[1]));
          if constexpr (!FOLD) asm volatile("" : "+v"(l));
          pv = vt + u * Sh::kVs;
          pz = sc + 12 * KT + 256 * u;
        } else {
          if (unpack_k) k_store(kd_of(2), ui);
          if (unpack_v) v_store(vt_of(1), ui);
        }
      }
      scalars(it + 2, it & (kDualWaves - 1));
      ph = ph == 2 ? 0 : ph + 1;
    };
    // ---- prologue: tiles 0..3 requested, 0 and 1 unpacked (V of tile 0 only), S of the first sub-tile and its maximum
    auto prologue = [&](int pass) {
#pragma unroll
      for (int t = 0; t < Sh::kSlots; ++t) fetch(t);
      if constexpr (SPAN) wait_vmcnt<2 * Sh::kMax>();
      __syncthreads();
#pragma unroll
      for (int i = 0; i < Sh::kUnits; ++i) {
        k_load(pk_of(0), i);
        k_store(kd_of(0), i);
        k_load(pk_of(1), i);
        k_store(kd_of(1), i);
        v_load(pk_of(0), i);
        v_store(vt_of(0), i);
      }
      scalars(0, 0);
      scalars(1, 1);
      if constexpr (SPAN) locate(Sh::kSlots);
      __syncthreads();
      if (active) {
#pragma unroll
        for (int ct = 0; ct <= kCt; ++ct)
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[ct][i] = 0.f;
        l = 0.f;
        start(s, sc_of(0), 0);
#pragma unroll
        for (int cs = 0; cs < kCs; ++cs) s = mfma32x32x16(k_op(kd_of(0), 0, cs), qop[cs], s);
        float rm = -INFINITY;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x4_t a4 = scalar4(sc_of(0), 0, 0, q), e4 = offset4(a4, sc_of(0), 0, q);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int key = kb + 8 * q + 4 * h + j;
            const float v = fmaf(s[4 * q + j], a4[j], -(qsum * e4[j]));
            rm = fmaxf(rm, (nplain == 0 && (key > row_pos || key >= ke)) ? -INFINITY : v);
          }
        }
        if (pass == 0) m = halves_max(rm) + kDualBias;
      }
      pop[0] = pop[1] = u32x4_t{0u, 0u, 0u, 0u};
      pv = vt_of(0);
      pz = sc_of(0) + 12 * KT;
    };
    using Yes = std::true_type;
    using No = std::false_type;
    // One pass over the split's keys. A row's probabilities are taken relative to its first sub-tile's maximum plus
    // kDualBias; should a score exceed that by more than kDualHeadroom (fp32 holds l, the zero-point sum and the
    // accumulators over 2^17 keys up to it), the workgroup runs the split again with the rows' true maxima.
    for (int pass = 0; pass < 2; ++pass) {
      ph = 0;
      rmax = -INFINITY;
      prologue(pass);
      int it = 0;
      if (active) {
        for (; it < nplain; ++it) tile(it, Yes{}, No{});
        for (; it < ntiles; ++it) tile(it, Yes{}, Yes{});
#pragma unroll
        for (int c = 0; c < kP; ++c)  // the last sub-tile's PV
          acc[c % (kCt + 1)] = mfma32x32x16(v_op(c), as_bf16x8(pop[c / (kCt + 1)]), acc[c % (kCt + 1)]);
      } else {
        for (; it < ntiles; ++it) tile(it, No{}, No{});
      }
      if constexpr (SPAN) wait_vmcnt<0>();
      rmax = halves_max(rmax);
      if (pass == 1 || !__syncthreads_or(rmax > kDualHeadroom)) break;
      if (rmax > kDualHeadroom) m += rmax;
    }
  }

  // ---- epilogue: the zero-point sum (FOLD: and l) from the zero-point tile (FOLD: rows 0..2, lane half 0), store
  float csum = acc[kCt][0];
  if constexpr (FOLD) {
    csum = __shfl(csum, col, 64);
    l = __shfl(acc[kCt][1] + acc[kCt][2], col, 64);
  } else {
    l += shfl_xor_f(l, 32);
  }
  if (!active) return;
  float x[HS / 2];  // channel 16 k + 8 h + i at x[8 k + i]
#pragma unroll
  for (int i = 0; i < HS / 2; ++i) x[i] = acc[(i >> 5) + (i & 1) * (HS / 64)][4 * ((i >> 3) & 3) + ((i >> 1) & 3)] - csum;
  const int64_t head = kvh * G + jh;
  if (S == 1) {
    const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
    for (int i = 0; i < HS / 2; ++i) x[i] *= inv;
    if (p.osigns) {
      // x <- ((x H) D) * scale, the butterflies over channel bits in ascending order as rht_kernel runs them
      dual_butterfly(x, 1, 8);
      dual_butterfly_halves(x, h);
      dual_butterfly(x, 8, HS / 2);
#pragma unroll
      for (int i = 0; i < HS / 2; ++i) {
        const float y = x[i] * p.osigns[16 * (i >> 3) + 8 * h + (i & 7)];
        x[i] = y * p.out_scale;
      }
    }
    if (!valid) return;
    uint16_t *orow = p.out + (int64_t)(q0 + tok) * p.os0 + head * p.os1 + 8 * h;
#pragma unroll
    for (int i = 0; i < HS / 2; i += 4)  // (output rows are 8-byte aligned)
      *reinterpret_cast<u32x2_t *>(orow + 16 * (i >> 3) + (i & 7)) =
          u32x2_t{pack_bf16x2(x[i], x[i + 1]), pack_bf16x2(x[i + 2], x[i + 3])};
  } else {
    if (!valid) return;
    const int k = pf_partial_exponent(l);
#pragma unroll
    for (int i = 0; i < HS / 2; ++i) x[i] = __builtin_amdgcn_ldexpf(x[i], -k);
    float *orow = p.so + (int64_t)(q0 + tok) * p.sos0 + head * p.sos1 + (int64_t)split * HS + 8 * h;
#pragma unroll
    for (int i = 0; i < HS / 2; i += 4)
      *reinterpret_cast<float4 *>(orow + 16 * (i >> 3) + (i & 7)) = make_float4(x[i], x[i + 1], x[i + 2], x[i + 3]);
    if (h == 0) {
      const int64_t st = (int64_t)(q0 + tok) * p.sts0 + head * p.sts1 + split;
      p.smax[st] = m + (float)k;
      p.ssum[st] = __builtin_amdgcn_ldexpf(l, -k);
    }
  }
}

template <int HS, int KFMT, bool FOLD>
void launch_dual(const PrefillParams &p, dim3 grid, bool span, hipStream_t s) {
  if (span) prefill_dual_kernel<HS, KFMT, true, FOLD><<<grid, kDualThreads, 0, s>>>(p);
  else prefill_dual_kernel<HS, KFMT, false, FOLD><<<grid, kDualThreads, 0, s>>>(p);
}

// Whether the value scales are folded into the scores: at head 128 below 8 query heads per KV head, with a softmax scale
// that every stored key scale (1e-6 at least) leaves well above the smallest that can be divided by.
bool dual_folds(const PrefillParams &p, int head_size) {
  return head_size == 128 && p.num_q_heads / p.num_kv_heads < 8 && p.scale_log2 > 1e-20f;
}

int prefill_dual_rows() { return kDualRows; }

void prefill_dual(const PrefillParams &p, int head_size, int key_format, dim3 grid, bool span, hipStream_t s) {
  const uint32_t share = dual_share(grid.y * grid.z);
  grid.x = ((grid.x + (1u << share) - 1) >> share) << share;
  const bool i4 = key_format == QP_CODES_INT4;
  if (head_size == 64) {
    if (i4) launch_dual<64, QP_CODES_INT4, false>(p, grid, span, s);
    else launch_dual<64, QP_CODES_INT8, false>(p, grid, span, s);
  } else if (dual_folds(p, head_size)) {
    if (i4) launch_dual<128, QP_CODES_INT4, true>(p, grid, span, s);
    else launch_dual<128, QP_CODES_INT8, true>(p, grid, span, s);
  } else {
    if (i4) launch_dual<128, QP_CODES_INT4, false>(p, grid, span, s);
    else launch_dual<128, QP_CODES_INT8, false>(p, grid, span, s);
  }
}

}  // namespace qp
