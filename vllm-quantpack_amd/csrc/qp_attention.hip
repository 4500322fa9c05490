// One attention step of a batch, routed on the device: the entry point that stands in for unified_attention_int4.
//
// Reference: the stock unified_attention_int4 with the reference's router around it (int4_kv.py:294-329). The
// reference copies the step's lengths to the host once per step (_step_lengths, int4_kv.py:260-278), sends the
// decode / MTP rows to the split-KV kernel as a sub-batch (index tensors built on the host) and the long chunks to
// its FlashAttention prefill, rotating q before and the output after (single_rht, :307-329). Here the split is a
// route table written by one small kernel, which both kernels read, so the step has no host synchronisation:
//   * short sequences (1..QP_DECODE_MAX_QUERY query tokens) get consecutive rows of the caller's split-KV segment
//     buffers, or of the workspace when the batch can have more such rows than the buffers; the decode kernel serves
//     them in token groups and the merge writes their output;
//   * every other sequence takes the MFMA prefill kernel (or its query-slice path), which skips the short ones.
// One longer sequence alone goes to the prefill kernel without a table.
// A batch with short sequences only keeps the tokens' own rows and no table; where the segment buffers hold those rows it
// needs no workspace and can be recorded in a HIP graph as it is. The randomized Hadamard rotation is fused: the kernels rotate each query row as it loads
// and the merge / the prefill epilogue rotate the output back before the one bf16 store.
#include "qp_common.h"

#include <algorithm>
#include <mutex>

namespace qp {

// One workgroup. route_row[i]: first segment-buffer row of short sequence i, -1 for the others. row_tok / row_seq[r]: token
// and sequence of row r, -1 / 0 for unused rows. rows_cap holds every short sequence's rows as long as q has the rows that
// cu_q covers; a sequence past it is left to the prefill rather than written past the table.
__global__ __launch_bounds__(256) void route_kernel(const int32_t *cu_q, int num_seqs, int rows_cap,
                                                    int32_t *route_row, int32_t *row_tok, int32_t *row_seq) {
  __shared__ int scan[256];
  const int tid = threadIdx.x;
  for (int r = tid; r < rows_cap; r += 256) {
    row_tok[r] = -1;
    row_seq[r] = 0;
  }
  __syncthreads();  // the fill above precedes every row this workgroup writes below
  int base = 0;
  for (int s0 = 0; s0 < num_seqs; s0 += 256) {
    const int i = s0 + tid;
    const int q0 = i < num_seqs ? cu_q[i] : 0;
    const int T = i < num_seqs ? cu_q[i + 1] - q0 : 0;
    const int cnt = (T >= 1 && T <= QP_DECODE_MAX_QUERY) ? T : 0;
    scan[tid] = cnt;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {  // inclusive prefix sum over the 256 sequences of this round
      const int v = tid >= off ? scan[tid - off] : 0;
      __syncthreads();
      scan[tid] += v;
      __syncthreads();
    }
    const int first = base + scan[tid] - cnt;
    if (i < num_seqs) {
      const bool fits = cnt > 0 && first + cnt <= rows_cap;
      route_row[i] = fits ? first : -1;
      if (fits) {
        for (int t = 0; t < cnt; ++t) {
          row_tok[first + t] = q0 + t;
          row_seq[first + t] = i;
        }
      }
    }
    base += scan[255];
    __syncthreads();  // every thread has read scan before the next round overwrites it
  }
}

}  // namespace qp

using namespace qp;

namespace {

struct AttentionPlan {
  bool plain_decode;  // short sequences only: decode + merge on the tokens' own rows
  bool routed;        // a route table splits the batch between decode and prefill
  bool one_chunk;     // a single long sequence beside segment buffers: the prefill without a table
  int rows_cap;       // segment-buffer rows the route table hands out
  int64_t off_route, off_tok, off_seq, off_segm, off_prefill, total;
  int min_keys;       // floor of a segment's length
  int64_t segm_rows;  // rows of split-KV partials in the workspace (0: the caller's segment buffers hold them)
  qp_prefill_args prefill;
  qp_decode_args decode;
};

int64_t up256(int64_t x) { return (x + 255) / 256 * 256; }

// Split-KV partials in the workspace instead of the caller's segment buffers: [rows, heads, segments, head size] rows,
// then the maxima and the sums, fp32, each part 256-byte aligned.
int64_t segm_bytes(int64_t triples, int hs) { return up256(4 * triples * hs) + 2 * up256(4 * triples); }

void segm_in_workspace(AttentionPlan &P, const qp_paged_cache *cache, uint8_t *ws) {
  const int hs = cache->head_size;
  qp_decode_args &d = P.decode;
  const int64_t triples = P.segm_rows * d.num_q_heads * d.num_segments;
  d.segm_output = reinterpret_cast<float *>(ws + P.off_segm);
  d.segm_output_stride[2] = hs;
  d.segm_output_stride[1] = (int64_t)d.num_segments * hs;
  d.segm_output_stride[0] = (int64_t)d.num_q_heads * d.segm_output_stride[1];
  d.segm_max = reinterpret_cast<float *>(ws + P.off_segm + up256(4 * triples * hs));
  d.segm_expsum = reinterpret_cast<float *>(ws + P.off_segm + up256(4 * triples * hs) + up256(4 * triples));
  d.segm_stat_stride[1] = d.num_segments;
  d.segm_stat_stride[0] = (int64_t)d.num_q_heads * d.num_segments;
  d.segm_rows = (int32_t)P.segm_rows;
}

// The merge of d's partials into a's output, with the inverse rotation when a asks for one.
qp_merge_args merge_of(const qp_decode_args &d, const qp_attention_args *a, int hs) {
  qp_merge_args m = {};
  m.segm_output = d.segm_output;
  for (int i = 0; i < 3; ++i) m.segm_output_stride[i] = d.segm_output_stride[i];
  m.segm_max = d.segm_max;
  m.segm_expsum = d.segm_expsum;
  m.segm_stat_stride[0] = d.segm_stat_stride[0];
  m.segm_stat_stride[1] = d.segm_stat_stride[1];
  m.cu_seqlens_q = a->cu_seqlens_q;
  m.seqused_k = a->seqused_k;
  m.num_seqs = a->num_seqs;
  m.num_tokens = a->num_tokens;
  m.num_q_heads = a->num_q_heads;
  m.head_size = hs;
  m.num_segments = d.num_segments;
  m.out = a->out;
  m.out_stride[0] = a->out_stride[0];
  m.out_stride[1] = a->out_stride[1];
  m.rht_signs = a->rht_signs;
  m.rht_out_scale = a->rht_out_scale;
  return m;
}

AttentionPlan plan_attention(const qp_paged_cache *cache, const qp_attention_args *a) {
  AttentionPlan P = {};
  const int hs = cache->head_size;
  const int G = cache->num_kv_heads > 0 ? a->num_q_heads / cache->num_kv_heads : 0;
  const bool segm = a->segm_output && a->segm_max && a->segm_expsum && a->segm_rows > 0 && a->num_segments >= 1;
  const bool decode_shape =
      segm && (hs == 64 || hs == 128 || hs == 256 || hs == 512) && G >= 1 && G <= 32 && (hs != 512 || G <= 16);
  // Rows of partials that the batch's short sequences can have: q may have more rows than cu_seqlens_q covers (a padded
  // batch). On the tokens' own rows every row of q needs one, so a batch whose q has more than the segment buffers hold
  // and than its sequences can have is routed, which numbers the covered rows only.
  const int64_t cap = (int64_t)QP_DECODE_MAX_QUERY * a->num_seqs;
  const int64_t rows = a->num_tokens < cap ? a->num_tokens : cap;
  P.plain_decode = decode_shape && a->max_query_len >= 1 && a->max_query_len <= QP_DECODE_MAX_QUERY &&
                   a->max_query_len * G <= 32 && a->num_tokens <= std::max<int64_t>(a->segm_rows, cap);
  // A single sequence of more than QP_DECODE_MAX_QUERY tokens needs no table to go to the prefill kernel: the route kernel
  // and the decode and merge launches that find nothing to do took 10 us of 55 (512 tokens of 32 heads of 64 over 4096).
  // The workspace has the sequences' table, used or not: a batch with longer sequences always asks for one, which tells it
  // from a decode step (DecodePlan, qp_attention_noalloc), and a call without one stays refused.
  const bool tables = decode_shape && !P.plain_decode;
  P.one_chunk = tables && a->num_seqs == 1 && a->num_tokens > QP_DECODE_MAX_QUERY &&
                a->max_query_len > QP_DECODE_MAX_QUERY;
  P.routed = tables && !P.one_chunk;
  // The caller's segment buffers hold those partials when they have that many rows; otherwise the partials go to the
  // workspace, so every short sequence takes the split-KV kernel (an engine that allocates 128 / KV heads rows sends
  // larger batches than that: 64 sequences over up to 8192 keys at 32 q / 8 KV heads took 280 us with the 48 past the
  // buffers' 16 rows on the prefill kernel, 76 us here).
  P.rows_cap = P.routed ? (int)rows : 0;
  P.segm_rows = (P.plain_decode || P.routed) && rows > a->segm_rows ? rows : 0;

  qp_decode_args &d = P.decode;
  d.query = a->query;
  d.query_stride[0] = a->query_stride[0];
  d.query_stride[1] = a->query_stride[1];
  d.cu_seqlens_q = a->cu_seqlens_q;
  d.seqused_k = a->seqused_k;
  d.block_table = a->block_table;
  d.block_table_stride = a->block_table_stride;
  d.num_seqs = a->num_seqs;
  d.num_tokens = a->num_tokens;
  d.num_q_heads = a->num_q_heads;
  d.max_query_len = a->max_query_len;
  d.num_segments = a->num_segments;
  d.softmax_scale = a->softmax_scale;
  d.segm_output = a->segm_output;
  for (int i = 0; i < 3; ++i) d.segm_output_stride[i] = a->segm_output_stride[i];
  d.segm_max = a->segm_max;
  d.segm_expsum = a->segm_expsum;
  d.segm_stat_stride[0] = a->segm_stat_stride[0];
  d.segm_stat_stride[1] = a->segm_stat_stride[1];
  d.segm_rows = a->segm_rows;
  d.query_signs = a->rht_signs;
  // In mixed batches that fill the device with workgroups, segments have at least 512 keys (two 32-key chunks for each
  // of a workgroup's 8 waves): the segment count is the same for every sequence, half of a mixed batch's workgroups are
  // token groups without tokens, and segments of a chunk or two cost more to start and to merge than to stream. 24
  // decodes over 600 to 14500 keys beside a chunk (24 q / 4 KV heads of 256, int8 keys): 183 against 197 us. Batches of
  // short sequences alone are better without: their small segments fill the launch's tail (32 sequences over 2100 to
  // 65000 keys: 181 us, 185 with the floor; 64 over 270 to 7400 keys of 8 heads of 128: 70 and 73 us).
  P.min_keys = P.routed && 4 * (int64_t)a->num_seqs * cache->num_kv_heads >= device_cus() ? 512 : 0;
  if (P.segm_rows > 0) {  // no more segments than keep the device's CUs busy, as the workspace grows with them
    const int64_t pairs = (int64_t)a->num_seqs * cache->num_kv_heads;
    const int64_t want = (8 * (int64_t)device_cus() + pairs - 1) / pairs;
    if (want < d.num_segments) d.num_segments = (int)want;
  }

  qp_prefill_args &f = P.prefill;
  f.query = a->query;
  f.query_stride[0] = a->query_stride[0];
  f.query_stride[1] = a->query_stride[1];
  f.cu_seqlens_q = a->cu_seqlens_q;
  f.seqused_k = a->seqused_k;
  f.block_table = a->block_table;
  f.block_table_stride = a->block_table_stride;
  f.num_seqs = a->num_seqs;
  f.num_tokens = a->num_tokens;
  f.num_q_heads = a->num_q_heads;
  f.max_query_len = a->max_query_len;
  f.max_seqlen_k = a->max_seqlen_k;
  f.num_splits = 0;
  f.softmax_scale = a->softmax_scale;
  f.out = a->out;
  f.out_stride[0] = a->out_stride[0];
  f.out_stride[1] = a->out_stride[1];
  f.rht_signs = a->rht_signs;
  f.rht_out_scale = a->rht_out_scale;
  f.query_signs = a->rht_signs;

  // workspace: [route_row | row_tok | row_seq | split-KV partials | prefill workspace]
  P.off_route = 0;
  P.off_tok = tables ? up256(4 * (int64_t)a->num_seqs) : 0;
  P.off_seq = P.off_tok + (P.routed ? up256(4 * (int64_t)P.rows_cap) : 0);
  P.off_segm = P.off_seq + (P.routed ? up256(4 * (int64_t)P.rows_cap) : 0);
  P.off_prefill =
      P.off_segm + (P.segm_rows > 0 ? segm_bytes(P.segm_rows * a->num_q_heads * P.decode.num_segments, hs) : 0);
  const int64_t pf = P.plain_decode ? 0 : qp_prefill_workspace_size(cache, &f);
  P.total = pf > 0 ? P.off_prefill + up256(pf) : P.off_prefill;
  f.workspace_bytes = pf;
  return P;
}

}  // namespace

extern "C" int64_t qp_attention_workspace_size(const qp_paged_cache *cache, const qp_attention_args *a) {
  if (!cache || !a || a->num_seqs <= 0 || a->num_tokens <= 0) return 0;
  return plan_attention(cache, a).total;
}

extern "C" int qp_attention(const qp_paged_cache *cache, const qp_attention_args *a, qp_stream_t stream) {
  QP_REQUIRE(cache && a, "qp_attention: null argument");
  QP_REQUIRE(a->query && a->cu_seqlens_q && a->seqused_k && a->block_table && a->out, "qp_attention: null tensor");
  QP_REQUIRE(a->num_seqs >= 0 && a->num_tokens >= 0 && a->max_query_len >= 0, "qp_attention: bad sizes");
  QP_REQUIRE(cache->num_kv_heads > 0 && a->num_q_heads > 0 && a->num_q_heads % cache->num_kv_heads == 0,
             "qp_attention: query heads must be a multiple of KV heads");
  if (a->num_seqs == 0 || a->num_tokens == 0) return QP_OK;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  AttentionPlan P = plan_attention(cache, a);
  uint8_t *ws = static_cast<uint8_t *>(a->workspace);
  if (P.total > 0)
    QP_REQUIRE(ws && a->workspace_bytes >= P.total && aligned(ws, 256),
               "qp_attention: this batch needs a 256-byte aligned workspace of qp_attention_workspace_size bytes");
  if (P.segm_rows > 0) segm_in_workspace(P, cache, ws);
  const int G = a->num_q_heads / cache->num_kv_heads;
  const int max_rows = a->max_decode_rows > 0 && a->max_decode_rows < 32 ? a->max_decode_rows : 32;
  if (P.plain_decode) {
    // rows above the cap (or two row tiles at head 512) run as token groups on the tokens' own rows
    const int rows = a->max_query_len * G;
    const bool groups = rows > max_rows || (rows > 16 && cache->head_size == 512);
    int st = groups ? decode_routed(cache, &P.decode, nullptr, max_rows, P.min_keys, s) : decode_plain(cache, &P.decode, P.min_keys, s);
    if (st != QP_OK) return st;
    const qp_merge_args m = merge_of(P.decode, a, cache->head_size);
    // (rows of a padded q that no sequence covers have no partials in the workspace, and their output stays as it is)
    return merge_routed(&m, nullptr, nullptr, 0, nullptr, P.segm_rows > 0, P.min_keys, s);
  }
  P.prefill.workspace = P.prefill.workspace_bytes > 0 ? ws + P.off_prefill : nullptr;
  if (!P.routed) {
    if (P.one_chunk) {  // (segment buffers that a routed batch is refused for are refused here too)
      const int st = decode_check(cache, &P.decode);
      if (st != QP_OK) return st;
    }
    return prefill_run(cache, &P.prefill, nullptr, s);
  }

  int32_t *route_row = reinterpret_cast<int32_t *>(ws + P.off_route);
  int32_t *row_tok = reinterpret_cast<int32_t *>(ws + P.off_tok);
  int32_t *row_seq = reinterpret_cast<int32_t *>(ws + P.off_seq);
  route_kernel<<<1, 256, 0, s>>>(a->cu_seqlens_q, a->num_seqs, P.rows_cap, route_row, row_tok, row_seq);
  int st = launch_status();
  if (st != QP_OK) return st;
  st = prefill_run(cache, &P.prefill, route_row, s);
  if (st != QP_OK) return st;
  // mixed batches: groups of at most 16 rows (one row tile) whatever max_decode_rows says, as the host does not know
  // each short sequence's query count here
  st = decode_routed(cache, &P.decode, route_row, 16, P.min_keys, s);
  if (st != QP_OK) return st;
  const qp_merge_args m = merge_of(P.decode, a, cache->head_size);
  return merge_routed(&m, row_tok, row_seq, P.rows_cap, nullptr, false, P.min_keys, s);
}

// ------------------------------------------------------------------------------ entry point without allocation
//
// The split-KV partials of qp_attention_noalloc live in this file-scope device array: one copy per GPU the library
// runs on, held until the process ends. Host code never passes `scratch` itself to a kernel (in host code the name
// stands for a host-side shadow, not a device address): each device's address comes from hipGetSymbolAddress, taken
// once per device with that device current, and only that pointer is used.
static __device__ __align__(256) uint8_t scratch[QP_NOALLOC_SCRATCH_BYTES];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void *g_scratch_ptr[kMaxDevices] = {};

// The current device's address of `scratch`, looked up on the device's first call.
int scratch_on_current_device(void **ptr) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail((int)e, std::string("qp_attention_noalloc: hipGetDevice: ") + hipGetErrorString(e));
  QP_SUPPORTED(dev >= 0 && dev < kMaxDevices, "qp_attention_noalloc: device index beyond 63");
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail(e != hipSuccess ? (int)e : QP_ERR_INVALID,
                  std::string("qp_attention_noalloc: hipGetSymbolAddress: ") + hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *ptr = g_scratch_ptr[dev];
  return QP_OK;
}

}  // namespace

extern "C" int qp_attention_noalloc(const qp_paged_cache *cache, const qp_attention_args *args, qp_stream_t stream) {
  QP_REQUIRE(cache && args, "qp_attention_noalloc: null argument");
  QP_REQUIRE(args->num_seqs >= 0 && args->num_tokens >= 0 && args->num_q_heads > 0 && cache->num_kv_heads > 0 &&
                 args->num_q_heads % cache->num_kv_heads == 0,
             "qp_attention_noalloc: bad sizes");
  const int hs = cache->head_size;
  const int G = args->num_q_heads / cache->num_kv_heads;
  QP_SUPPORTED(args->max_query_len >= 1 && args->max_query_len <= QP_DECODE_MAX_QUERY &&
                   args->max_query_len * G <= 32,
               "qp_attention_noalloc: only batches of sequences with 1..4 query tokens and at most 32 query rows per "
               "KV head (a decode step)");
  QP_SUPPORTED(hs == 64 || hs == 128 || hs == 256 || hs == 512,
               "qp_attention_noalloc: head size must be 64, 128, 256 or 512");
  QP_SUPPORTED(hs != 512 || G <= 16, "qp_attention_noalloc: head 512 takes at most 16 query heads per KV head");
  QP_REQUIRE(args->num_segments >= 1 && args->num_segments <= 2048, "qp_attention_noalloc: 1..2048 segments");
  // [segment rows: tokens x heads x segments x head_size | maxima | sums], fp32, each part 256-byte aligned
  const int64_t triples = (int64_t)args->num_tokens * args->num_q_heads * args->num_segments;
  const int64_t rows_bytes = (triples * hs * 4 + 255) / 256 * 256;
  const int64_t stat_bytes = (triples * 4 + 255) / 256 * 256;
  const int64_t need = rows_bytes + 2 * stat_bytes;
  if (need > QP_NOALLOC_SCRATCH_BYTES)
    return fail(QP_ERR_UNSUPPORTED, "qp_attention_noalloc: the batch's split-KV partials need " + std::to_string(need) +
                                        " bytes, more than the " + std::to_string(QP_NOALLOC_SCRATCH_BYTES) +
                                        "-byte static buffer (fewer segments, or qp_attention with caller buffers)");
  if (args->num_seqs == 0 || args->num_tokens == 0) return QP_OK;
  void *base = nullptr;
  const int st = scratch_on_current_device(&base);
  if (st != QP_OK) return st;
  qp_attention_args a = *args;
  float *rows = static_cast<float *>(base);
  a.segm_output = rows;
  a.segm_output_stride[2] = hs;
  a.segm_output_stride[1] = (int64_t)args->num_segments * hs;
  a.segm_output_stride[0] = (int64_t)args->num_q_heads * a.segm_output_stride[1];
  a.segm_max = reinterpret_cast<float *>(static_cast<uint8_t *>(base) + rows_bytes);
  a.segm_expsum = reinterpret_cast<float *>(static_cast<uint8_t *>(base) + rows_bytes + stat_bytes);
  a.segm_stat_stride[1] = args->num_segments;
  a.segm_stat_stride[0] = (int64_t)args->num_q_heads * args->num_segments;
  a.segm_rows = args->num_tokens;
  a.workspace = nullptr;
  a.workspace_bytes = 0;
  // a batch of short sequences whose rows all fit: qp_attention's decode + merge, which needs no workspace
  QP_SUPPORTED(qp_attention_workspace_size(cache, &a) == 0, "qp_attention_noalloc: not a batch of short sequences");
  return qp_attention(cache, &a, stream);
}
