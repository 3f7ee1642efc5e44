// C ABI of the FlashPrefill gfx950 path: argument validation, workspace
// layout and the launch sequence plan -> pool -> search -> attention. All
// launches go to the caller's stream; nothing here allocates or synchronises
// (except fp_read_status, which is documented to).
#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <mutex>
#include <string>

#include <algorithm>

#include "fp_internal.h"

namespace {

thread_local std::string g_last_error;

int fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
int fail(int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_last_error = buf;
  return code;
}

int hip_fail(hipError_t e, const char* what) {
  return fail(FP_E_LAUNCH, "%s: %s", what, hipGetErrorString(e));
}

size_t align_up(size_t x) { return (x + 255) & ~static_cast<size_t>(255); }

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int64_t elem_bytes(int dtype) { return dtype == FP_DTYPE_F32 ? 4 : 2; }

// Block size of the plan, the work items, the index lists and the attention:
// block_size itself for 64 and 128; for 256, selection blocks of 256 tokens
// (pooling, scoring, selection) over a 128-token plan, the selection writing
// each 256-row's list as the lists of its two 128-token rows (ratio 2), so
// that the attention walks 128-key tiles as the reference's kernels do.
int plan_block(const fp_problem* p) { return p->block_size == 256 ? 128 : p->block_size; }
int block_ratio(const fp_problem* p) { return p->block_size / plan_block(p); }

int validate(const fp_problem* p) {
  if (!p) return fail(FP_E_INVALID_ARG, "problem descriptor is NULL");
  if (!p->q || !p->k || !p->v || !p->o) return fail(FP_E_INVALID_ARG, "q/k/v/o must be non-NULL");
  if (p->dtype != FP_DTYPE_BF16 && p->dtype != FP_DTYPE_F16 && p->dtype != FP_DTYPE_F32)
    return fail(FP_E_UNSUPPORTED, "dtype %d unsupported (bf16, fp16 or fp32)", p->dtype);
  if (p->head_dim != 64 && p->head_dim != 128 && p->head_dim != 256)
    return fail(FP_E_UNSUPPORTED, "head_dim %d unsupported (64, 128 or 256)", p->head_dim);
  // head_dim 256 is built for bf16 / fp16 at blocks of 64 and 128: the fp32
  // kernels' padded 128-row tiles (133 KB each) and a 256-row, d = 256 query
  // block (128 KB) do not fit the 160 KB of LDS beside the rest
  if (p->head_dim == 256 && p->dtype == FP_DTYPE_F32)
    return fail(FP_E_UNSUPPORTED, "head_dim 256 is supported for bf16 and fp16 inputs, not fp32");
  if (p->head_dim == 256 && p->block_size == 256)
    return fail(FP_E_UNSUPPORTED, "head_dim 256 is supported at block_size 64 and 128, not 256");
  if (p->block_size != 64 && p->block_size != 128 && p->block_size != 256)
    return fail(FP_E_UNSUPPORTED, "block_size %d unsupported (64, 128 or 256)", p->block_size);
  if (p->num_q_heads < 1 || p->num_kv_heads < 1 || p->num_q_heads % p->num_kv_heads)
    return fail(FP_E_INVALID_ARG, "num_q_heads (%d) must be a positive multiple of num_kv_heads (%d)",
                p->num_q_heads, p->num_kv_heads);
  if (p->batch < 1 || p->batch > fp::kMaxBatch)
    return fail(FP_E_INVALID_ARG, "batch %d outside [1, %d]", p->batch, fp::kMaxBatch);
  if (p->max_seq_len < 1 || p->max_seq_len > fp::kMaxBlocks * plan_block(p))
    return fail(FP_E_INVALID_ARG, "max_seq_len %d outside [1, %d] (%d blocks of %d tokens)",
                p->max_seq_len, fp::kMaxBlocks * plan_block(p), fp::kMaxBlocks, plan_block(p));
  if (p->dtype == FP_DTYPE_F32 && p->block_size == 256) {
    // the fp32 search holds the 256-row query block (rows padded by 16 bytes)
    // and a row's fp32 (p, m) in LDS
    const int64_t nb = (p->max_seq_len + 127) / 128;
    const int64_t lds = 256 * (static_cast<int64_t>(p->head_dim) + 4) * 4 + 8 * nb;
    if (lds > 160 * 1024)
      return fail(FP_E_UNSUPPORTED, "fp32 inputs at block_size 256 support up to %lld tokens at "
                  "head_dim %d", static_cast<long long>((160 * 1024 - 256 * (p->head_dim + 4) * 4) / 8 * 128),
                  p->head_dim);
  }
  if (p->total_tokens < 0) return fail(FP_E_INVALID_ARG, "total_tokens < 0");
  if (!p->cu_seqlens) {
    if (p->uniform_seq_len < 0 || p->uniform_seq_len > p->max_seq_len)
      return fail(FP_E_INVALID_ARG, "uniform_seq_len %d outside [0, max_seq_len]", p->uniform_seq_len);
    if (static_cast<int64_t>(p->batch) * p->uniform_seq_len > p->total_tokens)
      return fail(FP_E_INVALID_ARG, "batch * uniform_seq_len exceeds total_tokens");
  }
  if (!aligned16(p->q) || !aligned16(p->k) || !aligned16(p->v) || !aligned16(p->o))
    return fail(FP_E_INVALID_ARG, "q/k/v/o must be 16-byte aligned");
  const int64_t strides[8] = {p->q_stride_tok, p->q_stride_head, p->k_stride_tok, p->k_stride_head,
                              p->v_stride_tok, p->v_stride_head, p->o_stride_tok, p->o_stride_head};
  const int64_t vec = 16 / elem_bytes(p->dtype);  // elements per 16 bytes
  for (int s = 0; s < 8; ++s)
    if (strides[s] < 0 || strides[s] % vec)
      return fail(FP_E_INVALID_ARG, "strides must be non-negative multiples of 16 bytes "
                                    "(%lld elements)", static_cast<long long>(vec));
  for (int s = 0; s < 8; ++s)
    if (strides[s] >= (int64_t(1) << 24))
      return fail(FP_E_UNSUPPORTED, "strides of 2^24 elements or more are not supported");
  if (p->min_budget < 0) return fail(FP_E_INVALID_ARG, "min_budget < 0");
  if (p->native_normalize != 0 && p->native_normalize != 1)
    return fail(FP_E_INVALID_ARG, "native_normalize must be 0 or 1");
  return FP_OK;
}

// Chunk slots per row of the fp32 attention and list entries per chunk. A
// problem of few rows would wait for its longest one (the card runs two
// workgroups per CU, 512 at once), and unlike the 16-bit split rows any row may
// be dense here, so every row gets 1536 / rows slots: 4K tokens x 8 heads, 256
// rows, d = 64: attention 169 us with 2 slots, 101 with 4, 98 with 6, 109 with
// 7 (more partials). From 769 rows on there is one slot. The partials are
// held to kF32PartialBytes and, with the rest of the workspace (`base` bytes),
// to the static scratch of fp_flashprefill_noalloc, so that no problem outgrows
// it for their sake.
struct F32Split {
  int chunks, blocks;
  size_t bytes;
};
F32Split f32_split(const fp_problem* p, int64_t nb_max, int64_t cap, size_t base) {
  constexpr int64_t kSlots = 1536;
  constexpr size_t kF32PartialBytes = size_t(64) << 20;
  F32Split r = {1, static_cast<int>(nb_max), 0};
  if (p->dtype != FP_DTYPE_F32) return r;
  const int64_t blk = plan_block(p), rows = p->num_q_heads * cap;
  const size_t per = static_cast<size_t>(rows) * 4 * (blk * p->head_dim + 2 * blk);
  int64_t n = std::min<int64_t>({fp::kF32MaxChunks, kSlots / rows, nb_max});
  n = std::min<int64_t>(n, kF32PartialBytes / per);
  if (n < 2 || base + n * per + 512 > FP_NOALLOC_SCRATCH_BYTES) return r;
  r.chunks = static_cast<int>(n);
  r.blocks = static_cast<int>((nb_max + n - 1) / n);
  r.bytes = n * per;
  return r;
}

int layout(const fp_problem* p, fp_ws_layout* L) {
  const int rc = validate(p);
  if (rc != FP_OK) return rc;
  memset(L, 0, sizeof(*L));
  const int64_t B = p->batch;
  const int64_t blk = plan_block(p);
  const int64_t nb_max = (p->max_seq_len + blk - 1) / blk;
  int64_t cap = (p->total_tokens + (blk - 1) * B) / blk;
  if (cap > B * nb_max) cap = B * nb_max;
  if (cap < 1) cap = 1;
  const int64_t full = cap / nb_max, rem = cap % nb_max;
  const int64_t tri = full * nb_max * (nb_max + 1) / 2 + rem * (rem + 1) / 2;
  L->nb_max = static_cast<int32_t>(nb_max);
  L->nb_sum_cap = cap;
  L->tri_cap = tri;
  const int64_t Hq = p->num_q_heads, Hkv = p->num_kv_heads, d = p->head_dim;
  if (Hq * cap > (int64_t(1) << 31)) return fail(FP_E_INVALID_ARG, "too many work items");
  if (Hq * tri >= (int64_t(1) << 31))
    return fail(FP_E_UNSUPPORTED, "index lists of 2^31 entries or more are not supported");
  // the search forms a lane's pooled-key offset (one chunk row of nb_sum_cap
  // 16-byte entries, plus a key) in 32 bits; the batch and length bounds of
  // validate() keep nb_sum_cap <= 4096 * 8192 = 2^25, this guards the rule
  const int64_t eb = elem_bytes(p->dtype);
  if (cap >= (int64_t(1) << 26))
    return fail(FP_E_UNSUPPORTED, "2^26 or more key blocks in one call are not supported");
  size_t off = 0;
  L->status_off = off;     off = align_up(off + 4);
  L->seq_tile_off = off;   off = align_up(off + 8 * (B + 1));
  L->seq_tri_off = off;    off = align_up(off + 8 * (B + 1));
  L->seq_start_off = off;  off = align_up(off + 8 * B);
  L->seq_len_off = off;    off = align_up(off + 4 * B);
  L->items_off = off;      off = align_up(off + sizeof(fp::ItemRec) * cap);
  L->mk_off = off;         off = align_up(off + eb * cap * Hkv * d);
  L->cnt_off = off;        off = align_up(off + 4 * Hq * cap);
  L->rowrec_off = off;     off = align_up(off + 16 * Hq * cap);
  L->idx_off = off;        off = align_up(off + 4 * Hq * tri);
  // Split rows (16-bit inputs, fp::UnitRec): a last_n row selects every causal
  // block, so with one workgroup per row it can outlast the rest of the
  // attention. Rows of more than C blocks run as chunks of at most C blocks.
  // C is about one workgroup slot's share of the attention, estimated from
  // below before the selection exists: every row's forced blocks (sink,
  // window and min_budget; at least the diagonal) plus the last_n rows' full
  // lists, over the resident slots of an MI355X (256 CUs; two workgroups each at
  // d = 64 as well, where three are resident: the count only sets the balance). A
  // chunk longer than a slot's share becomes the kernel's
  // critical path (one TP = 8 shard of a 128K sequence, 4 q / 1 kv heads:
  // attention 0.80 ms with 256-block chunks, 0.74 ms with 64); a much shorter
  // one adds per-chunk work (first loads, partial store, merge; 16-block
  // chunks made the same shard at 32K 4 % slower than 64). C is at least 8
  // and gives at most kMaxChunks chunks, evened out over the longest row
  // (Llama shapes, 32 heads: two chunks from 4K on, 4K call -5 %). At most
  // min(B, cap / (C + 1)) sequences have more than C blocks. Each chunk unit
  // keeps fp32 partials per query head (blk * d + 2 * blk floats), and their
  // region is held to kSplitPartialBytes: a batch whose units would need more
  // has enough long rows to balance the attention grid without splitting.
  constexpr int64_t kSplitPartialBytes = int64_t(64) << 20;
  constexpr int64_t kCUs = 256;
  int64_t split = 0, units = 0;
  if (p->dtype != FP_DTYPE_F32 && p->last_n_block > 0) {
    const int64_t slots = kCUs * ((blk == 128 ? 2 : 4) / (d == 256 ? 2 : 1));
    const int64_t forced = std::min<int64_t>(
        nb_max, std::max<int64_t>(1, static_cast<int64_t>(std::max(p->attention_sink, 0)) +
                                         std::max(p->window_size, 0) + std::max(p->min_budget, 0)));
    const int64_t work = Hq * cap * (forced + std::min<int64_t>(p->last_n_block, nb_max));
    split = std::max<int64_t>({8, (work + slots - 1) / slots,
                               (nb_max + fp::kMaxChunks - 1) / fp::kMaxChunks});
    const int64_t nchunks = (nb_max + split - 1) / split;
    split = std::max<int64_t>(8, (nb_max + nchunks - 1) / nchunks);
    if (nb_max > split) {
      const int64_t seqs = std::min<int64_t>(B, cap / (split + 1));
      const int64_t rows = seqs * std::min<int64_t>(p->last_n_block, nb_max);
      units = rows * ((nb_max + split - 1) / split);
      if (units * Hq * 4 * (blk * d + 2 * blk) > kSplitPartialBytes) units = 0;
    }
    if (units == 0) split = 0;
  }
  L->split_blocks = static_cast<int32_t>(split);
  L->unit_cap = units;
  // units region: count and queue words, the unit records, then one arrival
  // counter per (head, unit) for the split rows merged inside the attention
  L->units_off = off;      off = align_up(off + 64 + sizeof(fp::UnitRec) * units + 4 * Hq * units);
  L->part_off = off;
  off = align_up(off + (p->dtype == FP_DTYPE_F32 ? f32_split(p, nb_max, cap, off).bytes
                                                 : 4 * Hq * units * (blk * d + 2 * blk)));
  L->total_bytes = off;
  return FP_OK;
}

fp::SeqTables tables(const fp_ws_layout& L, void* ws) {
  char* base = static_cast<char*>(ws);
  fp::SeqTables t;
  t.status = reinterpret_cast<uint32_t*>(base + L.status_off);
  t.seq_tile = reinterpret_cast<int64_t*>(base + L.seq_tile_off);
  t.seq_tri = reinterpret_cast<int64_t*>(base + L.seq_tri_off);
  t.seq_start = reinterpret_cast<int64_t*>(base + L.seq_start_off);
  t.seq_len = reinterpret_cast<int32_t*>(base + L.seq_len_off);
  t.items = reinterpret_cast<fp::ItemRec*>(base + L.items_off);
  return t;
}

// Workgroups of the attention kernel per CU: waves per SIMD x 4 SIMDs / waves per
// workgroup.
int64_t resident_per_cu(int block, int head_dim) {
  return (head_dim == 256 ? 4 : head_dim == 64 ? 12 : 8) / (block / 32);
}

// Workgroups of the attention kernel resident on the current device at once:
// two per CU at block 128 (64 KB of LDS, 4 waves), four at block 64 (32 KB,
// 2 waves), half that at d = 256 (one wave per SIMD, twice the LDS), half as
// many again at d = 64 (three waves per SIMD, half the LDS), rounded up to a
// multiple of the 8 XCDs. The CU count is read once per device.
int resident_attn_workgroups(int block, int head_dim, int64_t* out) {
  constexpr int kDevs = 64;
  static std::mutex mu;
  static int cus[kDevs] = {};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
  if (dev < 0 || dev >= kDevs) return fail(FP_E_UNSUPPORTED, "device index %d", dev);
  std::lock_guard<std::mutex> lock(mu);
  if (cus[dev] == 0) {
    int n = 0;
    e = hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return hip_fail(e, "hipDeviceGetAttribute(CU count)");
    if (n < 1) return fail(FP_E_LAUNCH, "device reports %d CUs", n);
    cus[dev] = n;
  }
  *out = (cus[dev] * resident_per_cu(block, head_dim) + 7) / 8 * 8;
  return FP_OK;
}

float sm_scale_log2(int head_dim) {
  // fp32(1/sqrt(d)) * fp32(log2 e) in fp32, as the reference kernels compute it
  const float scale = static_cast<float>(1.0 / sqrt(static_cast<double>(head_dim)));
  const float log2e = static_cast<float>(1.4426950408889634);
  volatile float prod = scale * log2e;
  return prod;
}

int prepare(const fp_problem* p, void* ws, fp_ws_layout* L) {
  const int rc = layout(p, L);
  if (rc != FP_OK) return rc;
  if (!ws) return fail(FP_E_INVALID_ARG, "workspace is NULL");
  if (!aligned16(ws)) return fail(FP_E_INVALID_ARG, "workspace must be 16-byte aligned");
  return FP_OK;
}

int32_t* arrival_counters(const fp_problem* p, const fp_ws_layout& L, void* ws) {
  (void)p;
  return reinterpret_cast<int32_t*>(static_cast<char*>(ws) + L.units_off + 64 +
                                    sizeof(fp::UnitRec) * L.unit_cap);
}

fp::PlanArgs plan_args(const fp_problem* p, const fp_ws_layout& L, void* ws) {
  fp::PlanArgs a;
  a.tab = tables(L, ws);
  a.cu = p->cu_seqlens;
  a.B = p->batch;
  a.uniform_len = p->uniform_seq_len;
  a.max_seq_len = p->max_seq_len;
  a.nb_max = L.nb_max;
  a.total_tokens = p->total_tokens;
  a.nb_sum_cap = L.nb_sum_cap;
  a.block = plan_block(p);
  a.last_n = p->last_n_block;
  a.split_blocks = L.split_blocks;
  a.units = reinterpret_cast<int32_t*>(static_cast<char*>(ws) + L.units_off);
  a.unit_cap = L.unit_cap;
  a.arrivals = arrival_counters(p, L, ws);
  a.n_arrivals = static_cast<int64_t>(p->num_q_heads) * L.unit_cap;
  return a;
}

int run_plan(const fp_problem* p, const fp_ws_layout& L, void* ws, hipStream_t s) {
  const hipError_t e = fp::launch_plan(plan_args(p, L, ws), s);
  return e == hipSuccess ? FP_OK : hip_fail(e, "plan launch");
}

fp::PoolArgs pool_args(const fp_problem* p, const fp_ws_layout& L, void* ws) {
  fp::PoolArgs a;
  a.tab = tables(L, ws);
  a.k = static_cast<const uint16_t*>(p->k);
  a.kst = p->k_stride_tok;
  a.khs = p->k_stride_head;
  a.mk = reinterpret_cast<uint16_t*>(static_cast<char*>(ws) + L.mk_off);
  a.nb_sum_cap = L.nb_sum_cap;
  a.B = p->batch;
  a.Hkv = p->num_kv_heads;
  a.block = plan_block(p);
  a.ratio = block_ratio(p);
  return a;
}

int run_pool(const fp_problem* p, const fp_ws_layout& L, void* ws, hipStream_t s) {
  const hipError_t e = fp::launch_pool(pool_args(p, L, ws), p->dtype, p->head_dim,
                                       L.nb_sum_cap, s);
  return e == hipSuccess ? FP_OK : hip_fail(e, "pool launch");
}

fp::SearchArgs search_args(const fp_problem* p, const fp_ws_layout& L, void* ws) {
  fp::SearchArgs a;
  memset(&a, 0, sizeof(a));
  char* base = static_cast<char*>(ws);
  a.tab = tables(L, ws);
  a.q = static_cast<const uint16_t*>(p->q);
  a.qst = p->q_stride_tok;
  a.qhs = p->q_stride_head;
  a.mk = reinterpret_cast<const uint16_t*>(base + L.mk_off);
  a.idx = reinterpret_cast<int32_t*>(base + L.idx_off);
  a.cnt = reinterpret_cast<int32_t*>(base + L.cnt_off);
  a.rowrec = reinterpret_cast<int32_t*>(base + L.rowrec_off);
  a.tri_cap = L.tri_cap;
  a.nb_sum_cap = L.nb_sum_cap;
  a.B = p->batch;
  a.Hq = p->num_q_heads;
  a.Hkv = p->num_kv_heads;
  a.nb_max = L.nb_max;
  a.sm_scale_log2 = sm_scale_log2(p->head_dim);
  a.alpha = p->alpha;
  a.sink = p->attention_sink;
  a.window = p->window_size;
  a.last_n = p->last_n_block;
  a.native = p->native_normalize;
  a.min_budget = p->min_budget;
  return a;
}

int run_search(const fp_problem* p, const fp_ws_layout& L, void* ws, float* dp, float* dm,
               const float* in_p, const float* in_m, hipStream_t s) {
  fp::SearchArgs a = search_args(p, L, ws);
  a.dump_p = dp;
  a.dump_m = dm;
  a.in_p = in_p;
  a.in_m = in_m;
  const bool from_scores = in_p != nullptr;
  const hipError_t e = fp::launch_search(a, p->dtype, p->head_dim, p->block_size,
                                         static_cast<int64_t>(p->num_q_heads) * L.nb_sum_cap,
                                         from_scores, s);
  return e == hipSuccess ? FP_OK : hip_fail(e, "search launch");
}

// Whether the rules alone keep every block of every row, whatever the scores:
// every row is one of its sequence's last_n rows or has no block between the
// sink and the window, in sequences of up to nb_max blocks (2 + 4 + 2 blocks,
// i.e. 1,024 tokens, with the callers' settings). Selection blocks of 256 tokens
// are left to the search.
bool every_row_full(const fp_problem* p, const fp_ws_layout& L) {
  const int64_t rules = static_cast<int64_t>(std::max(p->attention_sink, 0)) +
                        std::max(p->window_size, 0) + std::max(p->last_n_block, 0);
  return block_ratio(p) == 1 && L.nb_max <= rules;
}

// Everything of a whole-operator call before the attention. At most
// kSmallPlanBatch sequences plan and pool in one launch (k_plan_pool), where the
// plan's own launch and latency are a visible part of a short call, and write the
// selection there too when it does not depend on the scores: a 1K call then has
// two launches instead of three (39.8 -> 33 us, 32 q / 8 kv heads; the search
// alone took 7).
int run_before_attention(const fp_problem* p, const fp_ws_layout& L, void* ws, hipStream_t s) {
  int rc;
  if (p->batch <= fp::kSmallPlanBatch) {
    const fp::SearchArgs sa = search_args(p, L, ws);
    const fp::FullRowsArgs f = {every_row_full(p, L) ? 1 : 0, sa.Hq, sa.idx, sa.cnt, sa.rowrec,
                                sa.tri_cap};
    const hipError_t e = fp::launch_plan_pool(plan_args(p, L, ws), pool_args(p, L, ws), f, p->dtype,
                                              p->head_dim, s);
    if (e != hipSuccess) return hip_fail(e, "plan + pool launch");
    if (f.on) return FP_OK;
  } else {
    if ((rc = run_plan(p, L, ws, s)) != FP_OK) return rc;
    if ((rc = run_pool(p, L, ws, s)) != FP_OK) return rc;
  }
  return run_search(p, L, ws, nullptr, nullptr, nullptr, nullptr, s);
}

int run_attn(const fp_problem* p, const fp_ws_layout& L, void* ws, hipStream_t s) {
  if (p->total_tokens == 0) return FP_OK;  // no rows; the kernels assume a non-empty K
  fp::AttnArgs a;
  char* base = static_cast<char*>(ws);
  a.tab = tables(L, ws);
  a.q = static_cast<const uint16_t*>(p->q);
  a.k = static_cast<const uint16_t*>(p->k);
  a.v = static_cast<const uint16_t*>(p->v);
  a.o = static_cast<uint16_t*>(p->o);
  a.qst = p->q_stride_tok;
  a.qhs = p->q_stride_head;
  a.kst = p->k_stride_tok;
  a.khs = p->k_stride_head;
  a.vst = p->v_stride_tok;
  a.vhs = p->v_stride_head;
  a.ost = p->o_stride_tok;
  a.ohs = p->o_stride_head;
  a.idx = reinterpret_cast<const int32_t*>(base + L.idx_off);
  a.cnt = reinterpret_cast<const int32_t*>(base + L.cnt_off);
  a.rowrec = reinterpret_cast<const int32_t*>(base + L.rowrec_off);
  a.tri_cap = L.tri_cap;
  a.nb_sum_cap = L.nb_sum_cap;
  a.B = p->batch;
  a.Hq = p->num_q_heads;
  a.Hkv = p->num_kv_heads;
  a.sm_scale_log2 = sm_scale_log2(p->head_dim);
  a.last_n = p->last_n_block;
  a.split_blocks = L.split_blocks;
  a.units = reinterpret_cast<const int32_t*>(base + L.units_off);
  a.part = reinterpret_cast<float*>(base + L.part_off);
  a.unit_cap = L.unit_cap;
  a.unit_slots = (static_cast<int64_t>(p->num_q_heads) * L.unit_cap + 7) / 8 * 8;
  a.total_slots = a.unit_slots + fp::attn_grid(p->num_q_heads, p->num_kv_heads, L.nb_sum_cap);
  a.queue = reinterpret_cast<int32_t*>(base + L.units_off) + fp::kQueueOff;
  // The chunks of a split row combine their partials themselves (the last to
  // finish reads the others' from L2) when they all run on one XCD: with Hq a
  // multiple of 8 the unit slots of head h are the slots of XCD h / (Hq / 8)
  // (map_item), which share one L2; and when a row has at most
  // kMaxInlineChunks chunks. Otherwise k_merge runs after the attention.
  a.arrivals = arrival_counters(p, L, ws);
  const int64_t max_chunks =
      L.split_blocks > 0 ? (L.nb_max + L.split_blocks - 1) / L.split_blocks : 0;
  a.merge_inline = p->num_q_heads % 8 == 0 && max_chunks <= fp::kMaxInlineChunks ? 1 : 0;
  a.ratio = block_ratio(p);
  const int blk = plan_block(p);
  hipError_t e;
  a.f32_chunks = 1;
  a.f32_chunk_blocks = L.nb_max;
  if (p->dtype == FP_DTYPE_F32) {
    const F32Split sp = f32_split(p, L.nb_max, L.nb_sum_cap, L.part_off);
    a.f32_chunks = sp.chunks;
    a.f32_chunk_blocks = sp.blocks;
    a.total_slots *= sp.chunks;
    e = fp::launch_attn_f32(a, p->head_dim, blk, s);
  } else {
    // Persistent grid (every resident workgroup loops over its XCD's queue)
    // once there are at least 4 slots per resident workgroup: it saves the
    // dispatcher's gap between a finished row and the next workgroup
    // (128K attention -3 to -4.5 %, 16K -1.7 %, 8K call -1.4 %). Below that,
    // one workgroup per slot (4K, 2.5 slots per workgroup: the persistent
    // loop's per-slot claim costs more than it saves, +3 %).
    int64_t resident = 0;
    const int rc = resident_attn_workgroups(blk, p->head_dim, &resident);
    if (rc != FP_OK) return rc;
    const bool persist = a.total_slots >= 4 * resident;
    const int64_t grid = persist ? resident : a.total_slots;
    e = fp::launch_attn(a, p->dtype, p->head_dim, blk, grid, persist, s);
  }
  if (e == hipSuccess && L.split_blocks > 0 && !a.merge_inline)
    e = fp::launch_merge(a, p->dtype, p->head_dim, blk, s);
  return e == hipSuccess ? FP_OK : hip_fail(e, "attention launch");
}

}  // namespace

// Static device scratch of the allocation-free entry point: the workspace of
// fp_flashprefill_noalloc (every region of fp_ws_layout) lives in this array,
// one copy per GPU, held until the process ends. Host code never uses the
// array's name as an address: the device address of each GPU's copy is read
// once per device with hipGetSymbolAddress (with that device current) and
// kept in g_scratch_ptr. Nothing in the workspace has to start at zero (the
// plan kernel writes every table and counter the later kernels read), so the
// scratch is never cleared; calls that overlap on one GPU share it and race.
static __device__ __align__(256) unsigned char scratch[FP_NOALLOC_SCRATCH_BYTES];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

int scratch_on_current_device(void** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
  if (dev < 0 || dev >= kMaxDevices) return fail(FP_E_UNSUPPORTED, "device index %d", dev);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
    if (!ptr) return fail(FP_E_LAUNCH, "hipGetSymbolAddress(scratch) returned NULL");
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return FP_OK;
}

int paged_valid(const fp_paged_args* a) {
  if (!a) return fail(FP_E_INVALID_ARG, "paged arguments are NULL");
  if (a->dtype != FP_DTYPE_BF16 && a->dtype != FP_DTYPE_F16)
    return fail(FP_E_UNSUPPORTED, "paged: dtype %d unsupported (bf16 or fp16)", a->dtype);
  if (a->head_dim != 64 && a->head_dim != 128 && a->head_dim != 256)
    return fail(FP_E_UNSUPPORTED, "paged: head_dim %d unsupported (64, 128 or 256)", a->head_dim);
  if (a->num_q_heads < 1 || a->num_kv_heads < 1 || a->num_q_heads % a->num_kv_heads)
    return fail(FP_E_INVALID_ARG, "paged: num_q_heads (%d) must be a positive multiple of "
                "num_kv_heads (%d)", a->num_q_heads, a->num_kv_heads);
  if (a->num_tokens < 0 || a->num_blocks < 1 || a->batch < 1 || a->block_size < 1 ||
      a->table_width < 0 || a->table_stride < 0)
    return fail(FP_E_INVALID_ARG, "paged: sizes out of range");
  if (a->num_tokens == 0) return FP_OK;
  if (!a->q || !a->o || !a->key_cache || !a->value_cache || !a->cu_seqlens || !a->seqused ||
      (!a->block_table && a->table_width > 0))
    return fail(FP_E_INVALID_ARG, "paged: NULL pointer");
  if (!aligned16(a->q) || !aligned16(a->o) || !aligned16(a->key_cache) ||
      !aligned16(a->value_cache))
    return fail(FP_E_INVALID_ARG, "paged: q, o and the caches must be 16-byte aligned");
  const int64_t st[10] = {a->q_stride_tok,    a->q_stride_head,  a->o_stride_tok,
                          a->o_stride_head,   a->kc_stride_block, a->kc_stride_slot,
                          a->kc_stride_head,  a->vc_stride_block, a->vc_stride_slot,
                          a->vc_stride_head};
  for (int i = 0; i < 10; ++i)
    if (st[i] < 0 || st[i] % 8)
      return fail(FP_E_INVALID_ARG, "paged: strides must be non-negative multiples of 8 elements");
  // a lane's offset inside a page (16 slots) is formed in 32 bits
  if (a->kc_stride_slot >= (int64_t(1) << 24) || a->vc_stride_slot >= (int64_t(1) << 24))
    return fail(FP_E_UNSUPPORTED, "paged: slot strides of 2^24 elements or more");
  // key positions, and query rows x heads (the merge's grid), are 32-bit
  if (static_cast<int64_t>(a->table_width) * a->block_size >= (int64_t(1) << 30))
    return fail(FP_E_UNSUPPORTED, "paged: 2^30 or more tokens per sequence");
  if (a->num_tokens * a->num_q_heads >= (int64_t(1) << 30))
    return fail(FP_E_UNSUPPORTED, "paged: 2^30 or more query rows");
  return FP_OK;
}

// Row tiles and chunk slots of a paged call. Tiles: `rt` rows (query tokens x
// the query heads of a KV head) of one sequence; at most T G / rt + B of them,
// and no more than each token's rows on their own would make. rt is 16
// (k_paged, decode) or, from kManyRows rows per sequence on average and up to
// head_dim 128 (O^T of 256 dims and three parts of P do not fit a wave's 256
// registers), 128 (k_paged_rows). Chunk slots:
// about kTarget workgroups in all (several rounds of the card's ~768 resident
// ones, so that sequences of different lengths balance), no more than
// kPagedMaxChunks, and none shorter than kPagedMinChunk keys. (k_paged_rows:
// its 512 resident workgroups; every chunk costs a pass over fp32 partials of all
// its rows: one sequence of 8,192 tokens with 512 new ones, 32 q / 8 kv heads, 160
// us with 512, 176 with 1024, 205 with 2048.) The line between the kernels: 8
// sequences of 3,000 tokens, 32 q / 8 kv heads, with 4, 8, 16 and 64 queries each
// (16, 32, 64 and 256 rows): k_paged 147 (32 of 4,000), 49, 84 and 254 us,
// k_paged_rows 153, 46, 45 and 90. The average decides, since only the device sees
// the sequences: one of 4,000 tokens with 2,000 new ones beside 60 of 8,000 with one
// query each runs in k_paged_rows as a whole, one chunk per row, 690 - 725 us, where
// the two kinds as calls of their own take 245 - 250 and 395.
struct PagedSplit {
  bool many;  // k_paged_rows
  int64_t tiles;
  int nc;
  size_t bytes;
};
PagedSplit paged_split(const fp_paged_args* a) {
  constexpr int64_t kManyRows = 32;
  PagedSplit r;
  const int64_t G = a->num_q_heads / a->num_kv_heads, T = a->num_tokens;
  r.many = a->head_dim <= 128 && T * G >= kManyRows * a->batch;
  const int64_t kTarget = r.many ? 512 : 8192, rt = r.many ? 128 : 16;
  r.tiles = std::min<int64_t>(T * ((G + rt - 1) / rt), T * G / rt + a->batch);
  const int64_t longest = static_cast<int64_t>(a->table_width) * a->block_size;
  const int64_t wgs = std::max<int64_t>(1, r.tiles * a->num_kv_heads);
  int64_t nc = std::min<int64_t>(fp::kPagedMaxChunks, (kTarget + wgs - 1) / wgs);
  nc = std::min<int64_t>(nc, (longest + fp::kPagedMinChunk - 1) / fp::kPagedMinChunk);
  r.nc = static_cast<int>(std::max<int64_t>(1, nc));
  r.bytes = r.nc > 1 ? static_cast<size_t>(T * a->num_q_heads * r.nc) * (a->head_dim + 2) * 4 : 0;
  return r;
}

}  // namespace

extern "C" {

int fp_abi_version(void) { return 6; }

const char* fp_last_error(void) { return g_last_error.c_str(); }

int fp_workspace_layout(const fp_problem* p, fp_ws_layout* out) {
  if (!out) return fail(FP_E_INVALID_ARG, "layout output is NULL");
  return layout(p, out);
}

size_t fp_workspace_bytes(const fp_problem* p) {
  fp_ws_layout L;
  return layout(p, &L) == FP_OK ? L.total_bytes : 0;
}

int fp_plan(const fp_problem* p, void* ws, void* stream) {
  fp_ws_layout L;
  int rc = prepare(p, ws, &L);
  if (rc != FP_OK) return rc;
  return run_plan(p, L, ws, static_cast<hipStream_t>(stream));
}

int fp_pool_k(const fp_problem* p, void* ws, void* stream) {
  fp_ws_layout L;
  int rc = prepare(p, ws, &L);
  if (rc != FP_OK) return rc;
  return run_pool(p, L, ws, static_cast<hipStream_t>(stream));
}

int fp_search(const fp_problem* p, void* ws, float* dump_p, float* dump_m, void* stream) {
  fp_ws_layout L;
  int rc = prepare(p, ws, &L);
  if (rc != FP_OK) return rc;
  if ((dump_p == nullptr) != (dump_m == nullptr))
    return fail(FP_E_INVALID_ARG, "dump_p and dump_m must both be set or both be NULL");
  return run_search(p, L, ws, dump_p, dump_m, nullptr, nullptr, static_cast<hipStream_t>(stream));
}

int fp_select(const fp_problem* p, void* ws, const float* p_scores, const float* m_scores,
              void* stream) {
  fp_ws_layout L;
  int rc = prepare(p, ws, &L);
  if (rc != FP_OK) return rc;
  if (!p_scores || !m_scores) return fail(FP_E_INVALID_ARG, "p_scores and m_scores must be non-NULL");
  return run_search(p, L, ws, nullptr, nullptr, p_scores, m_scores,
                    static_cast<hipStream_t>(stream));
}

int fp_sparse_attn_fwd(const fp_problem* p, void* ws, void* stream) {
  fp_ws_layout L;
  int rc = prepare(p, ws, &L);
  if (rc != FP_OK) return rc;
  return run_attn(p, L, ws, static_cast<hipStream_t>(stream));
}

int fp_flashprefill(const fp_problem* p, void* ws, void* stream) {
  fp_ws_layout L;
  int rc = prepare(p, ws, &L);
  if (rc != FP_OK) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if ((rc = run_before_attention(p, L, ws, s)) != FP_OK) return rc;
  return run_attn(p, L, ws, s);
}

int fp_flashprefill_noalloc(const fp_problem* p, void* stream) {
  fp_ws_layout L;
  int rc = layout(p, &L);
  if (rc != FP_OK) return rc;
  if (L.total_bytes > FP_NOALLOC_SCRATCH_BYTES)
    return fail(FP_E_INVALID_ARG,
                "problem needs %zu bytes of workspace; the static scratch of "
                "fp_flashprefill_noalloc holds %zu (use fp_flashprefill with a workspace)",
                L.total_bytes, static_cast<size_t>(FP_NOALLOC_SCRATCH_BYTES));
  void* ws = nullptr;
  if ((rc = scratch_on_current_device(&ws)) != FP_OK) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if ((rc = run_before_attention(p, L, ws, s)) != FP_OK) return rc;
  return run_attn(p, L, ws, s);
}

int fp_rope_qk(const fp_rope_args* a, void* stream) {
  if (!a) return fail(FP_E_INVALID_ARG, "rope args are NULL");
  if (a->dtype != FP_DTYPE_BF16 && a->dtype != FP_DTYPE_F16)
    return fail(FP_E_UNSUPPORTED, "rope: dtype %d unsupported (bf16 or fp16)", a->dtype);
  if (a->head_dim != 64 && a->head_dim != 128 && a->head_dim != 256)
    return fail(FP_E_UNSUPPORTED, "rope: head_dim %d unsupported (64, 128 or 256)", a->head_dim);
  if (a->num_tokens < 0 || a->num_q_heads < 0 || a->num_kv_heads < 0 || a->num_positions < 1)
    return fail(FP_E_INVALID_ARG, "rope: negative sizes or an empty table");
  if (a->num_tokens == 0) return FP_OK;
  if ((a->num_q_heads > 0 && !a->q) || (a->num_kv_heads > 0 && !a->k) ||
      (!a->positions && !a->cu_seqlens) || !a->cos_table || !a->sin_table)
    return fail(FP_E_INVALID_ARG, "rope: NULL pointer");
  if (!a->positions && (a->batch < 1 || a->batch > fp::kRopeMaxBatch))
    return fail(FP_E_INVALID_ARG, "rope: batch %d outside [1, %d]", a->batch, fp::kRopeMaxBatch);
  const int64_t st[4] = {a->q_stride_tok, a->q_stride_head, a->k_stride_tok, a->k_stride_head};
  for (int i = 0; i < 4; ++i)
    if (st[i] < 0 || st[i] % 8)
      return fail(FP_E_INVALID_ARG, "rope: strides must be non-negative multiples of 8 elements");
  if ((a->q && !aligned16(a->q)) || (a->k && !aligned16(a->k)) || !aligned16(a->cos_table) ||
      !aligned16(a->sin_table))
    return fail(FP_E_INVALID_ARG, "rope: q / k / tables must be 16-byte aligned");
  fp::RopeArgs r;
  r.q = a->q;
  r.q_stride_tok = a->q_stride_tok;
  r.q_stride_head = a->q_stride_head;
  r.k = a->k;
  r.k_stride_tok = a->k_stride_tok;
  r.k_stride_head = a->k_stride_head;
  r.num_q_heads = a->num_q_heads;
  r.num_kv_heads = a->num_kv_heads;
  r.head_dim = a->head_dim;
  r.positions = a->positions;
  // (read only when asked for: callers with positions may pass the struct as it
  // was before these two fields)
  r.cu = a->positions ? nullptr : a->cu_seqlens;
  r.batch = a->positions ? 0 : a->batch;
  r.num_tokens = a->num_tokens;
  r.cos_tab = a->cos_table;
  r.sin_tab = a->sin_table;
  r.num_positions = a->num_positions;
  r.q_norm = a->q_norm;
  r.k_norm = a->k_norm;
  r.eps = a->eps;
  const hipError_t e = fp::launch_rope(r, a->dtype, static_cast<hipStream_t>(stream));
  return e == hipSuccess ? FP_OK : hip_fail(e, "rope launch");
}

size_t fp_paged_workspace_bytes(const fp_paged_args* a) {
  return paged_valid(a) == FP_OK ? paged_split(a).bytes : 0;
}

int fp_paged_attention(const fp_paged_args* a, void* ws, void* stream) {
  const int rc = paged_valid(a);
  if (rc != FP_OK) return rc;
  if (a->num_tokens == 0) return FP_OK;
  const PagedSplit sp = paged_split(a);
  if (sp.bytes > 0 && !ws) return fail(FP_E_INVALID_ARG, "paged: workspace is NULL");
  if (!aligned16(ws)) return fail(FP_E_INVALID_ARG, "paged: workspace must be 16-byte aligned");
  fp::PagedArgs r;
  r.q = a->q;
  r.o = a->o;
  r.kc = a->key_cache;
  r.vc = a->value_cache;
  r.qst = a->q_stride_tok;
  r.qhs = a->q_stride_head;
  r.ost = a->o_stride_tok;
  r.ohs = a->o_stride_head;
  r.kcb = a->kc_stride_block;
  r.kcs = a->kc_stride_slot;
  r.kch = a->kc_stride_head;
  r.vcb = a->vc_stride_block;
  r.vcs = a->vc_stride_slot;
  r.vch = a->vc_stride_head;
  r.cu = a->cu_seqlens;
  r.used = a->seqused;
  r.table = a->block_table;
  r.cu64 = a->cu_is64;
  r.used64 = a->used_is64;
  r.table64 = a->table_is64;
  r.table_stride = a->table_stride;
  r.T = a->num_tokens;
  r.nblocks = a->num_blocks;
  r.B = a->batch;
  r.width = a->table_width;
  r.bs = a->block_size;
  r.bs_shift = -1;
  for (int sh = 0; sh < 31; ++sh)
    if ((1 << sh) == a->block_size) r.bs_shift = sh;
  r.Hq = a->num_q_heads;
  r.Hkv = a->num_kv_heads;
  r.G = a->num_q_heads / a->num_kv_heads;
  r.scale_log2 = a->softmax_scale * static_cast<float>(1.4426950408889634);
  r.nc = sp.nc;
  r.part = static_cast<float*>(ws);
  r.ml = sp.nc > 1 ? static_cast<float*>(ws) + a->num_tokens * a->num_q_heads * sp.nc * a->head_dim
                   : nullptr;
  const auto launch = sp.many ? fp::launch_paged_rows : fp::launch_paged;
  const hipError_t e = launch(r, a->dtype, a->head_dim, sp.tiles, static_cast<hipStream_t>(stream));
  return e == hipSuccess ? FP_OK : hip_fail(e, "paged attention launch");
}

int fp_kv_cache_write(const fp_kv_cache_args* a, void* stream) {
  if (!a) return fail(FP_E_INVALID_ARG, "kv-cache arguments are NULL");
  if (a->dtype != FP_DTYPE_BF16 && a->dtype != FP_DTYPE_F16)
    return fail(FP_E_UNSUPPORTED, "kv-cache dtype %d unsupported (bf16 or fp16 only)", a->dtype);
  if (a->num_tokens < 0 || a->num_blocks < 0 || a->block_size < 1 || a->num_kv_heads < 1 ||
      a->head_dim < 8 || a->head_dim % 8)
    return fail(FP_E_INVALID_ARG, "kv-cache sizes out of range (head_dim must be a multiple of 8)");
  if (a->num_tokens > 0x7fffffff) return fail(FP_E_INVALID_ARG, "too many tokens");
  if (a->num_tokens == 0) return FP_OK;
  if (!a->key || !a->value || !a->key_cache || !a->value_cache || !a->slot_mapping)
    return fail(FP_E_INVALID_ARG, "kv-cache pointers must be non-NULL");
  if (!aligned16(a->key) || !aligned16(a->value) || !aligned16(a->key_cache) ||
      !aligned16(a->value_cache))
    return fail(FP_E_INVALID_ARG, "key/value and caches must be 16-byte aligned");
  const int64_t strides[10] = {a->k_stride_tok, a->k_stride_head, a->v_stride_tok, a->v_stride_head,
                               a->kc_stride_block, a->kc_stride_slot, a->kc_stride_head,
                               a->vc_stride_block, a->vc_stride_slot, a->vc_stride_head};
  for (int i = 0; i < 10; ++i)
    if (strides[i] < 0 || strides[i] % 8)
      return fail(FP_E_INVALID_ARG, "kv-cache strides must be non-negative multiples of 8 elements");
  fp::KvCacheArgs k;
  k.key = a->key;
  k.value = a->value;
  k.k_stride_tok = a->k_stride_tok;
  k.k_stride_head = a->k_stride_head;
  k.v_stride_tok = a->v_stride_tok;
  k.v_stride_head = a->v_stride_head;
  k.key_cache = a->key_cache;
  k.value_cache = a->value_cache;
  k.kc_stride_block = a->kc_stride_block;
  k.kc_stride_slot = a->kc_stride_slot;
  k.kc_stride_head = a->kc_stride_head;
  k.vc_stride_block = a->vc_stride_block;
  k.vc_stride_slot = a->vc_stride_slot;
  k.vc_stride_head = a->vc_stride_head;
  k.slot_mapping = a->slot_mapping;
  k.num_tokens = a->num_tokens;
  k.num_slots = a->num_blocks * a->block_size;
  k.block_size = a->block_size;
  k.num_kv_heads = a->num_kv_heads;
  k.elem_bytes = 2;
  k.row_bytes = a->head_dim * 2;
  const hipError_t e = fp::launch_kv_cache_write(k, static_cast<hipStream_t>(stream));
  return e == hipSuccess ? FP_OK : hip_fail(e, "kv-cache write launch");
}

int fp_read_status(const fp_problem* p, void* ws, void* stream, uint32_t* status) {
  fp_ws_layout L;
  int rc = prepare(p, ws, &L);
  if (rc != FP_OK) return rc;
  if (!status) return fail(FP_E_INVALID_ARG, "status output is NULL");
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipError_t e = hipMemcpyAsync(status, static_cast<char*>(ws) + L.status_off, sizeof(uint32_t),
                                hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  return e == hipSuccess ? FP_OK : hip_fail(e, "status read");
}

}  // extern "C"
