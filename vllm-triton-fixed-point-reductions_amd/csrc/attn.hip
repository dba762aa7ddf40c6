// C-ABI entry points of the paged attention (kernels: attn_impl.h,
// instantiated per input type in attn_{bf16,f16,f32}.hip).
#include <algorithm>
#include <mutex>

#include "attn_impl.h"

using namespace fxpr;
using namespace fxpr::attn;

namespace {

constexpr int kMaxSplits = 64;      // automatic policy's largest split count
constexpr int64_t kMaxGridZ = 65535;  // splits are the launch grid's z dimension
// Split launches keep per-chunk partials; above this many bytes of them a
// launch runs unsplit instead (split counts never change the bits).
constexpr int64_t kSplitWsMax = int64_t(1) << 30;

inline int64_t align256(int64_t x) { return (x + 255) & ~int64_t(255); }

inline int acc_bytes(int int_bits) { return int_bits == 64 ? 8 : 4; }

// Chunks per row that a block-table row of max_blocks pages can hold.
inline int64_t chunk_slots(int max_blocks, int page_size) {
  return cdiv(cdiv(int64_t(max_blocks) * page_size, TILE), CT);
}

// Split-launch workspace: per (token, head) the chunk range, and per
// (token, head, chunk) the row maximum, the integer denominator and the
// integer weighted V row. Unsplit launches need none.
struct WsLayout {
  int64_t crange = -1, pmax = -1, den = -1, wv = -1, total = 0;
};

// (ws_rows: the query tokens that hold records, AttnArgs' W)
WsLayout ws_layout(int64_t ws_rows, int num_heads, int head_dim, int int_bits, bool split, int64_t slots) {
  WsLayout w;
  if (!split) return w;
  const int64_t rows = ws_rows * num_heads;
  w.crange = 0;
  w.total = align256(rows * 8);
  w.pmax = w.total;
  w.total += align256(rows * slots * 4);
  w.den = w.total;
  w.total += align256(rows * slots * acc_bytes(int_bits));
  w.wv = w.total;
  w.total += align256(rows * slots * head_dim * acc_bytes(int_bits));
  return w;
}

}  // namespace

// Split policy (this build's own; the reference's _pick_num_splits,
// attention.py:664-689, is the model for its shape). An explicit request wins
// (each workgroup's key chunks dealt evenly over the splits, as the
// reference's _split_tile_range deals tiles), up to the number of 512-key
// chunks a block-table row holds: splits past that would hold no keys (the
// reference's would be empty), so the launch runs that many. Automatic (0):
// no split for short contexts (<= 32 key tiles of 64) or when the
// (request, kv head, 16-row query tile) workgroups already number more than
// 8 x 256; otherwise one chunk per split (up to 64 splits), so every
// workgroup carries about the same work whatever its request's length
// (requests shorter than the longest get empty splits). Split counts never
// change bits.
namespace {
constexpr int kSplitChunks = 1;

struct SplitPlan {
  int splits, chunks_per_split;
};

SplitPlan plan_splits(int num_requests, int num_kv_heads, int group, int max_query_len, int max_blocks,
                      int page_size, int requested) {
  const int64_t tiles = cdiv(int64_t(max_blocks > 0 ? max_blocks : 1) * page_size, TILE);
  if (requested >= 1) {
    const int64_t cap = std::min<int64_t>(std::max<int64_t>(cdiv(tiles, CT), 1), kMaxGridZ);
    return {int(std::min<int64_t>(requested, cap)), 0};
  }
  if (tiles <= 32) return {1, 0};
  const int64_t qtiles = cdiv(int64_t(max_query_len > 1 ? max_query_len : 1) * group, QROWS);
  const int64_t base = int64_t(num_requests > 1 ? num_requests : 1) * num_kv_heads * qtiles;
  if (base > 8 * 256) return {1, 0};
  const int64_t chunks = cdiv(tiles, CT);
  int64_t s = cdiv(chunks, kSplitChunks);
  if (s > kMaxSplits) s = kMaxSplits;
  if (s <= 1) return {1, 0};
  return {int(s), int(cdiv(chunks, s))};
}

// The plan a launch runs: plan_splits, unsplit when the partials would exceed
// kSplitWsMax.
SplitPlan launch_plan(int num_requests, int64_t num_tokens, int num_heads, int num_kv_heads, int head_dim,
                      int int_bits, int max_query_len, int max_blocks, int page_size, int requested) {
  SplitPlan sp = plan_splits(num_requests, num_kv_heads, num_heads / num_kv_heads, max_query_len, max_blocks,
                             page_size, requested);
  if (sp.splits > 1 &&
      ws_layout(num_tokens, num_heads, head_dim, int_bits, true, chunk_slots(max_blocks, page_size)).total >
          kSplitWsMax)
    sp = {1, 0};
  return sp;
}

// Launches that may hold requests of kPrefillRows rows or more, where the DMA
// kernels can take them (Route::kLongDma): the two kinds of requests are split
// apart from each other, over tables of more than 32 key tiles. The host knows
// the table's width and not the contexts, so every number of splits is paid for
// by batches whose contexts are short: workgroups that find no keys (600 of them
// start and exit in a microsecond), records and a combine launch.
//   * Prefill workgroups (64 rows each): about tokens x heads / 64 of them.
//     Below kFullWgs (two per CU) their keys are split until there are about
//     kLongWgs; a chunk is the least a split can hold.
//   * Short requests, one workgroup per request and kv head (`rk` of them): up to
//     kFullWgs split into equal runs of chunks, about kShortWgs in all. (Beyond
//     it, 77 decode steps of up to 3000 keys beside 2 x 166 tokens, 16 heads of 64:
//     133 us unsplit, 156 split by chunk, 202 in runs of two.)
//   * Tables wider than kWideKeys say little about the contexts: the short
//     requests' own chunks are dealt evenly to splits that make up kFullWgs
//     workgroups (twice that for few), the prefill ones' to half as many, and a batch
//     of long requests on average is taken to hold no short ones. (Split 64 ways,
//     61 decode steps of up to 9300 keys beside 4 prompts of 22 tokens, 24/8 heads
//     of 64, took 730 us at a table of 131072 keys; 192 now, 181 unsplit.)
//   * A window of up to kSmallWindow keys leaves a few chunks per row whatever the
//     table: split where the launch leaves the GPU nearly empty.
//   * No short request is possible where the tokens are just requests x the
//     longest one's (4 prompts of 2048 tokens, table of 131072 keys: 366 us with
//     the short requests' split, 340 without).
// Against the plan before requests were split apart (us before / now, geometric
// mean): drawn batches with prompts, tables as wide as their longest context (up
// to 12288 keys) 1.40x, 7 of 272 more than 3 % slower, the worst 1.24x; tables of
// 8192 keys 1.53x, 8 of 78, 1.6x (83 decode steps under 300 keys beside 3 x 79
// tokens, 36 -> 58); 32768 1.9x, 7 of 101, 1.35x; 131072 2.1x, 1 of 74, 1.06x.
// Explicit requests split both that many times. Records need a workspace: per
// token when the prefill rows are split, else only for the short requests'
// tokens. Above kLongWsMax the launch runs unsplit; above kSplitWsMax where the
// split is explicit, or where there are so few prefill workgroups (kFewWgs) that
// they lose to the 16-row kernels' split, which holds as many records (one
// request, 32/8 heads of 128, over 30000 cached keys: 128 tokens, table of
// 131072 keys 885 us unsplit, 462 split by 16 rows, 197 split here; 256 at 65536
// 887 and 921. The wider cap at 256 and 512 tokens too would take 512 at 32768
// from 897 to 697, but 512 without cached keys from 22 to 36).
constexpr int64_t kFullWgs = 512, kLongWgs = 2048, kShortWgs = 8192, kFewWgs = 128;
constexpr int64_t kWideKeys = 16384, kSmallWindow = 2048, kWindowWgs = 140, kWindowShort = 128;
constexpr int64_t kLongTokens = 200;  // tokens per request besides the longest that mean "long on average"
constexpr int64_t kLongWsMax = int64_t(1) << 29;

struct LongLayout {
  LongPlan plan;
  WsLayout ws;
};

LongLayout long_plan(int num_requests, int64_t num_tokens, int num_heads, int num_kv_heads, int head_dim, int int_bits,
                     int max_query_len, int max_blocks, int page_size, int64_t window, int requested) {
  LongLayout l;
  const int group = num_heads / num_kv_heads;
  const int64_t slots = chunk_slots(max_blocks, page_size);
  const int64_t keys = int64_t(max_blocks > 0 ? max_blocks : 1) * page_size;
  const int64_t wgs = std::max<int64_t>(cdiv(num_tokens * num_heads, PQROWS), 1);
  int64_t ps = 1, ds = 1, per = 0;  // per: chunks per split of the short requests (0: dealt evenly)
  if (requested >= 1) {
    ps = ds = std::min<int64_t>({int64_t(requested), std::max<int64_t>(slots, 1), kMaxGridZ});
  } else if (cdiv(keys, TILE) > 32) {
    const int64_t rk = int64_t(num_requests) * num_kv_heads, others = num_tokens - max_query_len;
    const bool wide = keys > kWideKeys;
    bool shorts = num_tokens != int64_t(num_requests) * max_query_len;
    if (window > 0) {
      const int64_t chunks = std::min(slots, cdiv(window, TILE * CT) + 1);  // those a row's window can touch
      if (wgs <= kWindowWgs) ps = chunks;
      if (rk < kWindowShort) ds = chunks;
    } else {
      if (wgs < kFullWgs) ps = std::min(cdiv(wide ? kLongWgs / 2 : kLongWgs, wgs), slots);
      if (wide) {
        shorts = shorts && others < kLongTokens * (num_requests - 1);
        if (rk < kFullWgs) ds = std::min<int64_t>({cdiv(rk <= 64 ? 2 * kFullWgs : kFullWgs, rk), slots, kMaxSplits});
      } else if (rk <= kFullWgs) {
        per = std::max<int64_t>(rk * slots / kShortWgs, 1);
        ds = cdiv(slots, per);
      }
    }
    if (!shorts) ds = 1;
  }
  auto layout = [&](int64_t rows) { return ws_layout(rows, num_heads, head_dim, int_bits, true, slots); };
  const int64_t most = requested >= 1 ? kSplitWsMax : kLongWsMax;
  const bool few = wgs < kFewWgs && launch_plan(num_requests, num_tokens, num_heads, num_kv_heads, head_dim, int_bits,
                                                max_query_len, max_blocks, page_size, 0)
                                            .splits > 1;
  if (ps > 1) {
    l.ws = layout(num_tokens);
    if (l.ws.total > (few ? kSplitWsMax : most)) {
      ps = 1;
      if (requested >= 1) ds = 1;
    }
  }
  if (ps <= 1) {
    l.ws = WsLayout{};
    if (ds > 1) {
      // a short request holds fewer than kPrefillRows rows
      const int64_t cap = std::min<int64_t>(max_query_len, std::max<int64_t>((kPrefillRows - 1) / group, 1));
      l.plan.tok_cap = int(cap);
      l.ws = layout(int64_t(num_requests) * cap);
      if (l.ws.total > most) {
        ds = 1;
        l.plan.tok_cap = 0;
        l.ws = WsLayout{};
      }
    }
  }
  l.plan.pq_splits = int(ps);
  l.plan.splits = int(ds);
  l.plan.chunks_per_split = ds > 1 ? int(per) : 0;
  return l;
}

// rows (tokens x group) and 16-row chunk units up to which a batch counts as few
constexpr int64_t kFewRows = 256, kFewChunks = 3000;

// What a launch runs: its kernels, its splits and the records they need.
struct LaunchPlan {
  LongPlan lp;        // (splits: kLongDma only)
  SplitPlan sp{1, 0};  // the other routes' splits
  WsLayout ws;
};

LaunchPlan attention_plan(int io_dtype, int num_requests, int64_t num_tokens, int num_heads, int num_kv_heads,
                          int head_dim, int page_size, int max_query_len, int max_blocks, int64_t stride_k_slot,
                          int64_t stride_v_slot, int is_causal, int window_size, int int_bits, int requested) {
  LaunchPlan p;
  const bool dma = dma_takes(io_dtype, head_dim, page_size, stride_k_slot, stride_v_slot);
  const int group = num_heads / num_kv_heads;
  const int64_t max_rows = int64_t(max_query_len > 1 ? max_query_len : 1) * group;
  // 64-row workgroups serve 16-bit inputs with 16- / 32-bit sums, and only
  // requests of kPrefillRows rows or more
  const bool narrow_sums = io_dtype != FXPR_DTYPE_F32 && int_bits != 64;
  const bool wide = narrow_sums && head_dim <= 128 && max_rows >= kPrefillRows;
  // a window that leaves few keys per row (and bounds them on both sides)
  const int64_t keys = int64_t(max_blocks) * page_size;
  const int64_t window =
      is_causal && window_size > 0 && window_size <= kSmallWindow && window_size < keys ? window_size : 0;
  p.sp = launch_plan(num_requests, num_tokens, num_heads, num_kv_heads, head_dim, int_bits, max_query_len, max_blocks,
                     page_size, requested);
  // A few tokens in all, over tables that are not wide: one split launch of
  // 16-row workgroups spreads them further than 64-row ones, and takes two
  // launches instead of three. Both sides, us: 28 tokens in 3 requests over up to
  // 2500 keys (32/8 heads of 128) 23 against 42 apart; 45 in 14 beside 4096 cached
  // ones under a window of 1024 26 and 43; 77 in 3 over 6000 59 and 38 (308 rows:
  // apart). Over 348 drawn batches of up to 500 rows the rule is within 2 % of the
  // better of the two on average, always apart 7 %.
  const int64_t rows = num_tokens * group;
  const int64_t chunks = cdiv(window > 0 ? std::min<int64_t>(keys, window + max_query_len) : keys, TILE * CT);
  const bool few_rows = requested == 0 && p.sp.splits > 1 && keys <= kWideKeys && rows <= kFewRows &&
                        num_kv_heads * (cdiv(rows, QROWS) + num_requests) * chunks <= kFewChunks;
  if (wide && dma && !few_rows) {
    const LongLayout l = long_plan(num_requests, num_tokens, num_heads, num_kv_heads, head_dim, int_bits, max_query_len,
                                   max_blocks, page_size, window, requested);
    p.sp = SplitPlan{1, 0};
    p.lp = l.plan;
    p.lp.route = Route::kLongDma;
    p.ws = l.ws;
    return p;
  }
  p.ws = ws_layout(num_tokens, num_heads, head_dim, int_bits, p.sp.splits > 1, chunk_slots(max_blocks, page_size));
  // Just short of that, three 16-row tiles a request (33 to 47 rows), the DMA
  // kernel is the faster one at head_dim 128 (us, register loads / DMA: 1 x 10
  // tokens of group 4 over 1000 keys 30 / 27, 64 x 10 over 2000 296 / 262, 90
  // decode steps up to 4000 keys beside 2 x 10 tokens 223 / 213; 64 x 10 over
  // 500 69 / 76), register loads at 64 (4 x 40 tokens of group 1 over 500 keys
  // 13.3 / 15.9, 64 x 40 over 1000 143 / 166, 90 decode steps up to 2000 beside
  // 2 x 40 123 / 135; 64 x 40 over 2000 318 / 296).
  const bool three_tiles = max_rows > 2 * QROWS && max_rows < kPrefillRows;
  const bool by_registers = narrow_sums && head_dim == 64 && three_tiles && p.sp.splits <= 1;
  if (wide && p.sp.splits <= 1)
    p.lp.route = Route::kLong;
  else
    p.lp.route = dma && !by_registers ? Route::kRows16Dma : Route::kRows16;
  return p;
}

bool plan_args_ok(int num_requests, int64_t num_tokens, int num_heads, int num_kv_heads, int head_dim, int page_size,
                  int max_blocks, int num_kv_splits) {
  return num_requests > 0 && num_tokens > 0 && num_heads > 0 && num_kv_heads > 0 && head_dim > 0 && max_blocks > 0 &&
         page_size > 0 && num_heads % num_kv_heads == 0 && num_kv_splits >= 0;
}
}  // namespace

extern "C" int fxpr_attention_splits(int num_requests, int num_kv_heads, int group, int max_query_len,
                                     int max_blocks_per_seq, int page_size, int requested) {
  return plan_splits(num_requests, num_kv_heads, group, max_query_len, max_blocks_per_seq, page_size,
                     requested)
      .splits;
}

extern "C" int64_t fxpr_attention_workspace_bytes(int num_requests, int64_t num_tokens, int num_heads,
                                                  int num_kv_heads, int head_dim, int int_bits,
                                                  int num_kv_splits, int max_query_len,
                                                  int max_blocks_per_seq, int page_size) {
  // whatever the inputs' type, the cache's strides and the window: with the DMA
  // kernels or without, and the widest and the narrowest window
  auto need = [&](int io_dtype, int window) {
    return fxpr_attention_plan(io_dtype, num_requests, num_tokens, num_heads, num_kv_heads, head_dim, page_size,
                               max_query_len, max_blocks_per_seq, head_dim, head_dim, 1, window, int_bits,
                               num_kv_splits, nullptr);
  };
  return std::max({need(FXPR_DTYPE_BF16, 0), need(FXPR_DTYPE_BF16, 1), need(FXPR_DTYPE_F32, 0)});
}

extern "C" int64_t fxpr_attention_plan(int io_dtype, int num_requests, int64_t num_tokens, int num_heads,
                                       int num_kv_heads, int head_dim, int page_size, int max_query_len,
                                       int max_blocks_per_seq, int64_t stride_k_slot, int64_t stride_v_slot,
                                       int is_causal, int window_size, int int_bits, int num_kv_splits, int32_t* plan) {
  if (plan) std::fill(plan, plan + 4, 0);
  if (!plan_args_ok(num_requests, num_tokens, num_heads, num_kv_heads, head_dim, page_size, max_blocks_per_seq,
                    num_kv_splits))
    return 0;
  const LaunchPlan p = attention_plan(io_dtype, num_requests, num_tokens, num_heads, num_kv_heads, head_dim, page_size,
                                      max_query_len, max_blocks_per_seq, stride_k_slot, stride_v_slot, is_causal,
                                      window_size, int_bits, num_kv_splits);
  if (plan) {
    const bool apart = p.lp.route == Route::kLongDma;
    plan[0] = int(p.lp.route);
    plan[1] = apart ? p.lp.pq_splits : p.sp.splits;
    plan[2] = apart ? p.lp.splits : p.sp.splits;
    plan[3] = p.lp.tok_cap;
  }
  return p.ws.total;
}

// Pairs of neighbouring fp32 values, from -inf to inf, whose softcap descends.
namespace {
__global__ __launch_bounds__(256) void softcap_descents_kernel(float softcap, unsigned long long* count) {
  constexpr uint32_t kInf = 0x7f800000u;
  auto value = [](uint64_t i) {  // the i-th from -inf: -inf .. -0 at 0 .. kInf, 0 .. inf after it
    return __uint_as_float(i <= kInf ? 0x80000000u | (kInf - uint32_t(i)) : uint32_t(i - kInf - 1));
  };
  unsigned long long n = 0;
  const uint64_t step = uint64_t(gridDim.x) * 256;
  for (uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x; i < 2 * uint64_t(kInf) + 1; i += step)
    n += !(softcapped(value(i), softcap) <= softcapped(value(i + 1), softcap));
  if (n) atomicAdd(count, n);
}
}  // namespace

extern "C" int fxpr_debug_softcap_descents(float softcap_log2, unsigned long long* count, void* stream) {
  if (!count || !(softcap_log2 > 0.0f)) return FXPR_E_ARG;
  softcap_descents_kernel<<<dim3(4096), 256, 0, as_stream(stream)>>>(softcap_log2, count);
  return launch_status();
}

extern "C" int fxpr_unified_attention(
    const void* q, const void* k_cache, const void* v_cache, void* o, int io_dtype,
    const int32_t* query_start_loc, const int32_t* seq_lens, const int32_t* block_table,
    const float* alibi_slopes, int num_requests, int64_t num_tokens, int num_heads,
    int num_kv_heads, int head_dim, int page_size, int max_query_len, int max_blocks_per_seq,
    int64_t num_blocks, int64_t stride_q_token, int64_t stride_q_head, int64_t stride_k_block,
    int64_t stride_k_slot, int64_t stride_k_head, int64_t stride_v_block, int64_t stride_v_slot,
    int64_t stride_v_head, int64_t stride_o_token, int64_t stride_o_head, int64_t stride_bt_row,
    int is_causal, float softmax_scale_log2, float softcap_log2, int window_size, int int_bits,
    int frac_bits, int num_kv_splits, void* workspace, int64_t workspace_bytes, void* stream) {
  if (!valid_int_bits(int_bits) || frac_bits < 0 || frac_bits > 63) return FXPR_E_BITS;
  if (num_requests < 0 || num_tokens < 0 || num_heads <= 0 || num_kv_heads <= 0 || head_dim <= 0 ||
      page_size <= 0 || num_kv_splits < 0 || num_heads % num_kv_heads != 0)
    return FXPR_E_SHAPE;
  if (num_requests == 0 || num_tokens == 0) return FXPR_OK;
  if (max_blocks_per_seq <= 0 || num_blocks <= 0) return FXPR_E_SHAPE;
  if (!q || !k_cache || !v_cache || !o || !query_start_loc || !seq_lens || !block_table) return FXPR_E_ARG;
  if (io_dtype != FXPR_DTYPE_BF16 && io_dtype != FXPR_DTYPE_F16 && io_dtype != FXPR_DTYPE_F32)
    return FXPR_E_DTYPE;
  const int ch = io_dtype == FXPR_DTYPE_F32 ? 4 : 8;
  // vector loads of q / k / v rows need 16-byte alignment
  if (head_dim % ch != 0 || head_dim > 256 || (io_dtype == FXPR_DTYPE_F32 && head_dim > 128))
    return FXPR_E_SHAPE;
  if (stride_q_token % ch || stride_q_head % ch || stride_k_block % ch || stride_k_slot % ch ||
      stride_k_head % ch || stride_v_block % ch || stride_v_slot % ch || stride_v_head % ch ||
      !aligned(q, 16) || !aligned(k_cache, 16) || !aligned(v_cache, 16))
    return FXPR_E_ARG;
  // the kernels form cache offsets as 32 x 32 -> 64-bit products
  for (int64_t sv : {stride_k_block, stride_k_slot, stride_k_head, stride_v_block, stride_v_slot, stride_v_head})
    if (sv < 0 || sv > int64_t(0xffffffff)) return FXPR_E_ARG;
  const int64_t slots = chunk_slots(max_blocks_per_seq, page_size);
  if (slots > 0x7fffffff) return FXPR_E_SHAPE;
  LaunchPlan plan = attention_plan(io_dtype, num_requests, num_tokens, num_heads, num_kv_heads, head_dim, page_size,
                                   max_query_len, max_blocks_per_seq, stride_k_slot, stride_v_slot, is_causal,
                                   window_size, int_bits, num_kv_splits);
  if (plan.ws.total > 0 && (!workspace || workspace_bytes < plan.ws.total)) return FXPR_E_WORKSPACE;

  AttnArgs a{};
  a.q = q;
  a.k = k_cache;
  a.v = v_cache;
  a.o = o;
  a.qsl = query_start_loc;
  a.seq_lens = seq_lens;
  a.bt = block_table;
  a.alibi = alibi_slopes;
  char* base = static_cast<char*>(workspace);
  if (plan.ws.total > 0) {
    a.crange = reinterpret_cast<int*>(base + plan.ws.crange);
    a.pmax = reinterpret_cast<float*>(base + plan.ws.pmax);
    a.den_ws = base + plan.ws.den;
    a.wv_ws = base + plan.ws.wv;
  }
  a.chunk_slots = int(slots);
  a.sq_t = stride_q_token;
  a.sq_h = stride_q_head;
  a.sk_b = stride_k_block;
  a.sk_s = stride_k_slot;
  a.sk_h = stride_k_head;
  a.sv_b = stride_v_block;
  a.sv_s = stride_v_slot;
  a.sv_h = stride_v_head;
  a.so_t = stride_o_token;
  a.so_h = stride_o_head;
  a.sbt = stride_bt_row;
  a.num_heads = num_heads;
  a.num_kv_heads = num_kv_heads;
  a.group = num_heads / num_kv_heads;
  a.head_dim = head_dim;
  a.page_size = page_size;
  a.num_splits = plan.sp.splits;
  a.chunks_per_split = plan.sp.chunks_per_split;
  a.window = window_size > 0 ? window_size : 0;
  a.causal = is_causal ? 1 : 0;
  a.max_blocks = max_blocks_per_seq;
  a.num_requests = num_requests;
  a.num_blocks = num_blocks;
  a.num_tokens = num_tokens;
  a.lmax = int64_t(max_blocks_per_seq) * page_size;
  const int esz = io_dtype == FXPR_DTYPE_F32 ? 4 : 2;
  a.o_vec = stride_o_token % kCombineVec == 0 && stride_o_head % kCombineVec == 0 && aligned(o, kCombineVec * esz);
  a.ps_shift = (page_size & (page_size - 1)) == 0 ? __builtin_ctz(unsigned(page_size)) : -1;
  a.scale_log2 = softmax_scale_log2;
  a.softcap_log2 = softcap_log2;
  a.fxp_scale = pow2f(frac_bits);
  a.fxp_inv = pow2f(-frac_bits);
  const int max_qtiles = int(cdiv(int64_t(max_query_len > 1 ? max_query_len : 1) * a.group, QROWS));
  hipStream_t st = as_stream(stream);
  switch (io_dtype) {
    case FXPR_DTYPE_BF16: return run_attn_bf16(a, plan.lp, int_bits, num_requests, max_qtiles, num_tokens, st);
    case FXPR_DTYPE_F16: return run_attn_f16(a, plan.lp, int_bits, num_requests, max_qtiles, num_tokens, st);
    default: return run_attn_f32(a, plan.lp, int_bits, num_requests, max_qtiles, num_tokens, st);
  }
}

// ---------------------------------------------------------------------------
// The same launch without a caller workspace: split partials go to `scratch`,
// a file-scope device array of kStaticScratchBytes that each GPU the library
// runs on holds until the process ends. Its device address is looked up once
// per device (hipGetSymbolAddress with that device current) and kept in
// scratch_ptr; host code never passes the array's own name to a kernel. The
// partials need no zeroing (every slot a combine reads was written by the
// same launch). Calls that overlap on one GPU share the array and race.

namespace {

constexpr int64_t kStaticScratchBytes = FXPR_STATIC_SCRATCH_BYTES;
constexpr int kMaxDevices = 64;

__device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

std::mutex scratch_mu;
void* scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the stream's device (the current device
// for the null stream).
int static_scratch(hipStream_t st, void** out) {
  int cur = 0;
  hipError_t e = hipGetDevice(&cur);
  if (e != hipSuccess) return static_cast<int>(e);
  int dev = cur;
  if (st != nullptr) {
    e = hipStreamGetDevice(st, &dev);
    if (e != hipSuccess) return static_cast<int>(e);
  }
  if (dev < 0 || dev >= kMaxDevices) return FXPR_E_ARG;
  std::lock_guard<std::mutex> lock(scratch_mu);
  if (scratch_ptr[dev] == nullptr) {
    // the look-up (and a device switch) stays out of graph capture
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if ((e = hipStreamIsCapturing(st, &cs)) != hipSuccess) return static_cast<int>(e);
    if (cs != hipStreamCaptureStatusNone) return FXPR_E_CAPTURE;
    if (dev != cur && (e = hipSetDevice(dev)) != hipSuccess) return static_cast<int>(e);
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (dev != cur) {
      const hipError_t back = hipSetDevice(cur);
      if (e == hipSuccess) e = back;
    }
    if (e != hipSuccess) return static_cast<int>(e);
    scratch_ptr[dev] = p;
  }
  *out = scratch_ptr[dev];
  return FXPR_OK;
}

}  // namespace

extern "C" int fxpr_unified_attention_noalloc(
    const void* q, const void* k_cache, const void* v_cache, void* o, int io_dtype,
    const int32_t* query_start_loc, const int32_t* seq_lens, const int32_t* block_table,
    const float* alibi_slopes, int num_requests, int64_t num_tokens, int num_heads,
    int num_kv_heads, int head_dim, int page_size, int max_query_len, int max_blocks_per_seq,
    int64_t num_blocks, int64_t stride_q_token, int64_t stride_q_head, int64_t stride_k_block,
    int64_t stride_k_slot, int64_t stride_k_head, int64_t stride_v_block, int64_t stride_v_slot,
    int64_t stride_v_head, int64_t stride_o_token, int64_t stride_o_head, int64_t stride_bt_row,
    int is_causal, float softmax_scale_log2, float softcap_log2, int window_size, int int_bits,
    int frac_bits, int num_kv_splits, void* stream) {
  auto ws_need = [&](int splits) {
    return fxpr_attention_plan(io_dtype, num_requests, num_tokens, num_heads, num_kv_heads, head_dim, page_size,
                               max_query_len, max_blocks_per_seq, stride_k_slot, stride_v_slot, is_causal, window_size,
                               int_bits, splits, nullptr);
  };
  int64_t need = ws_need(num_kv_splits);
  if (need > 0 && num_kv_splits == 0) {
    // an automatic split of long requests apart from short ones needs records
    // where the batch's plain split count (often none) needs fewer or none:
    // this entry point runs the plain count (same bits), so that such a batch
    // still needs no scratch array, nor its look-up outside graph capture
    const int plain = launch_plan(num_requests, num_tokens, num_heads, num_kv_heads, head_dim, int_bits, max_query_len,
                                  max_blocks_per_seq, page_size, 0)
                          .splits;
    if (need > ws_need(plain)) {
      num_kv_splits = plain;
      need = ws_need(plain);
    }
  }
  if (need > kStaticScratchBytes) return FXPR_E_WORKSPACE;
  void* ws = nullptr;
  if (need > 0) {
    const int rc = static_scratch(as_stream(stream), &ws);
    if (rc != FXPR_OK) return rc;
  }
  return fxpr_unified_attention(q, k_cache, v_cache, o, io_dtype, query_start_loc, seq_lens, block_table,
                                alibi_slopes, num_requests, num_tokens, num_heads, num_kv_heads, head_dim,
                                page_size, max_query_len, max_blocks_per_seq, num_blocks, stride_q_token,
                                stride_q_head, stride_k_block, stride_k_slot, stride_k_head, stride_v_block,
                                stride_v_slot, stride_v_head, stride_o_token, stride_o_head, stride_bt_row,
                                is_causal, softmax_scale_log2, softcap_log2, window_size, int_bits, frac_bits,
                                num_kv_splits, ws, need, stream);
}
