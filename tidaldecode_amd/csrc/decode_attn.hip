// Host side of the decode-attention entry points: split planning and argument checks.  The
// kernels live in decode_attn.cuh and are instantiated in decode_attn_{f16,bf16}.hip.
#include "sparse_attn.cuh"

namespace tidal {

static int g_num_cus = 0;

static int num_cus() {
  if (g_num_cus == 0) {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
        n > 0)
      g_num_cus = n;
    else
      g_num_cus = 256;  // MI355X
  }
  return g_num_cus;
}

static int64_t align256(int64_t x) { return (x + 255) & ~(int64_t)255; }

// Workspace layout: [ticket counters, fixed size | partial o | partial (m, l)].  The counters sit
// at a fixed place so that plans of different shapes sharing one workspace never find another
// plan's partial results where they expect zeroed tickets.  A counter has 64 bytes to itself: the
// tickets of a launch are all taken within a microsecond, and counters that share a line queue up
// behind one another at the memory channel (measured: 0.4 us of a 9.7 us launch).
constexpr int kTicketStride = 16;  // int32 words between counters
constexpr int64_t kTickets = 16384;
constexpr int64_t kTicketBytes = kTickets * kTicketStride * 4;

// The short-list kernel (sparse_attn.cuh) covers a list in one pass of at most 64 workgroups per
// head; longer lists go to the streaming kernel, whose waves pipeline several tiles.
constexpr int64_t kSparseMaxItems = 64 * 256;

// Workgroups per head row of a balanced launch (decode_attn_balanced_kernel): as many rounds of one per
// compute unit as give every sequence one; at most kMergedPieces of a sequence are merged.
static int balanced_slots(int n_hrows, int batch) {
  const int round = num_cus() / n_hrows < 1 ? 1 : num_cus() / n_hrows;
  const int64_t slots = ceil_div64(batch, round) * round, merged = (int64_t)batch * kMergedPieces;
  return (int)(slots < merged ? slots : merged);
}

// Whether the balanced launch is worth its search and the merges it adds, from the longest sequence that the plan
// is for; chunk: that of the even plan.  Its workgroups of one tile (`tile` tokens) take `per_tile` us; the lengths
// and the search 1 - 2 us; where the even plan cuts no sequence, starting to merge at all 3 - 6 us, and partials of
// eight heads queue up at the memory.  It pays where equal lengths would gain by more than that, and where the
// even plan's workgroups last so long that their differences are worth more than the search (equal lengths then
// lose 1 - 5 %).  One MI355X, bf16, logits out, even | balanced (with a search of 0.06 us a sequence, now 0.02),
// us: 8/1 heads x 128, 2 x 400 12.4 | 12.7, 2 x 800 18.6 | 13.4, 24 x 800 20.8 | 23.6, 24 x 1600 35.0 | 26.3; 28/4
// heads, 8 x 800 21.9 | 25.8, 24 x 1600 41.3 | 37.7; 32/8 heads, 8 x 400 9.9 | 10.8, 8 x 800 16.3 | 13.0, 24 of 1 ..
// 1600 29.0 | 27.3 and 24 x 1600 31.5 | 33.1, 24 of 1 .. 4000 62.9 | 51.4, 64 x 800 (as many sequences as slots: none
// is cut) 42.9 | 50.2; 32/8 heads x 64, 8 x 400 10.6 | 12.2, 8 x 800 13.8 | 12.8; 16/4 heads x 256, 8 x 100 10.2 |
// 12.0, 8 x 200 13.7 | 12.6.
static bool balancing_pays(int head_dim, int qpg, int n_hrows, int batch, int64_t max_items, int tile, int64_t chunk,
                           int slots) {
  const int64_t tiles = ceil_div64(max_items, tile), even = ceil_div64(max_items, chunk);
  int64_t piece = ceil_div64(tiles * batch, slots);
  if (piece < ceil_div64(tiles, kMergedPieces)) piece = ceil_div64(tiles, kMergedPieces);
  const int64_t longest = tiles < chunk / tile ? tiles : chunk / tile;
  if (slots <= batch || tiles < 1 || piece > longest) return false;
  const double per_tile = head_dim == 256 ? 2.35 : (head_dim == 64 ? 1.35 : (qpg == 8 ? 1.75 : 1.25));
  const double merge = even > 1 ? 1.5 : (head_dim == 256 ? 6.0 : (head_dim == 64 ? 3.0 : (qpg == 8 ? 5.4 : 4.8)));
  const double more = (double)n_hrows * batch * (ceil_div64(tiles, piece) - even);
  const double cost = merge + (qpg == 8 ? more * head_dim * (0.036 / 128) : 0.0);
  return (double)(longest - piece) * per_tile > cost || (double)longest * per_tile >= (even > 1 ? 8.0 : 20.0);
}

// What a short-list launch takes beyond its fixed 3 us, in us: workgroups of nw waves, `tiles` tiles of a workgroup
// each (but for the last), rows x splits of them, dealt evenly to the compute units.  A compute unit by itself
// takes 11 ns a token of 128 dimensions and 0.8 for every further trip of a wave; all together read 8 TB/s at
// most; splits are merged, 16 partials at a time.  The constants fit nine head shapes, lists of 64 to 6000 tokens and
// six workgroup shapes each (us, lists of 200 | 400 | 1300 | 4096 tokens): 32 heads x 128, four waves x 128 tokens
// 6.2 | 6.4 | 9.1 | 16.1, eight x 256 5.6 | 7.8 | 8.7 | 15.5, eight x 512 5.6 | 8.8 | 12.1 | 15.5; 28/4 heads 7.5 | 7.5 |
// 7.7 | 9.4, 6.1 | 8.9 | 9.3 | 9.6, 6.2 | 9.3 | 12.7 | 13.1; 40 heads x 64, four waves x 256 4.8 | 6.6 | 7.5 | 13.5,
// eight x 512 4.9 | 6.6 | 9.1 | 15.3.  Powers of two alone, which the chunks were, cost 32 heads 5 % at 6000 tokens.
static float short_list_cost(int head_dim, int qpg, int rows, int items, int nw, int tiles, int splits) {
  const int wave_tile = 4096 / head_dim, cus = num_cus();
  const int wgs = rows * splits, active = wgs < cus ? wgs : cus;
  const int tokens = splits > 1 ? tiles * nw * wave_tile : (items + wave_tile - 1) / wave_tile * wave_tile;
  const float per_cu = (float)((wgs + cus - 1) / cus) * (float)tokens * (float)head_dim;
  const float alone = per_cu * (qpg > 1 ? 0.0125f / 128.f : 0.0112f / 128.f) + 0.8f * (float)(tiles - 1);
  const float together = per_cu * (float)active * (4.f / 8.0e6f);
  float merge = splits == 1 && tiles == 1 ? 0.02f * (float)(nw - tokens / wave_tile) : 0.f;  // idle waves
  if (splits > 1)
    merge = (qpg == 8 ? 2.f : (qpg > 1 ? 1.75f : 1.4f)) + (float)((splits - 1) / 16) * (qpg == 8 ? 1.f : 0.7f) +
            (qpg > 1 ? 0.02f : 0.01f) * (float)splits;
  return (alone > together ? alone : together) + merge;
}

static bool is_pow2(int64_t x) { return x > 0 && (x & (x - 1)) == 0; }

// Token-slot lists without score output go to the short-list kernel, and of the others the calls that read up to 72 MiB
// (width: elements of K a token, and as many of V) and, in a batch, up to 2048 tokens a sequence.
// Its one trip from list to rows saves the streaming kernel's pipeline where that never fills.  Two selection
// layers, one sparse one and their top-k, us, streaming -> short-list: 32 heads x 128 at 300 tokens 35.5 -> 31.6,
// 4000 59.3 -> 56.2, 6000 (98 MB) 68.7 -> 71.8; 16 heads 8000 58.5 -> 55.1; 32/8 heads 2500 46.0 -> 42.5, 8000 57.2 ->
// 49.7; 28/4 heads 4000 52.2 -> 44.4; 4 sequences of 500 .. 2000, 32/8 heads, 54.7 -> 46.7; 6 of 1000 .. 4000 (101 MB)
// 69.6 -> 74.6.  Where the pool then excludes the short-list kernel its chunks serve the streaming kernel no worse than
// those planned for that: pages of 12 tokens, 8 sequences of 2000, 28/4 heads 13.4 | 14.5, one of 4000, 32/8 heads 10.4 |
// 11.6, 16 of 1500, 32/8 heads 24.4 | 24.4.
static bool short_list_pays(bool slots, bool scores, int64_t batch, int64_t max_items, int64_t width) {
  return (slots && !scores) || ((batch == 1 || max_items <= 2048) && batch * max_items * width <= (72 << 20) / 4);
}

}  // namespace tidal

// Scratch of td_decode_attn_noalloc: ticket counters and split partials in device memory that
// belongs to the library image, for callers that must not allocate.  Zero when the image is
// loaded; every launch leaves the ticket counters zero again.
static __device__ __align__(256) unsigned char scratch[TD_STATIC_SCRATCH_BYTES];

namespace tidal {

// Device address of `scratch` on the current device.  The array's name is a host-side handle, not
// a device address: the address is looked up once per device (each device holds its own copy)
// and that pointer is what the launches get.
static int static_scratch(void** out) {
  constexpr int kMaxDevices = 64;
  static void* ptr_of[kMaxDevices] = {};
  int dev = 0;
  TD_HIP_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices)
    return fail(TD_ERR_UNSUPPORTED, "td_decode_attn_noalloc: device %d (at most %d devices)", dev, kMaxDevices);
  void* ptr = __atomic_load_n(&ptr_of[dev], __ATOMIC_ACQUIRE);
  if (ptr == nullptr) {
    TD_HIP_CHECK(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    if (ptr == nullptr) return fail(TD_ERR_HIP, "hipGetSymbolAddress returned a NULL scratch address");
    __atomic_store_n(&ptr_of[dev], ptr, __ATOMIC_RELEASE);
  }
  *out = ptr;
  return TD_OK;
}

}  // namespace tidal

using namespace tidal;

// kernel family that served this thread's last td_decode_attn call
static thread_local const char* g_last_kernel = "none";

extern "C" const char* td_last_decode_kernel(void) { return g_last_kernel; }

extern "C" int td_num_cus(void) { return num_cus(); }

extern "C" int td_decode_make_plan(int32_t batch, int32_t num_qo_heads, int32_t num_kv_heads,
                              int32_t head_dim, int32_t idx_rows, int64_t max_items,
                              td_decode_plan* plan) {
  TD_REQUIRE(plan != nullptr, "td_decode_make_plan: plan is NULL");
  TD_REQUIRE(batch >= 1, "td_decode_make_plan: batch %d < 1", batch);
  TD_REQUIRE(num_kv_heads >= 1 && num_qo_heads >= num_kv_heads && num_qo_heads % num_kv_heads == 0,
             "td_decode_make_plan: num_qo_heads %d must be a positive multiple of num_kv_heads %d",
             num_qo_heads, num_kv_heads);
  if (head_dim != 64 && head_dim != 128 && head_dim != 256)
    return fail(TD_ERR_UNSUPPORTED, "td_decode_make_plan: head_dim %d (supported: 64, 128, 256)",
                head_dim);
  TD_REQUIRE(idx_rows == 1 || idx_rows == num_kv_heads || idx_rows == num_qo_heads,
             "td_decode_make_plan: idx_rows %d must be 1, num_kv_heads (%d) or num_qo_heads (%d)",
             idx_rows, num_kv_heads, num_qo_heads);
  TD_REQUIRE(max_items >= 0 && max_items < ((int64_t)1 << 30), "td_decode_make_plan: max_items %lld",
             (long long)max_items);

  const int qpg = qpg_for(num_qo_heads, num_kv_heads, idx_rows, head_dim);
  const int subs = qpg > 1 ? (num_qo_heads / num_kv_heads + qpg - 1) / qpg : 1;
  const int n_hrows = qpg > 1 ? num_kv_heads * subs : num_qo_heads;
  {
    // Planning happens before the launches it serves (and outside any stream capture): a good
    // moment to look up this device's static scratch for td_decode_attn_noalloc.  Without a
    // device the lookup fails and is simply tried again by that entry point.
    void* unused = nullptr;
    (void)static_scratch(&unused);
  }

  // ---- short lists: the sparse-layer kernel -------------------------------------------------------
  // Chunks are a multiple of the workgroup tile; the streaming kernel at 8 waves x 4 rows (tile 128, 256 at
  // head_dim 64) can run the same plan when a call turns out not to fit the short-list kernel.
  int sw = plan->sparse_waves, sr = plan->sparse_rows;
  plan->balanced = 0;
  // one query head per list walk, or a KV head's up to eight query heads sharing its list; the streaming kernel takes
  // what has more head slots than there are tickets, as it needs but one a head row
  bool sparse = sw >= 0 && sr >= 0 && head_dim <= 128 && subs == 1 && max_items > 0 &&
                max_items <= kSparseMaxItems && (int64_t)batch * n_hrows * qpg <= kTickets &&
                (plan->chunk_tokens == 0 || is_pow2(plan->chunk_tokens));
  if ((qpg > 1 || head_dim == 64) && sr == 16) sparse = false;  // 8 rows per lane only
  if (sparse && !sparse_shape_supported(sw == 0 ? 8 : sw, sr == 0 ? 8 : sr, qpg)) {
    // head_dim 64 and other groups had no short-list kernel to preset once, and keep ignoring what it does not have
    const int group = num_qo_heads / num_kv_heads;
    if (head_dim == 128 && (qpg == 1 ? is_pow2(group) : qpg == group))
      return fail(TD_ERR_UNSUPPORTED,
                  "td_decode_make_plan: no short-list kernel with %d waves x %d rows (4 or 8 waves, 8 or "
                  "16 rows)", sw, sr);
    sparse = false;
  }
  if (sparse) {
    // Workgroup shape and chunk with the least cost; more tiles or fewer waves have to gain.  Splits whose partials
    // do not fit the built-in scratch are left alone, as that would refuse callers who have no other.
    int64_t chunk = plan->chunk_tokens;
    const int rows_all = n_hrows * batch;
    auto fits = [&](int64_t splits) {
      return splits == 1 || kTicketBytes + (int64_t)rows_all * qpg * splits * (head_dim + 2) * 4 + 512 <=
                                (int64_t)TD_STATIC_SCRATCH_BYTES;
    };
    if (chunk == 0 && sr != 16) {
      const int items = (int)max_items;
      float best = 0.f;
      const int preset = sw;
      for (int nw = 8; nw >= 4; nw -= 4) {
        if (preset != 0 && preset != nw) continue;
        const int stile = nw * (4096 / head_dim), most = (items + stile - 1) / stile;
        for (int tiles = 1;; tiles += tiles < 4 ? 1 : (tiles < 16 ? tiles / 4 * 2 : tiles / 2)) {
          if (tiles > most) tiles = most;
          const int splits = (most + tiles - 1) / tiles;
          if (splits <= 64 && fits(splits)) {
            const float cost = short_list_cost(head_dim, qpg, rows_all, items, nw, tiles, splits);
            if (best == 0.f || cost < best - 0.01f) {
              best = cost;
              sw = nw;
              chunk = (int64_t)tiles * stile;
            } else if (cost > best + 3.f && rows_all * splits <= num_cus()) {
              break;  // longer walks on fewer compute units: no merge costs that much
            }
          }
          if (tiles == most) break;
        }
      }
    } else if (chunk == 0) {
      chunk = 256;
      while (!fits(ceil_div64(max_items, chunk))) chunk <<= 1;
    }
    while (ceil_div64(max_items, chunk) > 64) chunk <<= 1;
    if (sr == 0) sr = 8;
    if (sw == 0) sw = (chunk < 32768 / head_dim || sr == 16) ? 4 : 8;
    const int stile = sw * (512 / head_dim) * sr;
    if (plan->chunk_tokens == 0 && chunk < stile) chunk = stile;  // a preset shape with a larger tile
    if (chunk % stile != 0 || chunk % (16384 / head_dim) != 0) {
      sparse = false;
    } else {
      plan->chunk_tokens = (int32_t)chunk;
      plan->max_splits = (int32_t)ceil_div64(max_items, chunk);
      plan->waves_per_block = 8;
      plan->tile_rows = 4;
      plan->sparse_waves = sw;
      plan->sparse_rows = sr;
    }
  }
  if (sparse) {
    if (plan->fused_merge < 0) plan->fused_merge = 1;
    plan->fused_merge = plan->fused_merge ? 1 : 0;
    const int64_t n_part = (int64_t)batch * n_hrows * qpg * plan->max_splits;
    plan->workspace_bytes = kTicketBytes + align256(n_part * head_dim * 4) + align256(n_part * 2 * 4);
    return TD_OK;
  }
  plan->sparse_waves = plan->sparse_rows = 0;

  int nw = plan->waves_per_block;
  if (nw == 0) nw = 8;
  if (qpg > 1) nw = 8;  // the shared-row kernels exist for 8 waves only
  // K/V rows per lane group and tile of the streaming kernel: 4 unless the caller presets 2
  // (short token-slot lists have a kernel of their own, above).
  int rows = plan->tile_rows;
  if (rows == 0) rows = 4;
  if (!shape_supported(head_dim, qpg, nw, rows))
    return fail(TD_ERR_UNSUPPORTED,
                "td_decode_make_plan: no kernel for head_dim %d, %d query heads per shared KV row, %d "
                "waves per block, %d rows per tile",
                head_dim, qpg, nw, rows);
  // tokens one pass of the workgroup covers: waves x instructions x rows per instruction
  const int tile = nw * rows * (64 / (head_dim / 8));

  // Aim at one round of workgroups that fills the chip, never less than one pass per workgroup,
  // never more than 64 partials per head.  The one-head-per-row kernels fit two 8-wave workgroups
  // on a compute unit (128 registers: four waves per SIMD), so their round is 2 per compute unit.
  // The shared-row kernels (141-256 registers) fit ONE: with twice as many workgroups the second
  // half waits for the first, and a few workgroups over one round double the launch (32/8 heads
  // x 128 at 100K tokens: 31 splits = 248 workgroups 84 us, 62 splits = 496 workgroups 90 us,
  // 34 splits = 272 workgroups 120 us; at 32K 33 us against 41, at 10K 18 against 26).  Their
  // round is kept a little under the compute-unit count: 256 workgroups on 256 compute units
  // measured like a round and a bit (124 us), 248 and fewer did not.
  const int64_t target_blocks = qpg > 1 ? (int64_t)num_cus() - num_cus() / 32 : (int64_t)num_cus() * 2;
  int64_t splits = target_blocks / ((int64_t)n_hrows * batch);
  if (splits < 1) splits = 1;
  if (splits > 64) splits = 64;
  int64_t chunk = max_items > 0 ? ceil_div64(max_items, splits) : tile;
  // A batch is planned from its longest sequence: chunks of that size leave the short sequences
  // with one long-running workgroup per head and the launch waits for the longest.  Finer chunks
  // balance a ragged batch (8 sequences of 14K-63K tokens: 935 -> 769 us at 4096 tokens) and end
  // closer together; from 1024 tokens down the merges take back what that gives.  32 heads x 128,
  // fp16, logits out, chunks of 4096 | 1024 tokens (or as near as the built-in scratch allows): 8
  // sequences of 8192 .. 65536 1017 | 998 us, of 500 .. 8000 136 | 118; 16 heads, 8 of 2000 .. 30000
  // 254 | 240; 40 heads, 3 of 2000 .. 40000 210 | 196.  Equal lengths, which need no balance, lose a
  // little: 8 of 8192 180.7 | 183.3.
  if (batch > 1 && qpg == 1 && chunk > 1024) {
    const int64_t per_split = (int64_t)batch * n_hrows * (head_dim + 2) * 4;
    int64_t fit = ((int64_t)TD_STATIC_SCRATCH_BYTES - kTicketBytes - 512) / per_split;  // splits it holds
    if (fit < ceil_div64(max_items, 4096)) fit = ceil_div64(max_items, 4096);
    const int64_t finest = ceil_div64(max_items, fit < 64 ? fit : 64);
    const int64_t wanted = finest > 1024 ? ceil_div64(finest, tile) * tile : 1024;
    if (chunk > wanted) chunk = wanted;
    if (chunk > 4096) chunk = 4096;
  }
  // Shared rows in a batch: whole rounds of one workgroup per compute unit.  The split count with
  // the fewest rounds per split wins, chunks of 1024 tokens at least
  // (32/8 heads, 16 sequences x 8192 tokens: 2 splits = 256 workgroups 94 us, 3 splits 110, 1
  // split 130; 8 x 32768: 4 splits 172 us, 3 splits 187, 8 splits of 4096 tokens 182; 12 x 16384:
  // 5 splits = 2 rounds 136 us, 8 splits = 3 rounds 136, 4 splits 151, 3 splits 187).
  if (batch > 1 && qpg > 1 && max_items > 0) {
    const int64_t r = (int64_t)n_hrows * batch, cus = num_cus();
    int64_t s_max = max_items / 1024;
    s_max = s_max < 1 ? 1 : (s_max > 64 ? 64 : s_max);
    int64_t best_s = 1, best_rounds = ceil_div64(r, cus);
    for (int64_t s_try = 2; s_try <= s_max; ++s_try) {
      const int64_t rounds = ceil_div64(r * s_try, cus);
      // more splits in as many rounds always gain; more rounds have to gain 1/16 per split
      const bool better = rounds <= best_rounds ? rounds * best_s < best_rounds * s_try
                                                : rounds * best_s * 16 < best_rounds * s_try * 15;
      if (better) {
        best_s = s_try;
        best_rounds = rounds;
      }
    }
    chunk = ceil_div64(max_items, best_s);
  }
  if (plan->chunk_tokens > 0) chunk = plan->chunk_tokens;
  chunk = ceil_div64(chunk, tile) * tile;
  int64_t max_splits = max_items > 0 ? ceil_div64(max_items, chunk) : 1;
  if (max_splits > 64) {  // keep the merge bounded: widen the chunks
    chunk = ceil_div64(ceil_div64(max_items, 64), tile) * tile;
    max_splits = ceil_div64(max_items, chunk);
  }
  if (max_splits < 1) max_splits = 1;
  // room for the partials of a balanced launch (one per slot and head slot), unless that alone would take
  // the plan beyond the built-in scratch
  plan->balanced = batch > 1 && batch <= kBalancedMaxBatch && qpg > 1 && plan->chunk_tokens == 0 &&
                   balancing_pays(head_dim, qpg, n_hrows, batch, max_items, tile, chunk, balanced_slots(n_hrows, batch));
  if (plan->balanced) {
    const int64_t wanted = ceil_div64(balanced_slots(n_hrows, batch), batch);
    const int64_t bytes = kTicketBytes + (int64_t)batch * n_hrows * qpg * wanted * (head_dim + 2) * 4 + 512;
    if (wanted > max_splits && bytes <= (int64_t)TD_STATIC_SCRATCH_BYTES) max_splits = wanted;
  }

  plan->chunk_tokens = (int32_t)chunk;
  plan->max_splits = (int32_t)max_splits;
  plan->waves_per_block = nw;
  plan->tile_rows = rows;
  if (plan->fused_merge < 0) plan->fused_merge = 1;
  plan->fused_merge = plan->fused_merge ? 1 : 0;
  TD_REQUIRE((int64_t)batch * n_hrows <= kTickets,
             "td_decode_make_plan: batch %d x %d head rows exceeds the %lld ticket counters", batch,
             n_hrows, (long long)kTickets);
  const int64_t n_part = (int64_t)batch * n_hrows * qpg * max_splits;  // head slots incl. padding
  plan->workspace_bytes = kTicketBytes + align256(n_part * head_dim * 4) + align256(n_part * 2 * 4);
  return TD_OK;
}

// Argument checks and the kernel parameter block shared by td_decode_attn and td_gather_probe.
static int build_params(const td_paged_kv* kv, const td_index_list* list, const td_decode_plan* plan,
                        const void* q, void* o, int32_t batch, int32_t num_qo_heads, float sm_scale,
                        void* scores, int32_t scores_dtype, int64_t score_stride, float* lse,
                        const td_fresh_token* fresh, void* workspace, int64_t workspace_bytes,
                        DecodeParams& p, int& qpg_out, int& n_hrows_out) {
  TD_REQUIRE(kv && list && plan && q && o, "td_decode_attn: NULL argument");
  TD_REQUIRE(kv->data != nullptr, "td_decode_attn: kv->data is NULL");
  TD_REQUIRE(batch >= 1, "td_decode_attn: batch %d < 1", batch);
  const int Hkv = kv->num_kv_heads, D = kv->head_dim, P = kv->page_size;
  if (D != 64 && D != 128 && D != 256)
    return fail(TD_ERR_UNSUPPORTED,
                "BatchDecodeWithPagedKVCache failed to dispatch: head_dim %d (supported: 64, 128, 256)",
                D);
  TD_REQUIRE(Hkv >= 1 && num_qo_heads >= Hkv && num_qo_heads % Hkv == 0,
             "td_decode_attn: num_qo_heads %d must be a positive multiple of num_kv_heads %d",
             num_qo_heads, Hkv);
  TD_REQUIRE(P >= 1 && kv->max_pages >= 1, "td_decode_attn: page_size %d / max_pages %lld", P,
             (long long)kv->max_pages);
  TD_REQUIRE(kv->max_pages * P < ((int64_t)1 << 31), "td_decode_attn: pool too large for int32 slots");
  TD_REQUIRE(kv->layout == TD_NHD || kv->layout == TD_HND, "td_decode_attn: layout %d", kv->layout);
  if (kv->dtype != TD_F16 && kv->dtype != TD_BF16)
    return fail(TD_ERR_UNSUPPORTED,
                "BatchDecodeWithPagedKVCache failed to dispatch with dtype %d (supported: fp16, bf16)",
                kv->dtype);
  TD_REQUIRE(list->idx_rows == 1 || list->idx_rows == Hkv || list->idx_rows == num_qo_heads,
             "td_decode_attn: idx_rows %d must be 1, %d or %d", list->idx_rows, Hkv, num_qo_heads);
  TD_REQUIRE(list->kind == TD_IDX_PAGES || list->kind == TD_IDX_SLOTS, "td_decode_attn: kind %d",
             list->kind);
  TD_REQUIRE(list->n_list_host >= 0, "td_decode_attn: n_list_host %d", list->n_list_host);
  TD_REQUIRE(list->count_arr == nullptr || list->indptr != nullptr,
             "td_decode_attn: count_arr needs indptr (the first column of every sequence)");
  TD_REQUIRE(list->idx != nullptr || list->n_list_host == 0,
             "td_decode_attn: idx is NULL but n_list_host is %d", list->n_list_host);
  TD_REQUIRE(list->idx_rows == 1 || list->idx_row_stride >= list->n_list_host,
             "td_decode_attn: idx_row_stride %d < n_list_host %d", list->idx_row_stride,
             list->n_list_host);
  TD_REQUIRE(list->last_page_len >= 0 && list->last_page_len <= P,
             "td_decode_attn: last_page_len %d not in [0, %d]", list->last_page_len, P);
  TD_REQUIRE(list->last_page_idx >= 0 && list->last_page_idx < kv->max_pages,
             "td_decode_attn: last_page_idx %d outside the pool of %lld pages", list->last_page_idx,
             (long long)kv->max_pages);
  TD_REQUIRE(plan->chunk_tokens > 0 && plan->max_splits >= 1 && plan->waves_per_block > 0 &&
                 plan->tile_rows > 0 &&
                 plan->chunk_tokens % (plan->waves_per_block * plan->tile_rows * (64 / (D / 8))) == 0,
             "td_decode_attn: plan not produced by td_decode_make_plan");
  // the planned split must cover every token the list can describe
  const int64_t max_items = (int64_t)list->n_list_host * (list->kind == TD_IDX_PAGES ? P : 1) +
                            (list->last_page_len_arr ? P : list->last_page_len);
  if (max_items > (int64_t)plan->chunk_tokens * plan->max_splits)
    return fail(TD_ERR_STATE,
                "td_decode_attn: the list describes up to %lld tokens but the plan covers %lld "
                "(call td_decode_make_plan / begin_forward for this budget first)",
                (long long)max_items, (long long)plan->chunk_tokens * plan->max_splits);
  if (scores) {
    TD_REQUIRE(scores_dtype == TD_F32 || scores_dtype == kv->dtype,
               "td_decode_attn: scores dtype %d must be fp32 or the KV dtype", scores_dtype);
    TD_REQUIRE(score_stride > 0, "td_decode_attn: score_stride %lld", (long long)score_stride);
  }

  const int qpg = qpg_for(num_qo_heads, Hkv, list->idx_rows, D);
  const int subs = qpg > 1 ? (num_qo_heads / Hkv + qpg - 1) / qpg : 1;
  const int n_hrows = qpg > 1 ? Hkv * subs : num_qo_heads;
  qpg_out = qpg;
  n_hrows_out = n_hrows;

  const int64_t n_part = (int64_t)batch * n_hrows * qpg * plan->max_splits;
  const int64_t off_o = kTicketBytes;
  const int64_t off_ml = off_o + align256(n_part * D * 4);
  const int64_t need = off_ml + align256(n_part * 2 * 4);
  TD_REQUIRE((int64_t)batch * n_hrows <= kTickets,
             "td_decode_attn: batch %d x %d head rows exceeds the ticket counters", batch, n_hrows);
  TD_REQUIRE(plan->max_splits <= 64, "td_decode_attn: plan has %d splits (limit 64)",
             plan->max_splits);
  if (plan->max_splits > 1) {
    if (workspace == nullptr || workspace_bytes < need)
      return fail(TD_ERR_STATE,
                  "td_decode_attn: workspace of %lld bytes is smaller than the %lld the plan needs "
                  "(call td_decode_make_plan / begin_forward first)",
                  (long long)workspace_bytes, (long long)need);
  }

  p.q = q;
  p.o = o;
  p.kv = kv->data;
  p.page_stride = (int64_t)2 * P * Hkv * D;
  p.v_offset = (int64_t)P * Hkv * D;
  if (kv->layout == TD_NHD) {
    p.entry_stride = Hkv * D;
    p.head_stride = D;
  } else {
    p.entry_stride = D;
    p.head_stride = P * D;
  }
  p.page_size = P;
  p.page_shift = -1;
  for (int sft = 0; sft < 31; ++sft)
    if ((1 << sft) == P) p.page_shift = sft;
  p.max_slot = (uint32_t)(kv->max_pages * P - 1);
  p.page_stride_b = (uint32_t)(p.page_stride * 2);
  p.entry_stride_b = (uint32_t)(p.entry_stride * 2);
  p.lean = (p.page_shift >= 0 && (int64_t)kv->max_pages * p.page_stride * 2 < ((int64_t)1 << 32)) ? 1 : 0;
  p.fresh_k = p.fresh_v = nullptr;
  p.fresh_cos = p.fresh_sin = nullptr;
  p.fresh_slot = nullptr;
  if (fresh) {
    TD_REQUIRE(fresh->k && fresh->v && fresh->cos && fresh->sin && fresh->dst_slot,
               "td_decode_attn: fresh token with a NULL member");
    p.fresh_k = fresh->k;
    p.fresh_v = fresh->v;
    p.fresh_cos = fresh->cos;
    p.fresh_sin = fresh->sin;
    p.fresh_slot = fresh->dst_slot;
  }
  p.num_qo_heads = num_qo_heads;
  p.n_hrows = n_hrows;
  p.vheads = n_hrows * qpg;
  p.subs = subs;
  p.q_per_kv = num_qo_heads / Hkv;
  p.idx = list->idx;
  p.idx_row_stride = list->idx_rows == 1 ? 0 : list->idx_row_stride;
  p.idx_cols = list->idx_row_stride > 0 ? list->idx_row_stride : 0;
  p.idx_per_kv = (qpg == 1 && list->idx_rows == Hkv && Hkv != num_qo_heads) ? 1 : 0;
  p.page_mode = list->kind == TD_IDX_PAGES ? 1 : 0;
  p.max_page = (uint32_t)(kv->max_pages - 1);
  p.indptr = list->indptr;
  p.count_arr = list->count_arr;
  p.n_list_host = list->n_list_host;
  p.last_len_arr = list->last_page_len_arr;
  p.last_idx_arr = list->last_page_idx_arr;
  p.last_len = list->last_page_len;
  p.last_idx = list->last_page_idx;
  p.chunk_tokens = plan->chunk_tokens;
  p.chunk_magic = plan->chunk_tokens > 1 ? (uint32_t)((((uint64_t)1 << 32) + plan->chunk_tokens - 1) / plan->chunk_tokens) : 0;
  p.num_kv_heads = Hkv;
  p.kv_magic = ((1u << 24) + (uint32_t)p.q_per_kv - 1) / (uint32_t)p.q_per_kv;
  p.list_shift = p.page_mode ? p.page_shift : 0;
  p.max_splits = plan->max_splits;
  p.fused_merge = plan->fused_merge;
  p.scale_log2 = sm_scale * kLog2e;
  p.scores = scores;
  p.scores_f32 = scores_dtype == TD_F32 ? 1 : 0;
  p.score_stride = score_stride;
  p.lse = lse;
  char* ws = reinterpret_cast<char*>(workspace);
  p.ws_cnt = reinterpret_cast<int32_t*>(ws);
  p.ticket_stride = kTicketStride;
  p.batch = batch;
  // Balanced: the full attention of a batch on the shared-row kernels, merged in the launch, when the
  // workspace holds its partials and the caller has not set the chunks.
  p.slots = 0;
  if (plan->balanced && qpg > 1 && batch > 1 && batch <= kBalancedMaxBatch && list->kind == TD_IDX_PAGES &&
      plan->fused_merge) {
    const int slots = balanced_slots(n_hrows, batch);
    if ((int64_t)batch * plan->max_splits >= slots) p.slots = slots;
  }
  p.ws_o = reinterpret_cast<float*>(ws ? ws + off_o : nullptr);
  p.ws_ml = reinterpret_cast<float*>(ws ? ws + off_ml : nullptr);

  return TD_OK;
}

// Whether a call runs on the short-list kernel of its plan: one query head per list walk or a whole group per shared
// list, chunks that are a multiple of the kernel's workgroup tile, a ticket a head slot, and little to read.  Returns 0
// (no), kSparseLean (power-of-two pages, pool below 4 GiB, strides within the 24-bit multiplier: 32-bit row offsets) or
// kSparseWide (any page size, 64-bit row offsets; token-slot lists without score output at head_dim 128 only, 8 rows per
// lane, groups of 1, 2, 4 or 8, and a list per query head in groups of a power of two: the others stay with the streaming
// kernel, as nobody measured them).
enum { kSparseNo = 0, kSparseLean = 1, kSparseWide = 2 };
static int sparse_kernel_fits(const DecodeParams& p, const td_decode_plan* plan,
                              const td_index_list* list, int qpg, int head_dim, bool emit) {
  const bool slots = list->kind == TD_IDX_SLOTS;
  const int64_t listed = (int64_t)list->n_list_host * (slots ? 1 : p.page_size);
  if (plan->sparse_waves <= 0 || !sparse_shape_supported(plan->sparse_waves, plan->sparse_rows, qpg) ||
      (int64_t)p.batch * p.vheads > kTickets)
    return kSparseNo;
  const int stile = plan->sparse_waves * (512 / head_dim) * plan->sparse_rows;
  if (!(head_dim <= 128 && p.subs == 1 && listed + p.page_size <= 2 * kSparseMaxItems && plan->chunk_tokens % stile == 0 &&
        (plan->sparse_rows == 8 || (head_dim == 128 && slots && !emit))))
    return kSparseNo;
  if (!short_list_pays(slots, emit, p.batch, listed + (list->last_page_len_arr ? p.page_size : list->last_page_len),
                       (int64_t)(list->idx_rows == p.num_qo_heads ? p.num_qo_heads : p.num_kv_heads) * head_dim))
    return kSparseNo;
  if (p.lean && p.page_stride_b < (1u << 24) && p.entry_stride_b < (1u << 24)) return kSparseLean;
  // a page's bytes and an entry's offset inside it stay 32-bit; the page base is a 64-bit product
  const bool plain = slots && !emit && head_dim == 128 && (qpg == 1 ? is_pow2(p.q_per_kv) : p.q_per_kv == qpg);
  if (plain && plan->sparse_rows == 8 && p.page_stride * 2 < ((int64_t)1 << 32)) return kSparseWide;
  return kSparseNo;
}

extern "C" int td_short_list_pays(int32_t batch, int32_t num_qo_heads, int32_t num_kv_heads, int32_t head_dim,
                                  int32_t idx_rows, int64_t max_items, int32_t kind, int32_t has_scores) {
  const int64_t width = (int64_t)(idx_rows == num_qo_heads ? num_qo_heads : num_kv_heads) * head_dim;
  return short_list_pays(kind == TD_IDX_SLOTS, has_scores != 0, batch, max_items, width) ? 1 : 0;
}

extern "C" int td_decode_attn(const td_paged_kv* kv, const td_index_list* list,
                              const td_decode_plan* plan, const void* q, void* o, int32_t batch,
                              int32_t num_qo_heads, float sm_scale, void* scores,
                              int32_t scores_dtype, int64_t score_stride, float* lse,
                              const td_fresh_token* fresh, void* workspace,
                              int64_t workspace_bytes, void* stream) {
  DecodeParams p;
  int qpg, n_hrows;
  const int prc = build_params(kv, list, plan, q, o, batch, num_qo_heads, sm_scale, scores, scores_dtype,
                               score_stride, lse, fresh, workspace, workspace_bytes, p, qpg, n_hrows);
  if (prc != TD_OK) return prc;
  const int D = kv->head_dim;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const bool page_mode = list->kind == TD_IDX_PAGES;
  dim3 grid(n_hrows, batch, plan->max_splits);
  const bool merge_kernel = plan->max_splits > 1 && !plan->fused_merge;
  int rc;
  const int fits = sparse_kernel_fits(p, plan, list, qpg, D, scores != nullptr);
  if (fits != kSparseNo) {
    const bool wide = fits == kSparseWide;
    if (qpg > 1)
      rc = kv->dtype == TD_F16
               ? launch_sparse_shared_f16(p, D, plan->sparse_waves, qpg, wide, merge_kernel, grid, st)
               : launch_sparse_shared_bf16(p, D, plan->sparse_waves, qpg, wide, merge_kernel, grid, st);
    else if (kv->dtype == TD_F16)
      rc = launch_sparse_f16(p, D, plan->sparse_waves, plan->sparse_rows, false, wide, merge_kernel, grid, st);
    else
      rc = launch_sparse_bf16(p, D, plan->sparse_waves, plan->sparse_rows, false, wide, merge_kernel, grid, st);
    if (rc != TD_OK) return rc;
    TD_HIP_CHECK(hipGetLastError());
    g_last_kernel = wide ? "short-list, 64-bit offsets" : "short-list";
    return TD_OK;
  }
  if (fresh && !p.lean)
    return fail(TD_ERR_UNSUPPORTED,
                "td_decode_attn: the fused decode step needs a power-of-two page_size and a pool below 4 GiB, but for "
                "token-slot lists of up to %lld entries at head_dim 128 without score output, one per query head "
                "(groups of a power of two) or per 2, 4 or 8 of them (page_size %d, pool %lld bytes); use td_rope_append_decode first",
                (long long)kSparseMaxItems, kv->page_size, (long long)(kv->max_pages * p.page_stride * 2));
  if (kv->dtype == TD_F16)
    rc = launch_decode_f16(p, D, qpg, plan->waves_per_block, plan->tile_rows, page_mode, scores != nullptr,
                           merge_kernel, grid, st);
  else
    rc = launch_decode_bf16(p, D, qpg, plan->waves_per_block, plan->tile_rows, page_mode, scores != nullptr,
                            merge_kernel, grid, st);
  if (rc != TD_OK) return rc;
  TD_HIP_CHECK(hipGetLastError());
  g_last_kernel = p.lean ? "streaming" : "streaming, 64-bit offsets";
  return TD_OK;
}

extern "C" int td_decode_attn_noalloc(const td_paged_kv* kv, const td_index_list* list,
                                      const td_decode_plan* plan, const void* q, void* o,
                                      int32_t batch, int32_t num_qo_heads, float sm_scale,
                                      void* scores, int32_t scores_dtype, int64_t score_stride,
                                      float* lse, const td_fresh_token* fresh, void* stream) {
  TD_REQUIRE(plan != nullptr, "td_decode_attn_noalloc: plan is NULL");
  if (plan->workspace_bytes > (int64_t)TD_STATIC_SCRATCH_BYTES)
    return fail(TD_ERR_STATE,
                "td_decode_attn_noalloc: the plan needs %lld bytes of scratch, the built-in scratch holds "
                "%lld (fewer sequences, heads or splits, or td_decode_attn with a workspace)",
                (long long)plan->workspace_bytes, (long long)TD_STATIC_SCRATCH_BYTES);
  void* ws = nullptr;
  const int rc = static_scratch(&ws);
  if (rc != TD_OK) return rc;
  return td_decode_attn(kv, list, plan, q, o, batch, num_qo_heads, sm_scale, scores, scores_dtype,
                        score_stride, lse, fresh, ws, (int64_t)TD_STATIC_SCRATCH_BYTES, stream);
}

// ---------------------------------------------------------------------------------------------
// Measurement aid: the memory side of a sparse layer alone.  Same grid, same interleaved tiles,
// same list -> slot -> K row / V row non-temporal 16-byte loads as decode_attn_kernel for token
// -slot lists, but no arithmetic, no merge: every wave folds what it loaded into one word and
// stores it.  Its duration is the floor that the attention launch is compared with.
// ---------------------------------------------------------------------------------------------
template <int D, int U, int NW>
__global__ __launch_bounds__(NW * 64) void gather_probe_kernel(const DecodeParams p, uint32_t* out) {
  constexpr int LPR = D / 8, TPI = 64 / LPR, TILE = U * TPI;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane / LPR, li = lane % LPR;
  const int hrow = blockIdx.x, b = blockIdx.y, split = blockIdx.z;
  const int kv_head = hrow / p.q_per_kv;
  SeqList s;
  int list_beg;
  const int n_splits = seq_items(p, b, s, list_beg);
  if (split >= n_splits) return;
  const int idx_row = p.idx_per_kv ? kv_head : hrow;
  s.row = p.idx + (int64_t)idx_row * p.idx_row_stride + list_beg;
  const int c1 = s.n_list;  // listed slots only
  const char* kbase = reinterpret_cast<const char*>(p.kv);
  const char* vbase = kbase + p.v_offset * 2;
  const uint32_t head_byte_off = (uint32_t)(kv_head * p.head_stride + li * 8) * 2u;
  const int STEP = n_splits * NW * TILE;
  u32x4 fold = {0u, 0u, 0u, 0u};
  for (int t = (split * NW + wave) * TILE; t < c1; t += STEP) {
    u32x4 kb[U], vb[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      int i = t + u * TPI + g;
      i = i < c1 ? i : c1 - 1;
      uint32_t slot = (uint32_t)s.row[i];
      slot = slot > p.max_slot ? p.max_slot : slot;
      const uint32_t page = slot >> p.page_shift, entry = slot & ((1u << p.page_shift) - 1u);
      const uint32_t off = page * p.page_stride_b + entry * p.entry_stride_b + head_byte_off;
      kb[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(kbase + off));
      vb[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(vbase + off));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) fold ^= kb[u] ^ vb[u];
  }
  uint32_t w = fold.x ^ fold.y ^ fold.z ^ fold.w;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) w ^= (uint32_t)__shfl_xor((int)w, off, 64);
  if (lane == 0)
    out[(((int64_t)b * gridDim.x + hrow) * gridDim.z + split) * NW + wave] = w;
}

extern "C" int td_gather_probe(const td_paged_kv* kv, const td_index_list* list,
                               const td_decode_plan* plan, int32_t batch, int32_t num_qo_heads,
                               void* out, int64_t out_bytes, void* stream) {
  TD_REQUIRE(out != nullptr, "td_gather_probe: NULL out");
  DecodeParams p;
  int qpg, n_hrows;
  const int prc = build_params(kv, list, plan, out, out, batch, num_qo_heads, 1.f, nullptr, TD_F32, 0,
                               nullptr, nullptr, out, (int64_t)1 << 40, p, qpg, n_hrows);
  if (prc != TD_OK) return prc;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int fits = qpg == 1 && kv->head_dim == 128 && list->kind == TD_IDX_SLOTS && is_pow2(p.q_per_kv)
                       ? sparse_kernel_fits(p, plan, list, qpg, kv->head_dim, false)
                       : kSparseNo;
  if (fits != kSparseNo && list->last_page_len == 0 && !list->last_page_len_arr) {
    // the short-list kernel's own loads-only form; it reads `out` as q and writes nothing
    TD_REQUIRE(out_bytes >= (int64_t)batch * num_qo_heads * kv->head_dim * 2,
               "td_gather_probe: out holds %lld bytes, %lld needed", (long long)out_bytes,
               (long long)batch * num_qo_heads * kv->head_dim * 2);
    const dim3 sgrid(n_hrows, batch, plan->max_splits);
    const bool wide = fits == kSparseWide;
    const int src =
        kv->dtype == TD_F16
            ? launch_sparse_f16(p, 128, plan->sparse_waves, plan->sparse_rows, true, wide, false, sgrid, st)
            : launch_sparse_bf16(p, 128, plan->sparse_waves, plan->sparse_rows, true, wide, false, sgrid, st);
    if (src != TD_OK) return src;
    TD_HIP_CHECK(hipGetLastError());
    return TD_OK;
  }
  const int nw = plan->waves_per_block, rows = plan->tile_rows;
  if (!(list->kind == TD_IDX_SLOTS && p.lean && qpg == 1 && kv->head_dim == 128 &&
        ((nw == 8 && (rows == 4 || rows == 2)) || (nw == 16 && rows == 4)) &&
        list->last_page_len == 0 && !list->last_page_len_arr))
    return fail(TD_ERR_UNSUPPORTED,
                "td_gather_probe: token-slot lists without a forced last page, one query head per "
                "row, head_dim 128, power-of-two pages, pool below 4 GiB only");
  TD_REQUIRE(out_bytes >= (int64_t)batch * n_hrows * plan->max_splits * nw * 4,
             "td_gather_probe: out holds %lld bytes, %lld needed", (long long)out_bytes,
             (long long)batch * n_hrows * plan->max_splits * nw * 4);
  const dim3 grid(n_hrows, batch, plan->max_splits);
  uint32_t* outw = reinterpret_cast<uint32_t*>(out);
  if (nw == 16)
    hipLaunchKernelGGL((gather_probe_kernel<128, 4, 16>), grid, dim3(1024), 0, st, p, outw);
  else if (rows == 2)
    hipLaunchKernelGGL((gather_probe_kernel<128, 2, 8>), grid, dim3(512), 0, st, p, outw);
  else
    hipLaunchKernelGGL((gather_probe_kernel<128, 4, 8>), grid, dim3(512), 0, st, p, outw);
  TD_HIP_CHECK(hipGetLastError());
  return TD_OK;
}
