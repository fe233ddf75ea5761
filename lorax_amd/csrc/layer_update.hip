// Host-side router of one LoRA layer update - no device code in this file.
//
// Restates lorax_amd/layers.py's general path (LoraLinear._decode and _prefill: which launches, which problems share
// one, in which order) over the records of lorax_build_batch_tables, and issues the launches through the library's own
// entry points.  In Python that took 33 us (rank 16, a short prefill) to 204 us (q/k/v of four ranks) per call around
// two to nine launches of 3 to 15 us each: a decode step of one request spent 1.72 ms in 0.22 ms of kernels.
#include "kernels.h"

namespace {

constexpr int kMaxJobs = 256;        // (projection, rank group) pairs of one call
constexpr int kMaxKernelRank = 128;
constexpr int64_t kMaxBgmvRows = 65535;  // rows of a BGMV launch and records of one routing plan
constexpr int64_t kShortBatchRows = 512;  // largest batch of the streaming shrink and of lorax_sgmv_lora_multi at rank 8
constexpr int64_t kShortBatchRows16 = 128;  // ... and of the latter at rank 16 (lorax_prefill_in_one_launch)
constexpr int kFusedSlab = 128 * 1024;      // bytes of A that the single-launch updates read again per slice or row chunk
constexpr int kFusedWidthMax = 16384;       // columns up to which repeating the shrink per slice can pay (an LM head: no)
constexpr int kNumCus = 256;
constexpr int kGroupedRank = 64;      // lorax_shrink_summed_rank
constexpr int kGroupedTileRows = 32;  // highest row tiles that lorax_sgmv_shrink_groups takes several groups of in one launch
constexpr int kShrinkBatch = 16;      // groups of one call of lorax_sgmv_shrink_groups

struct Job {
  const lorax_table_group_t* g;
  int64_t y_offset;
  int32_t width;
  char* v;  // [num_tokens, rank] piece of the workspace
  const void* a_stack;  // stacked weights: the plan's records name entries of these tensors; else null
  const void* b_stack;
};

// What every launch of the call shares.
struct Call {
  const char* tables;
  void* y;
  int64_t y_stride;
  const void* x;
  int64_t rows;
  int32_t h_in;
  int64_t layer_idx;
  void* tmp;
  int64_t tmp_bytes;
  int32_t dtype;
  void* stream;
};

bool fused_rank(int r, int64_t h_in) { return (r == 8 || r == 16) && r * h_in * 2 <= kFusedSlab; }

const void* at(const Call& c, int64_t off) { return c.tables + off; }

lorax_bgmv_problem_t plan_problem(const Call& c, const Job& j, void* y, const void* x, int64_t y_offset, int64_t y_stride,
                                  int32_t h_out, int32_t h_in, const void* a_stack, const void* b_stack) {
  return {y, x, nullptr, nullptr, y_offset, y_stride, h_out, static_cast<const int64_t*>(at(c, j.g->plan_off)),
          j.g->num_chunks, h_in, a_stack, b_stack};
}

// One planned launch for up to 16 jobs: x -> v (shrink) or v -> y (expand).
int bgmv_jobs(const Call& c, const Job* const* jobs, int count, bool shrink) {
  lorax_bgmv_problem_t p[lorax::kMaxBgmvProblems];
  for (int i = 0; i < count; ++i) {
    const Job& j = *jobs[i];
    const int r = j.g->rank;
    p[i] = shrink ? plan_problem(c, j, j.v, c.x, 0, r, r, c.h_in, j.a_stack, nullptr)
                  : plan_problem(c, j, c.y, j.v, j.y_offset, c.y_stride, j.width, r, nullptr, j.b_stack);
  }
  return lorax_bgmv_multi(p, count, c.rows, shrink ? c.h_in : p[0].h_in, c.layer_idx, 1.0f, shrink ? 0 : 1, c.dtype, c.stream);
}

int decode(const Call& c, Job* const* jobs, int count) {
  lorax_decode_job_t route[kMaxJobs];
  for (int i = 0; i < count; ++i) route[i] = {jobs[i]->g->rank, jobs[i]->width, jobs[i]->g->num_chunks};
  if (lorax_decode_in_one_launch(route, count, c.rows, c.h_in)) {
    for (int r : {8, 16}) {
      lorax_bgmv_problem_t p[lorax::kMaxFusedBgmvProblems];
      int n = 0;
      for (int i = 0; i <= count; ++i) {
        if (n > 0 && (i == count || n == lorax::kMaxFusedBgmvProblems)) {
          if (int rc = lorax_bgmv_lora_multi(p, n, c.rows, c.h_in, r, c.layer_idx, 1.0f, c.dtype, c.stream)) return rc;
          n = 0;
        }
        if (i < count && jobs[i]->g->rank == r)
          p[n++] = plan_problem(c, *jobs[i], c.y, c.x, jobs[i]->y_offset, c.y_stride, jobs[i]->width, 0, jobs[i]->a_stack,
                                jobs[i]->b_stack);
      }
    }
    return LORAX_OK;
  }
  for (int i = 0; i < count; i += lorax::kMaxBgmvProblems) {
    const int n = count - i < lorax::kMaxBgmvProblems ? count - i : lorax::kMaxBgmvProblems;
    if (int rc = bgmv_jobs(c, jobs + i, n, true)) return rc;
    if (int rc = bgmv_jobs(c, jobs + i, n, false)) return rc;
  }
  return LORAX_OK;
}

int prefill(const Call& c, Job* const* jobs, int count) {
  const Job* expand[kMaxJobs];
  const Job* shorts[kMaxJobs];
  int32_t expand_segments[kMaxJobs];
  int num_expand = 0, num_shorts = 0;
  lorax_sgmv_shrink_problem_t problems[kShrinkBatch][lorax::kMaxShrinkGroup];
  lorax_sgmv_tiles_t tiles[kShrinkBatch];
  lorax_sgmv_shrink_group_t shrinks[kShrinkBatch];
  int num_shrinks = 0;
  auto flush_shrinks = [&]() {
    const int n = num_shrinks;
    num_shrinks = 0;
    return lorax_sgmv_shrink_groups(shrinks, n, c.x, c.rows, c.h_in, c.layer_idx, 1.0f, 0, c.tmp, c.tmp_bytes, c.dtype,
                                    c.stream);
  };
  // `jobs` is ordered by group of equal rank and segment tables: [first, end) of each
  struct Group {
    int first, end;
    bool fused;      // shrink and expand in one launch
    bool split;      // segments of a few rows go to the per-token kernels, where every projection has a plan over them
    int32_t n_long;  // segments for the segment kernels
    bool planned;    // the tables' row-tile plans cover these
  } group_of[kMaxJobs];
  lorax_shrink_plan_t plans[kMaxJobs];
  int num_groups = 0, num_plans = 0;
  for (int i = 0; i < count; i = group_of[num_groups++].end) {
    const lorax_table_group_t& g = *jobs[i]->g;
    Group& q = group_of[num_groups];
    q = {i, i, false, c.rows <= kMaxBgmvRows, 0, false};
    int widest = 0;
    for (; q.end < count && jobs[q.end]->g->rank == g.rank && jobs[q.end]->g->segments_id == g.segments_id; ++q.end) {
      const Job& j = *jobs[q.end];
      widest = j.width > widest ? j.width : widest;
      q.split = q.split && j.g->plan_off >= 0 && j.g->num_chunks <= kMaxBgmvRows;
    }
    q.fused = lorax_prefill_in_one_launch(g.rank, c.h_in, c.rows, widest) != 0;
    q.n_long = q.split ? g.num_long_segments : g.num_segments;
    q.planned = q.n_long == g.num_long_segments;
    if (!q.fused && q.n_long > 0)
      plans[num_plans++] = {g.rank, q.end - i, q.planned ? g.num_shrink_tiles : 0, q.planned ? g.shrink_tile_rows : 0};
  }
  const int stacked = lorax_shrink_summed_rank(plans, num_plans, c.rows, c.h_in);
  for (int q = 0; q < num_groups; ++q) {
    const auto [i, end, fused, split, n_long, planned] = group_of[q];
    const lorax_table_group_t& g = *jobs[i]->g;
    const int32_t* starts = static_cast<const int32_t*>(at(c, g.starts_off));
    const int32_t* ends = static_cast<const int32_t*>(at(c, g.ends_off));
    if (fused) {
      for (int k = i; k < end; k += lorax::kMaxSgmvLoraProblems) {
        lorax_sgmv_lora_problem_t p[lorax::kMaxSgmvLoraProblems];
        int n = 0;
        for (; n < lorax::kMaxSgmvLoraProblems && k + n < end; ++n) {
          const Job& j = *jobs[k + n];
          p[n] = {c.y, static_cast<const int64_t*>(at(c, j.g->a_ptr_off)), static_cast<const int64_t*>(at(c, j.g->b_ptr_off)),
                  j.y_offset, c.y_stride, j.width};
        }
        if (int rc = lorax_sgmv_lora_multi(p, n, c.x, starts, ends, g.num_segments, c.rows, c.h_in, g.rank, c.layer_idx,
                                           1.0f, c.dtype, c.stream))
          return rc;
      }
      continue;
    }
    // one shrink of up to four projections: of a short batch at any rank, else of a summed rank
    const int fit = stacked / g.rank > 0 ? stacked / g.rank : 1;
    const int step = c.rows <= kShortBatchRows || fit >= lorax::kMaxShrinkGroup ? lorax::kMaxShrinkGroup : fit;
    for (int k = i; k < end && n_long > 0; k += step) {
      lorax_sgmv_shrink_problem_t* p = problems[num_shrinks];
      int n = 0;
      for (; n < step && k + n < end; ++n)
        p[n] = {jobs[k + n]->v, static_cast<const int64_t*>(at(c, jobs[k + n]->g->a_ptr_off))};
      tiles[num_shrinks] = {static_cast<const lorax_sgmv_tile_t*>(at(c, g.shrink_tiles_off)), g.num_shrink_tiles,
                            g.shrink_tile_rows};
      shrinks[num_shrinks] = {p, n, g.rank, starts, ends, n_long, planned ? &tiles[num_shrinks] : nullptr};
      if (++num_shrinks == kShrinkBatch)
        if (int rc = flush_shrinks()) return rc;
    }
    for (int k = i; k < end; ++k) {
      if (n_long > 0) {
        expand_segments[num_expand] = n_long;
        expand[num_expand++] = jobs[k];
      }
      if (split) shorts[num_shorts++] = jobs[k];
    }
  }
  if (num_shrinks > 0)
    if (int rc = flush_shrinks()) return rc;
  for (int i = 0; i < num_shorts; i += lorax::kMaxBgmvProblems) {
    const int n = num_shorts - i < lorax::kMaxBgmvProblems ? num_shorts - i : lorax::kMaxBgmvProblems;
    if (int rc = bgmv_jobs(c, shorts + i, n, true)) return rc;
  }
  for (int i = 0; i < num_expand; i += lorax::kMaxExpandProblems) {
    lorax_sgmv_expand_problem_t p[lorax::kMaxExpandProblems];
    lorax_sgmv_tiles_t tiles_of[lorax::kMaxExpandProblems];
    int n = 0;
    for (; n < lorax::kMaxExpandProblems && i + n < num_expand; ++n) {
      const Job& j = *expand[i + n];
      const lorax_table_group_t& g = *j.g;
      tiles_of[n] = {static_cast<const lorax_sgmv_tile_t*>(at(c, g.expand_tiles_off)), g.num_expand_tiles, g.expand_tile_rows};
      p[n] = {c.y, j.v, static_cast<const int64_t*>(at(c, g.b_ptr_off)), static_cast<const int32_t*>(at(c, g.starts_off)),
              static_cast<const int32_t*>(at(c, g.ends_off)), expand_segments[i + n], g.rank, j.width, j.y_offset, c.y_stride,
              expand_segments[i + n] == g.num_long_segments ? &tiles_of[n] : nullptr};
    }
    if (int rc = lorax_sgmv_expand_multi(p, n, c.rows, c.layer_idx, 1, c.dtype, c.stream)) return rc;
  }
  for (int i = 0; i < num_shorts; i += lorax::kMaxBgmvProblems) {
    const int n = num_shorts - i < lorax::kMaxBgmvProblems ? num_shorts - i : lorax::kMaxBgmvProblems;
    if (int rc = bgmv_jobs(c, shorts + i, n, false)) return rc;
  }
  return LORAX_OK;
}

int update(const Call& c, const lorax_table_group_t* groups, int32_t num_groups, const lorax_layer_slice_t* slices,
           int32_t num_slices, char* v, int64_t v_bytes) {
  Job jobs[kMaxJobs];
  int count = 0;
  for (int s = 0; s < num_slices; ++s)
    for (int i = 0; i < num_groups; ++i) {
      const lorax_table_group_t& g = groups[i];
      if (g.layer_type != slices[s].layer_type) continue;
      if (count == kMaxJobs || g.rank < 8 || g.rank % 8 != 0 || g.rank > kMaxKernelRank) return LORAX_EROUTE;
      if (count > 0 && g.use_sgmv != jobs[0].g->use_sgmv) return LORAX_EROUTE;
      // shapes that only the reference's prefill layouts serve
      if (g.use_sgmv != 0 && g.rank % 16 != 0 && c.h_in % 128 != 0 && c.rows > kShortBatchRows) return LORAX_EROUTE;
      if (g.use_sgmv != 0 && (g.segments_id < 0 || g.shrink_tiles_off < 0 || g.expand_tiles_off < 0)) return LORAX_EROUTE;
      if (g.use_sgmv == 0 && g.plan_off < 0) return LORAX_EROUTE;
      jobs[count++] = {&g, slices[s].y_offset, slices[s].width, nullptr, nullptr, nullptr};
    }
  if (count == 0) return LORAX_OK;
  const bool by_segments = jobs[0].g->use_sgmv != 0;
  // Jobs in order of the first appearance of their rank (prefill: of their rank and segment tables).
  auto alike = [&](const Job& a, const Job& b) {
    return a.g->rank == b.g->rank && (!by_segments || a.g->segments_id == b.g->segments_id);
  };
  Job* order[kMaxJobs];
  bool taken[kMaxJobs] = {};
  int placed = 0;
  int64_t used = 0;
  for (int i = 0; i < count; ++i)
    for (int k = i; k < count && !taken[i]; ++k) {
      if (k == i) order[placed++] = &jobs[i];
      else if (!taken[k] && alike(jobs[i], jobs[k])) {
        taken[k] = true;
        order[placed++] = &jobs[k];
      }
    }
  for (int i = 0; i < count; ++i) {  // [num_tokens, rank] each; ranks are multiples of 8, so every piece is 16-byte aligned
    order[i]->v = v + used;
    used += c.rows * order[i]->g->rank * 2;
  }
  if (used > v_bytes) return lorax::report_error(LORAX_ESPACE, "layer update: the workspace is smaller than num_tokens * ranks");
  return by_segments ? prefill(c, order, count) : decode(c, order, count);
}

// Runs `launch` with `device` current.
template <typename Launch>
int on_device(int device, const Launch& launch) {
  int current = 0;
  if (hipError_t e = hipGetDevice(&current)) return lorax::report_error(LORAX_ELAUNCH, hipGetErrorString(e));
  if (current != device)
    if (hipError_t e = hipSetDevice(device)) return lorax::report_error(LORAX_ELAUNCH, hipGetErrorString(e));
  const int rc = launch();
  if (current != device) (void)hipSetDevice(current);
  return rc;
}

}  // namespace

// The single-launch update (lorax_bgmv_lora_multi) pays where the A slab is small and one workgroup covers a
// projection's columns (4096 at rank 8, 2048 at rank 16).  A wider projection is cut into slices that each repeat the
// shrink, and is faster as a shrink launch plus an expand launch - unless the batch has few routing records: then the
// repeated shrinks run on idle CUs and the second launch is what costs.  Measured at hidden sizes 1024 to 8192, 1 to 4
// tokens per record, fused against two launches in us: 2 x 14336 columns at rank 8 (hidden 4096) 4.3 and 6.1 at 1
// record, 9.9 and 11.0 at 32 of 4 tokens, 18.9 and 17.6 at 64 of 4 (512 slices for 256 CUs), 11.8 and 13.3 at 64 of 1;
// one of 14336 9.8 and 10.6 at 64 of 4 (256 slices); 8192 + 1024 + 1024 over 8192 at rank 8 13.0 and 13.7 at 64 of 4;
// 2 x 14336 at rank 16 (4096) 10.7 and 11.3 at 16 of 4, 19.6 and 17.0 at 32 of 4.  More slices than CUs pay only where
// the records hold about one token each and the slab is at most half the limit (14336 + 1024 over 8192, 64 of 1: 12.2
// and 11.2).
extern "C" int lorax_decode_in_one_launch(const lorax_decode_job_t* jobs, int32_t num_jobs, int64_t num_tokens, int32_t h_in) {
  if (num_jobs < 1 || jobs == nullptr) return 0;
  bool wide = false, few = true;
  int64_t slices = 0;
  const int few_records = jobs[0].rank == 8 ? 64 : 16;
  for (int i = 0; i < num_jobs; ++i) {
    const lorax_decode_job_t& j = jobs[i];
    if (!fused_rank(j.rank, h_in)) return 0;
    const int cols = 256 / (j.rank / 8) * 16;
    wide = wide || j.width > cols;
    few = few && j.rank == jobs[0].rank && j.records <= few_records && j.width <= kFusedWidthMax;
    slices += static_cast<int64_t>(j.records) * ((j.width + cols - 1) / cols);
  }
  if (!wide) return 1;
  return few && (slices <= kNumCus || (num_tokens <= few_records && jobs[0].rank * h_in * 2 <= kFusedSlab / 2));
}

// The single-launch update of a short prefill batch (lorax_sgmv_lora_multi) reads A again for every four rows: a
// Mistral-7B block of one run at rank 16 takes 49 us per layer in one launch per group and 51 in two at 128 rows, 61 and
// 54 at 192, 116 and 72 at 512; at rank 8 56 and 65 at 512.
extern "C" int lorax_prefill_in_one_launch(int32_t rank, int32_t h_in, int64_t num_tokens, int32_t widest) {
  return fused_rank(rank, h_in) && num_tokens <= (rank == 8 ? kShortBatchRows : kShortBatchRows16) && widest <= kFusedWidthMax;
}

// lorax_sgmv_shrink_groups takes several groups in one launch only if all of them come in tiles of up to 32 rows.  There a
// workgroup holds its group's A tile next to its rows of x: at a summed rank of 128 two stages of 36 KB fit where two
// workgroups share a CU, at 64 three of 20 KB, and the tiles of the high ranks are no longer the ones the launch waits for -
// unless one projection's rank is above 64, for which the launch waits as before.  Whole layers in one process, 514 to 7321
// rows in 8 to 300 runs, attention projections of hidden size 4096, gate/up and down, a 70B layer (time at 64 over that at
// 128, geometric mean and range): ranks 8 to 64 0.93, 0.96 and 0.97 (0.86 to 1.00), 32 and 64 0.95, 0.97 and 0.97 (0.88 to
// 1.02), 16 and 32 0.98, 1.00 and 1.00 (0.91 to 1.05), 64 alone 0.95 and 0.99 (0.87 to 1.07: 3017 rows in tiles of 16 make
// a third round where two groups of 128 end with the second), 32 and 128 1.04, 1.00 and 1.01 (0.94 to 1.19).
// One group of up to 128 stays whole (q, k and v of 2009 rows at rank 32 in one group 56 us a layer, in two 64).
extern "C" int lorax_shrink_summed_rank(const lorax_shrink_plan_t* groups, int32_t num_groups, int64_t num_tokens, int32_t h_in) {
  if (num_groups < 1 || groups == nullptr || num_tokens <= kShortBatchRows || h_in % 128 != 0) return kMaxKernelRank;
  int calls = 0;
  for (int i = 0; i < num_groups; ++i) {
    const lorax_shrink_plan_t& g = groups[i];
    if (g.rank < 1 || g.rank > kGroupedRank || g.num_tiles < 1 || g.tile_rows > kGroupedTileRows) return kMaxKernelRank;
    const int fit = kGroupedRank / g.rank < lorax::kMaxShrinkGroup ? kGroupedRank / g.rank : lorax::kMaxShrinkGroup;
    calls += (g.num_problems + fit - 1) / fit;
  }
  const bool alone = num_groups == 1 && groups[0].num_problems * groups[0].rank <= kMaxKernelRank;
  return alone || calls > kShrinkBatch ? kMaxKernelRank : kGroupedRank;
}

extern "C" int lorax_layer_update(const lorax_table_group_t* groups, int32_t num_groups, const void* tables,
                                  const lorax_layer_slice_t* slices, int32_t num_slices, void* y, int64_t y_stride,
                                  const void* x, int64_t num_tokens, int32_t h_in, int64_t layer_idx, void* v, int64_t v_bytes,
                                  void* tmp, int64_t tmp_bytes, int32_t dtype, int32_t device, void* stream) {
  if (num_groups < 0 || num_slices < 0 || num_tokens < 0)
    return lorax::report_error(LORAX_EINVAL, "layer update: negative size");
  if (num_groups == 0 || num_slices == 0 || num_tokens == 0) return LORAX_OK;
  if (groups == nullptr || tables == nullptr || slices == nullptr || y == nullptr || x == nullptr || v == nullptr)
    return lorax::report_error(LORAX_EINVAL, "null pointer argument (groups, tables, slices, y, x or v)");
  // The segment kernels clamp their rows to num_tokens; the per-token kernels take them from the plan's records.
  int widest = 0;
  for (int s = 0; s < num_slices; ++s) widest = slices[s].width > widest ? slices[s].width : widest;
  for (int s = 0; s < num_slices; ++s)
    for (int i = 0; i < num_groups; ++i) {
      const lorax_table_group_t& g = groups[i];
      if (g.layer_type != slices[s].layer_type || g.plan_off < 0 || num_tokens >= g.num_tokens) continue;
      if (g.use_sgmv == 0 || !lorax_prefill_in_one_launch(g.rank, h_in, num_tokens, widest))
        return lorax::report_error(LORAX_EINVAL, "layer update: x and y have fewer rows than the batch of the routing tables");
    }
  const Call c{static_cast<const char*>(tables), y, y_stride, x, num_tokens, h_in, layer_idx, tmp, tmp_bytes, dtype, stream};
  return on_device(device, [&] { return update(c, groups, num_groups, slices, num_slices, static_cast<char*>(v), v_bytes); });
}

extern "C" int lorax_stacked_update(const lorax_stacked_slice_t* slices, int32_t num_slices, const int64_t* plan, int32_t records,
                                    void* y, int64_t y_stride, const void* x, int64_t num_tokens, int32_t h_in, void* v,
                                    int64_t v_bytes, int32_t dtype, int32_t device, void* stream) {
  if (num_slices < 0 || num_slices > lorax::kMaxBgmvProblems || num_tokens < 0 || records < 0)
    return lorax::report_error(LORAX_EINVAL, "stacked update: number of slices (at most 16), rows or plan records out of range");
  if (num_slices == 0 || num_tokens == 0) return LORAX_OK;
  if (slices == nullptr || plan == nullptr || y == nullptr || x == nullptr || v == nullptr)
    return lorax::report_error(LORAX_EINVAL, "null pointer argument (slices, plan, y, x or v)");
  lorax_table_group_t groups[lorax::kMaxBgmvProblems];
  Job jobs[lorax::kMaxBgmvProblems];
  Job* order[lorax::kMaxBgmvProblems];
  int64_t used = 0;
  for (int i = 0; i < num_slices; ++i) {
    const lorax_stacked_slice_t& s = slices[i];
    if (s.rank < 8 || s.rank % 8 != 0 || s.rank > kMaxKernelRank || s.a_stack == nullptr || s.b_stack == nullptr) return LORAX_EROUTE;
    groups[i] = lorax_table_group_t{};
    groups[i].rank = s.rank;
    groups[i].num_chunks = records;
    jobs[i] = {&groups[i], s.y_offset, s.width, static_cast<char*>(v) + used, s.a_stack, s.b_stack};
    order[i] = &jobs[i];
    used += num_tokens * s.rank * 2;
  }
  if (used > v_bytes) return lorax::report_error(LORAX_ESPACE, "stacked update: the workspace is smaller than num_tokens * ranks");
  const Call c{reinterpret_cast<const char*>(plan), y, y_stride, x, num_tokens, h_in, 0, nullptr, 0, dtype, stream};
  // (a batch of base-model tokens only: nothing is launched, but its operands are checked like any other's)
  if (records == 0) return decode(c, order, num_slices);
  return on_device(device, [&] { return decode(c, order, num_slices); });
}
