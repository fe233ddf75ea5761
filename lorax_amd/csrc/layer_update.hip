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
constexpr int kFewChunks8 = 64, kFewChunks16 = 16;  // plan records up to which wide projections run fused, by rank
constexpr int64_t kShortBatchRows16 = 128;  // ... and of the latter at rank 16 (measured: _native.sgmv_lora_fits)

struct Job {
  const lorax_table_group_t* g;
  int64_t y_offset;
  int32_t width;
  char* v;  // [num_tokens, rank] piece of the workspace
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

// The single-launch update pays where the A slab is small and, in decode, one workgroup covers the projection's
// columns or the batch has few records (the rules of _native.bgmv_lora_fits and sgmv_lora_fits, where they are explained).
bool fused_rank(int r, int h_in) { return (r == 8 || r == 16) && r * h_in * 2 <= 128 * 1024; }
bool decode_fused(const Job& j, int h_in, bool one_rank) {
  const int r = j.g->rank;
  return fused_rank(r, h_in) && (j.width <= (256 / (r / 8)) * 16 ||
                                 (one_rank && j.width <= 16384 && j.g->num_chunks <= (r == 8 ? kFewChunks8 : kFewChunks16)));
}

// A short prefill batch runs shrink and expand of a rank's projections in one launch over the segments.
bool prefill_fused(int r, int h_in, int64_t rows, int widest) {
  return fused_rank(r, h_in) && rows <= (r == 8 ? kShortBatchRows : kShortBatchRows16) && widest <= 16384;
}

const void* at(const Call& c, int64_t off) { return c.tables + off; }

lorax_bgmv_problem_t plan_problem(const Call& c, const Job& j, void* y, const void* x, int64_t y_offset, int64_t y_stride,
                                  int32_t h_out, int32_t h_in) {
  return {y, x, nullptr, nullptr, y_offset, y_stride, h_out, static_cast<const int64_t*>(at(c, j.g->plan_off)),
          j.g->num_chunks, h_in, nullptr, nullptr};
}

// One planned launch for up to 16 jobs: x -> v (shrink) or v -> y (expand).
int bgmv_jobs(const Call& c, const Job* const* jobs, int count, bool shrink) {
  lorax_bgmv_problem_t p[lorax::kMaxBgmvProblems];
  for (int i = 0; i < count; ++i) {
    const Job& j = *jobs[i];
    const int r = j.g->rank;
    p[i] = shrink ? plan_problem(c, j, j.v, c.x, 0, r, r, c.h_in)
                  : plan_problem(c, j, c.y, j.v, j.y_offset, c.y_stride, j.width, r);
  }
  return lorax_bgmv_multi(p, count, c.rows, shrink ? c.h_in : p[0].h_in, c.layer_idx, 1.0f, shrink ? 0 : 1, c.dtype, c.stream);
}

int decode(const Call& c, Job* const* jobs, int count) {
  bool fused = true;
  bool one_rank = true;
  for (int i = 0; i < count; ++i) one_rank = one_rank && jobs[i]->g->rank == jobs[0]->g->rank;
  for (int i = 0; i < count; ++i) fused = fused && decode_fused(*jobs[i], c.h_in, one_rank);
  if (fused) {
    for (int r : {8, 16}) {
      lorax_bgmv_problem_t p[lorax::kMaxFusedBgmvProblems];
      int n = 0;
      for (int i = 0; i <= count; ++i) {
        if (n > 0 && (i == count || n == lorax::kMaxFusedBgmvProblems)) {
          if (int rc = lorax_bgmv_lora_multi(p, n, c.rows, c.h_in, r, c.layer_idx, 1.0f, c.dtype, c.stream)) return rc;
          n = 0;
        }
        if (i < count && jobs[i]->g->rank == r)
          p[n++] = plan_problem(c, *jobs[i], c.y, c.x, jobs[i]->y_offset, c.y_stride, jobs[i]->width, 0);
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
  constexpr int kShrinkBatch = 16;
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
  // `jobs` is ordered by group of equal rank and segment tables
  for (int i = 0, end = 0; i < count; i = end) {
    const lorax_table_group_t& g = *jobs[i]->g;
    int widest = 0;
    for (end = i; end < count && jobs[end]->g->rank == g.rank && jobs[end]->g->segments_id == g.segments_id; ++end)
      widest = jobs[end]->width > widest ? jobs[end]->width : widest;
    const int32_t* starts = static_cast<const int32_t*>(at(c, g.starts_off));
    const int32_t* ends = static_cast<const int32_t*>(at(c, g.ends_off));
    if (prefill_fused(g.rank, c.h_in, c.rows, widest)) {
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
    // segments of a few rows go to the per-token kernels where every projection has a plan over them
    bool split = c.rows <= kMaxBgmvRows;
    for (int k = i; k < end; ++k) split = split && jobs[k]->g->plan_off >= 0 && jobs[k]->g->num_chunks <= kMaxBgmvRows;
    const int32_t n_long = split ? g.num_long_segments : g.num_segments;
    const bool planned = n_long == g.num_long_segments;  // the tables' row-tile plans cover these segments
    // one shrink launch for up to four projections: of a short batch at any rank, else of a summed rank of 128
    const int step = c.rows <= kShortBatchRows || kMaxKernelRank / g.rank >= lorax::kMaxShrinkGroup ? lorax::kMaxShrinkGroup
                                                                                                   : kMaxKernelRank / g.rank;
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
      jobs[count++] = {&g, slices[s].y_offset, slices[s].width, nullptr};
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

}  // namespace

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
      if (g.use_sgmv == 0 || !prefill_fused(g.rank, h_in, num_tokens, widest))
        return lorax::report_error(LORAX_EINVAL, "layer update: x and y have fewer rows than the batch of the routing tables");
    }
  const Call c{static_cast<const char*>(tables), y, y_stride, x, num_tokens, h_in, layer_idx, tmp, tmp_bytes, dtype, stream};
  int current = 0;
  if (hipError_t e = hipGetDevice(&current)) return lorax::report_error(LORAX_ELAUNCH, hipGetErrorString(e));
  if (current != device)
    if (hipError_t e = hipSetDevice(device)) return lorax::report_error(LORAX_ELAUNCH, hipGetErrorString(e));
  const int rc = update(c, groups, num_groups, slices, num_slices, static_cast<char*>(v), v_bytes);
  if (current != device) (void)hipSetDevice(current);
  return rc;
}
