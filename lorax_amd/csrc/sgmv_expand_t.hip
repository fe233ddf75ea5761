// SGMV expand over the transposed B stack: y[s:e, off:off+h_out] += T(v[s:e, :r] @ B_i), with B_i
// stored as B_i^T = [h_out, r] (the layout the decode path keeps resident anyway).
//
// Same arithmetic and rounding as sgmv_expand.hip.  The MFMA product is v (16 rows of a block, first
// operand) times B (second operand), and with B^T in memory the second operand needs no transposition:
// the 16 bytes B^T[column(j, c)][32 s + 8 g ...] that lane (c, g) of accumulator j needs come straight from
// global memory into registers (fetched by the lane that makes the access contiguous and handed over with
// a cross-lane move, see the kernel).  There is no LDS staging, no barrier and no LDS gather in a tile's
// prologue - which, for the short segments a prefill batch is full of, took longer than the rows
// themselves.
//
// The columns of a wave's panel are dealt to the accumulators so that a lane ends up with NJ ADJACENT
// columns of four rows (see the kernel).  A y access of the wave is then four whole runs of 32 * NJ
// bytes, one per row, and the texture path handles it as a few cache lines.  (With the product the other
// way round - B^T first, v second - a lane holds 8 adjacent columns of ONE row and neighbouring lanes
// hold different rows: every 16-byte piece is then a separate cache-line lookup, 64 per instruction, and
// the kernel is bound by the address path of the CU at 60 % of what it reaches now; counters:
// TA_ADDR_STALLED_BY_TC_CYCLES at 60 % and TA_BUSY at 80 % of the kernel's duration.)
//
// Work split: a workgroup owns one row tile - or `sub_rows` rows of one - and 4 column panels of 16 * NJ; wave w takes
// panel w and walks ALL 16-row blocks of its rows.  The tile search runs once per workgroup.  There is no separate
// path for segments of a few rows: rows past the tile's end are clamped for loads and predicated for stores, and
// MFMA work on padding is free in a kernel that waits on memory.
//
// One launch serves up to 16 problems - the projections of a layer that share their input, of every LoRA rank in the
// batch: a problem owns a run of workgroup numbers and the workgroup picks the body for its problem's rank.  Apart,
// they are launches of a few dozen workgroups each (1024 columns x 800 rows: 40 workgroups, 14 us; q, k and v of a
// thousand-row batch 15 + 14 + 14 us), and a batch whose adapters have four ranks issues four times as many.
#include "kernels.h"
#include "sgmv_tile_plan.h"
#include "sgmv_tiles.h"

namespace lorax {

constexpr int kExpTWaves = 4;
constexpr int kExpTThreads = kExpTWaves * kWave;
constexpr int kExpTStages = 2;  // register stages of the row-block pipeline (a third one costs occupancy)
constexpr int kExpTLaneCols = 4;  // adjacent output columns per lane
constexpr int kExpandFill = 1024;  // workgroups below which a launch gets lower pieces

// What a workgroup has to know about its problem.
struct ExpandSlot {
  const void* v;
  void* y;
  const int64_t* w_ptrs;
  const int32_t* s_start;
  const int32_t* s_end;
  const int32_t* tiles;  // the caller's plan, or null
  int64_t y_offset;
  int64_t y_stride;
  int num_segments;
  int r;
  int h_out;
  int num_tiles;   // records of the plan
  int tile_rows;   // no record of the plan is taken higher; without a plan the height the search cuts
  int tile_slots;  // row tiles counted for the grid
  int subs;        // pieces of sub_rows rows a tile is cut into; the last one takes what is left
};
template <int MAX>
struct ExpandLaunch {
  ExpandSlot p[MAX];
  int wg_end[MAX];  // problem i owns the workgroups [wg_end[i - 1], wg_end[i])
};

// NJ accumulators per wave, a panel of 16 * NJ output columns.  Accumulator j stands for the columns
// n0 + NJ * c + j (c = lane & 15), so a lane ends up with NJ ADJACENT columns of the rows 4g .. 4g + 3
// (g = lane >> 4) of a 16-row block, and the 16 lanes of one g cover 32 * NJ contiguous bytes of a row.
template <typename D, int KS, int NJ>
__device__ __forceinline__ void expand_tile(const ExpandSlot& P, const typename D::E* BT, const RowTile& rt, int panel,
                                            bool acc_y) {
  using E = typename D::E;
  using vec8 = typename D::vec8;
  typedef E yvec __attribute__((ext_vector_type(NJ)));
  constexpr int kCols = 16 * NJ;
  const int lane = threadIdx.x & (kWave - 1);
  const int c = lane & 15;
  const int g = lane >> 4;
  const int r = P.r, h_out = P.h_out;

  // MFMA operand layout: lane g * 16 + c holds the eight k values 32 s + 8 g ... of operand row / column c.
  // Fetched that way, neighbouring lanes read different rows, r * 2 bytes apart, and every 16-byte piece
  // is a cache-line lookup of its own.  So the operands are FETCHED with lane l taking piece l & 3 of row
  // l >> 2 - a quad of lanes reads 64 contiguous bytes - and then change lanes through the LDS crossbar
  // (ds_bpermute, no LDS memory): the lane g * 16 + c takes the registers of lane 4 c + g.
  const int lc = lane >> 2;
  const int from_lane = (c * 4 + g) * 4;  // ds_bpermute addresses lanes in bytes
  auto to_operand_lanes = [&](vec8 fetched) {
    const u32x4 raw = __builtin_bit_cast(u32x4, fetched);
    u32x4 mine;
#pragma unroll
    for (int d = 0; d < 4; ++d)
      mine[d] = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(from_lane, static_cast<int>(raw[d])));
    return __builtin_bit_cast(vec8, mine);
  };
  bool k_ok[KS];  // of the operand lane: chunks beyond the rank are zeroed after the exchange
  int l_off[KS];  // of the fetching lane: chunks beyond the rank are fetched from chunk 0
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    k_ok[s] = s * 32 + g * 8 < r;
    l_off[s] = s * 32 + (lane & 3) * 8 < r ? s * 32 + (lane & 3) * 8 : 0;
  }
  const int nmb = (rt.row_end - rt.row0 + 15) / 16;
  const int n0 = panel * kCols;
  // h_out is a multiple of 8 and so is NJ * c: a lane's NJ columns are inside the matrix or outside it
  // as a whole.  Loads are unconditional: rows past the tile are clamped to its last row and a lane
  // past h_out reads the panel's first columns (both valid memory); only the stores are predicated.
  const bool col_ok = n0 + NJ * c < h_out;
  const int col = col_ok ? n0 + NJ * c : n0;
  // Addresses inside a tile: a wave-uniform 64-bit base and a 32-bit offset per lane (a tile spans at
  // most tile_rows * y_stride elements).
  const E* vtile = static_cast<const E*>(P.v) + static_cast<int64_t>(rt.row0) * r;
  E* ytile = static_cast<E*>(P.y) + static_cast<int64_t>(rt.row0) * P.y_stride + P.y_offset + n0;
  const uint32_t ycol = static_cast<uint32_t>(col - n0);
  const uint32_t ystride = static_cast<uint32_t>(P.y_stride);
  const int last = rt.row_end - rt.row0 - 1;
  auto load_block = [&](int mb, vec8(&vf)[KS], yvec(&yv)[4]) {
    // v rows are fetched like the B^T rows below: lane l takes piece l & 3 of row l >> 2 of the block, and
    // finish_block moves the pieces to the lanes the MFMA wants them in
    const uint32_t voff = static_cast<uint32_t>(min(mb * 16 + lc, last)) * static_cast<uint32_t>(r);
#pragma unroll
    for (int s = 0; s < KS; ++s) vf[s] = load8<D>(vtile + (voff + l_off[s]));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t row = static_cast<uint32_t>(min(mb * 16 + g * 4 + i, last));
      yv[i] = *(const LORAX_GLOBAL yvec*)(ytile + (row * ystride + ycol));
    }
  };
  auto block_of = [&](int i) { return min(i, nmb - 1); };

  // first row blocks and the panel's operands go out together: one memory round trip
  vec8 vr[kExpTStages][KS];
  yvec yr[kExpTStages][4];
#pragma unroll
  for (int s = 0; s < kExpTStages - 1; ++s) load_block(block_of(s), vr[s], yr[s]);
  // B^T operands: lane l fetches piece l & 3 of the row of operand column l >> 2
  vec8 bf[NJ][KS];
  const int lcol = (n0 + NJ * lc < h_out) ? n0 + NJ * lc : n0;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
#pragma unroll
    for (int s = 0; s < KS; ++s)
      bf[j][s] = keep_if<D>(k_ok[s], to_operand_lanes(load8<D>(BT + static_cast<int64_t>(lcol + j) * r + l_off[s])));
  }

  auto finish_block = [&](bool live, int mb, vec8(&vf)[KS], yvec(&yv)[4]) {
    f32x4 acc[NJ];
#pragma unroll
    for (int s = 0; s < KS; ++s) vf[s] = to_operand_lanes(vf[s]);
    if (r < KS * 32) {  // uniform; chunks beyond the rank hold chunk 0: an infinity there times B's zeros would be NaN
#pragma unroll
      for (int s = 0; s < KS; ++s) vf[s] = keep_if<D>(k_ok[s], vf[s]);
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) acc[j] = D::mfma16(vf[s], bf[j][s], acc[j]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = mb * 16 + g * 4 + i;
      yvec out;
#pragma unroll
      for (int j = 0; j < NJ; ++j)  // overwrite mode: the old y counts as zero
        out[j] = accumulate<D>(acc_y ? yv[i][j] : static_cast<E>(0.0f), acc[j][i]);
      if (live && col_ok && row <= last)
        *(LORAX_GLOBAL yvec*)(ytile + (static_cast<uint32_t>(row) * ystride + ycol)) = out;
    }
  };

  // Ring of kExpTStages register stages with static indices: the y and v loads of the next
  // kExpTStages - 1 blocks are in flight while one block is multiplied and stored.  Surplus
  // trips of the last round re-load the last block and store nothing.
  for (int i = 0; i < nmb; i += kExpTStages) {
#pragma unroll
    for (int s = 0; s < kExpTStages; ++s) {
      constexpr int kAhead = kExpTStages - 1;
      load_block(block_of(i + s + kAhead), vr[(s + kAhead) % kExpTStages], yr[(s + kAhead) % kExpTStages]);
      __builtin_amdgcn_sched_barrier(0);
      finish_block(i + s < nmb, block_of(i + s), vr[s], yr[s]);
    }
  }
}

// KS: 32-wide k steps of the largest rank in the launch; MIXED: the problems' ranks differ in it.
// MAX: problems the arguments hold (kFewProblems or all).
// Registers: launches of several ranks are held to 128 (ranks up to 64: four waves per SIMD) and 168 (rank 128: three).  The
// bodies take a few more by themselves, and the short tiles of such batches, mostly waiting for their first loads, gain from
// the wave: GPU time of two Mistral-7B layers of 2062 rows at ranks 8 to 64 444 -> 425 us, of a gate/up and down block of
// 2741 rows at ranks 32 and 128 207 -> 199.  One rank alone is left as it is: at rank 64 four waves gain 1-3 % in attention
// projections and lose 1 % in large launches (a 70B layer of 4573 rows 591 -> 598 us), at rank 128 three spill (748 -> 782).
template <typename D, int KS, int NJ, bool MIXED, int MAX>
__global__ __launch_bounds__(kExpTThreads, MIXED ? (KS == 2 ? 4 : 3) : 1) void sgmv_expand_t_kernel(const ExpandLaunch<MAX> batch, int count, int num_tokens,
                                                                    int64_t layer_idx, int accumulate_into_y,
                                                                    int sub_rows) {
  using E = typename D::E;
  constexpr int kCols = 16 * NJ;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);  // wave-uniform, in a scalar register
  // Workgroup numbering: problem by problem, inside one piece by piece, panel groups fastest, and the numbers go round
  // robin over the XCDs as the hardware deals them: every XCD gets the same share of every problem and of every segment,
  // and the long segments, which the table builder lists first, start first.  (Numbered so that each XCD owned a run of
  // one problem's panel groups, a batch whose segments differ waited for the XCD with the most rows: 28672 columns x
  // 2062 rows of ranks 8 to 64 111 us, dealt out 68; 786 rows of rank 64 42 and 32 us.)  A panel group has one XCD,
  // where all pieces of a segment find its panel of B^T in the L2, wherever the number of groups is a multiple of the
  // XCDs; an XCD then takes adjacent groups (15136 rows: 624 -> 615 us for a step of the large prefill).  Elsewhere every XCD
  // fetches every panel, in about the same time: 27 groups x 9126 rows of rank 64 162 -> 185 MB, 61.8 -> 59.1 us, 27 x 4096 of
  // rank 128 71 -> 91 MB, 31.4 -> 32.4 us; with 56 groups (10658 rows, rank 64) 433 -> 377 MB.
  int vid = static_cast<int>(blockIdx.x);
  int prob = 0;
  if (count > 1) {  // lane i looks at problem i's range: one trip to the kernel arguments
    const int end = batch.wg_end[lane < MAX ? lane : MAX - 1];
    prob = __popcll(__ballot(lane + 1 < count && vid >= end));
    if (prob > 0) vid -= read_lane(end, prob - 1);
  }
  const ExpandSlot& P = batch.p[prob];
  const bool acc_y = accumulate_into_y != 0;
  const int groups = (P.h_out + kCols * kExpTWaves - 1) / (kCols * kExpTWaves);
  const int piece = vid / groups;
  int group = vid - piece * groups;
  constexpr int kXcdCount = static_cast<int>(kXcds);
  if (groups % kXcdCount == 0) group = group % kXcdCount * (groups / kXcdCount) + group / kXcdCount;
  const int panel = group * kExpTWaves + wave;
  const int sub = piece % P.subs;
  const TileList plan{P.tiles, P.num_tiles, P.tile_rows};
  const int64_t pre_w = preload_segment_entry(P.w_ptrs, P.num_segments);
  for (int tile = piece / P.subs;; tile += P.tile_slots) {
    RowTile rt;
    // small remainders are merged into the segment's other tiles: a tile's prologue (the search and the panel
    // operands) costs as much as a hundred rows
    if (!get_row_tile<true>(plan, P.s_start, P.s_end, P.num_segments, num_tokens, P.tile_rows, tile, rt)) break;
    const int64_t stack = segment_entry(pre_w, P.w_ptrs, rt.seg);
    if (P.tiles != nullptr && stack == 0) break;  // a caller's plan that names a segment without a stack
    if (P.subs > 1) {
      rt.row0 += sub * sub_rows;
      if (sub + 1 < P.subs) rt.row_end = min(rt.row_end, rt.row0 + sub_rows);
      if (rt.row0 >= rt.row_end) continue;
    }
    if (panel * kCols >= P.h_out) break;
    const E* BT = reinterpret_cast<const E*>(stack) + layer_idx * P.h_out * static_cast<int64_t>(P.r);
    if constexpr (MIXED) {
      if (P.r <= 32) expand_tile<D, 1, NJ>(P, BT, rt, panel, acc_y);
      else if (KS == 2 || P.r <= 64) expand_tile<D, 2, NJ>(P, BT, rt, panel, acc_y);
      else expand_tile<D, 4, NJ>(P, BT, rt, panel, acc_y);
    } else {
      expand_tile<D, KS, NJ>(P, BT, rt, panel, acc_y);
    }
  }
}

template <typename D, int KS, bool MIXED, int MAX>
static hipError_t launch_expand_t_max(const ExpandArgs& a, hipStream_t stream) {
  constexpr int kCols = 16 * kExpTLaneCols;
  ExpandLaunch<MAX> b{};
  // The kernel addresses a tile with 32-bit element offsets, and without a plan a tile is up to 9/8 of the searched
  // height + 15 rows high (merged remainders): rows of more than 2^23 elements get lower tiles.
  auto fits = [](int64_t rows, int64_t stride) { return stride * rows < (1ll << 32); };
  int64_t panel_groups[kMaxExpandProblems];
  int height[kMaxExpandProblems];  // of the problem's tallest tile
  for (int i = 0; i < a.count; ++i) {
    const ExpandProblem& q = a.p[i];
    ExpandSlot& s = b.p[i];
    s = ExpandSlot{q.v, q.y, q.w_ptrs, q.s_start, q.s_end, nullptr, q.y_offset, q.y_stride, q.num_segments, q.r, q.h_out,
                   0, 0, 0, 1};
    // With the caller's tile plan the tile count is exact (no workgroup without work); the plan is ignored when its
    // tiles would overflow the 32-bit offsets.
    if (q.tiles != nullptr && q.num_tiles > 0 && q.tile_rows >= 1 && tuning().expand_rows == 0 && fits(q.tile_rows, q.y_stride)) {
      s.tiles = q.tiles;
      s.num_tiles = s.tile_slots = q.num_tiles;
      // The pieces are counted for the plan's own height, but its records may be rewritten between the replays of a
      // captured launch: one that is higher (to the highest the planner cuts) is walked to its end by its last piece.
      height[i] = q.tile_rows;
      s.tile_rows = q.tile_rows < kExpandTileRowsMax && fits(kExpandTileRowsMax, q.y_stride) ? kExpandTileRowsMax : q.tile_rows;
    } else {
      int rows = tuning().expand_rows > 0 ? (tuning().expand_rows + 15) / 16 * 16 : kExpandTileRows;
      while (rows > 16 && !fits(rows + rows / 8 + 16, q.y_stride)) rows /= 2;
      height[i] = rows + rows / 8 + 16;
      if (!fits(height[i], q.y_stride)) return hipErrorInvalidValue;
      s.tile_rows = rows;
      const int64_t tiles = (a.num_tokens + rows - 1) / rows + q.num_segments;
      s.tile_slots = static_cast<int>(tiles < 65535 ? tiles : 65535);
    }
    panel_groups[i] = (q.h_out + kCols * kExpTWaves - 1) / (kCols * kExpTWaves);
  }
  // Rows per workgroup.  A wave takes its 16-row blocks one after the other, about half a microsecond each, so a
  // launch of fewer workgroups than the chip holds at once is as long as its tallest tile: such launches get lower
  // pieces, which fetch their panel of B^T (r / 128 of the bytes of the y rows of 64-row pieces) once per piece.
  auto workgroups = [&](int rows) {
    int64_t n = 0;
    for (int i = 0; i < a.count; ++i)
      n += panel_groups[i] * b.p[i].tile_slots * ((height[i] + rows - 1) / rows);
    return n;
  };
  int sub_rows = 1 << 20;
  for (int rows : {128, 64, 32}) {
    if (workgroups(sub_rows) >= kExpandFill) break;
    sub_rows = rows;
  }
  if (tuning().expand_sub > 0) sub_rows = (tuning().expand_sub + 15) / 16 * 16;
  int64_t total = 0;
  for (int i = 0; i < a.count; ++i) {
    ExpandSlot& s = b.p[i];
    s.subs = (height[i] + sub_rows - 1) / sub_rows;
    total += panel_groups[i] * s.tile_slots * s.subs;
    if (total >= INT32_MAX) return hipErrorInvalidValue;
    b.wg_end[i] = static_cast<int>(total);
  }
  if (total == 0) return hipSuccess;
  hipLaunchKernelGGL((sgmv_expand_t_kernel<D, KS, kExpTLaneCols, MIXED, MAX>), dim3(static_cast<unsigned>(total)),
                     dim3(kExpTThreads), 0, stream, b, a.count, static_cast<int>(a.num_tokens), a.layer_idx, a.accumulate,
                     sub_rows);
  return hipGetLastError();
}

template <typename D, int KS, bool MIXED>
static hipError_t launch_expand_t_ks(const ExpandArgs& a, hipStream_t stream) {
  return a.count <= kFewProblems ? launch_expand_t_max<D, KS, MIXED, kFewProblems>(a, stream)
                                 : launch_expand_t_max<D, KS, MIXED, kMaxExpandProblems>(a, stream);
}

template <typename D>
static hipError_t launch_expand_t_dtype(const ExpandArgs& a, hipStream_t stream) {
  int lo = 4, hi = 1;
  for (int i = 0; i < a.count; ++i) {
    const int ks = (a.p[i].r + 31) / 32;
    lo = ks < lo ? ks : lo;
    hi = ks > hi ? ks : hi;
  }
  if (lo != hi) return hi <= 2 ? launch_expand_t_ks<D, 2, true>(a, stream) : launch_expand_t_ks<D, 4, true>(a, stream);
  switch (hi) {
    case 1:
      return launch_expand_t_ks<D, 1, false>(a, stream);
    case 2:
      return launch_expand_t_ks<D, 2, false>(a, stream);
    case 3:
      return launch_expand_t_ks<D, 3, false>(a, stream);
    default:
      return launch_expand_t_ks<D, 4, false>(a, stream);
  }
}

hipError_t launch_sgmv_expand_t(const ExpandArgs& a, hipStream_t stream) {
  return a.dtype == LORAX_F16 ? launch_expand_t_dtype<F16>(a, stream) : launch_expand_t_dtype<BF16>(a, stream);
}

}  // namespace lorax
