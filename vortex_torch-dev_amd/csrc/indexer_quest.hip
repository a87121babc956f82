// Fused indexer step of the Quest flow for gfx950: the envelope score of
// every middle page for each of the G query heads, the maximum over the query
// heads and the top-k select — one launch, one workgroup per segment
// (request, kv head).
//
// For a block table built by the decode planner, at every middle page p of a
// segment s with more than topk of them, with e = dense[p]:
//   sum[p, g]  = bf16(sum_d max(bf16(q[s*G+g, d] * ymax[e, d]),
//                               bf16(q[s*G+g, d] * ymin[e, d])))
//   aggr[p]    = max_g sum[p, g]
//   sparse[sparse_indptr[s] + bos + i] = the i-th best page by aggr
// exactly what Multiply (twice), Maximum, Sum(dim=2), Max(dim=1) and topK
// write when launched one by one: the row sums use the shared Quest pass
// (vtx_score.h), whose per-lane column order and xor tree are the row-sum
// kernel's.  The [pages, G, D] products and their maximum are not written.
#include "vtx_cmean.h"
#include "vtx_device.h"
#include "vtx_fused_schedule.h"
#include "vtx_host.h"
#include "vtx_score.h"
#include "vtx_select.h"

namespace {

struct QuestArgs {
  const uint16_t* q;     // [segments * G, D]
  const uint16_t* ymax;  // [y_rows, D]
  const uint16_t* ymin;  // [y_rows, D]
  int64_t y_rows;
  uint16_t* sum;         // [sum_rows, G, 1]
  int64_t sum_rows;
  uint16_t* aggr;        // [aggr_len]
  int64_t aggr_len;
  const int32_t* dindptr;
  const int32_t* sindptr;
  const int32_t* didx;
  int64_t didx_len;
  int32_t* sidx;
  int64_t sidx_len;
  int32_t segments, G, dim, topk, bos, eos, row_cap;
  const int32_t* sched;  // the planner's workgroup schedule, or null (passed to the kernel up front)
};

// Quest score of one envelope (mx, mn: the lane's 16-byte column vector of
// each) for the lane's query slice: the lane's partial in column order and
// the xor tree over the LPR lanes, as quest_pass_multi computes it.
template <int LPR>
__device__ __forceinline__ float quest_vec(const vtx::U4& mx, const vtx::U4& mn, const float (&xs)[8]) {
  float s = vtx::quest_add(mx, mn, xs, 0.f);
#pragma unroll
  for (int d = LPR / 2; d >= 1; d >>= 1) s += vtx::xshfl(s, d);
  return s;
}

// kCmRegs > 0: the launch also runs the layer's CMax + CMin into the envelope
// pools (loc: up to 64 * kCmRegs entries, rows of one vector per lane), as
// the block-sparse fused kernel runs its CMean (vtx_cmean.h); its tiles go to
// the workgroups that finish first, after their own select.
//
// The planner's workgroup schedule (sched), the leading preloaded arguments
// and the check of the predicted bounds (before anything is written) work as
// in the GQA kernel (indexer_gqa.hip).
template <int T, int LPR, int VPL, int kG, int kCmRegs>
__global__ __launch_bounds__(T, (VPL == 1 ? 4 : (VPL <= 4 ? 2 : 1))) void quest_fused_kernel(
    const int32_t* sched, const int64_t* loc, int32_t segments, int32_t loc_n, QuestArgs a, vtx::CmArgs cma) {
  constexpr int kWaves = T / vtx::kWave;
  constexpr int kRowsPerLoad = vtx::kWave / LPR;
  // Two rows per position: half the GeMM's pass keeps the loads of a pass in
  // registers (a quarter with the in-launch page reduce, whose code would
  // otherwise push the pass past 128 registers).  The pass size does not
  // change the sums (each is the xor tree of its LPR lanes' partials
  // whatever the slot layout).
  constexpr int kPass = (VPL == 1 && kCmRegs == 0) ? 32 : 16;
  constexpr bool cm_on = kCmRegs > 0 && VPL == 1;
  constexpr int kLocRegs = kCmRegs > 0 ? kCmRegs : 1;
  // Rows of one vector per lane and every query head in one pass: a wave's
  // share of up to 64 pages has its row ids in one load and goes through two
  // register buffers of kStep pages, the next one's rows in flight while one
  // is scored.  Half of this kernel's time was VALU work and the other half
  // waits of up to four dependent passes; with the buffers, and two columns
  // rounded by one instruction (quest_add), 512 segments of up to 512 pages
  // take 21.2 us per layer instead of 24.7, 8 of 256 pages 12.2 instead of
  // 16.1.  Steps of 8 pages: 20.9 and 13.5 us.
  constexpr int kStep = 16;
  const bool piped = VPL == 1 && a.G <= kG;  // uniform
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ vtx::SelectShared<T> sh;
  __shared__ vtx::BitonicShared<T> bsh;  // cached segments of up to T pages with k <= 32

  const int lane = vtx::lane_id();
  const int wave = vtx::uniform(threadIdx.x / vtx::kWave);
  const int grp = lane / LPR;
  const int col = lane % LPR;
  const int k = a.topk;
  const int D = a.dim;
  const int G = a.G;

  long long cm_pos[kLocRegs];
  if constexpr (cm_on) vtx::closing_load(loc, loc_n, cm_pos);
  const vtx::SchedPick pick = vtx::sched_pick(sched, segments);
  const int seg = pick.seg;
  long long start, n, obase;
  if (pick.predicted) {
    start = (long long)pick.pe[0] + a.bos;
    n = (long long)pick.pe[1] - a.eos - start;
    obase = (long long)pick.pe[2] + a.bos;
  } else {
    start = (long long)a.dindptr[seg] + a.bos;
    n = (long long)a.dindptr[seg + 1] - a.eos - start;
    obase = (long long)a.sindptr[seg] + a.bos;
  }
  auto is_active = [&]() {
    return k > 0 && n > k && start >= 0 && start + n <= a.sum_rows && start + n <= a.aggr_len &&
           start + n <= a.didx_len && obase >= 0 && obase + k <= a.sidx_len;
  };
  bool active = is_active();
  if constexpr (!cm_on) {
    if (!active && !pick.predicted) return;  // uniform: the separate ops write nothing for this segment either
  }
  // the first pass's row ids, then the check of the predicted bounds, in one
  // round trip (as in the GQA kernel)
  long long share = 0;
  int my_row = -1;
  auto first_pass = [&]() {
    share = (n + kWaves - 1) / kWaves;
    share = (share + kRowsPerLoad - 1) / kRowsPerLoad * kRowsPerLoad;
    const int most = piped ? vtx::kWave : kPass;
    if (share > most) share = most;
    const long long p0 = (long long)wave * share;
    const long long cnt = p0 < n ? min(share, n - p0) : 0;
    my_row = lane < cnt ? a.didx[start + p0 + lane] : -1;
  };
  if (active) first_pass();  // uniform
  if (pick.predicted) {      // uniform
    const int32_t* bp = lane == 1 ? a.dindptr + seg + 1 : lane == 2 ? a.sindptr + seg : a.dindptr + seg;
    const int32_t bv = *bp;
    const int32_t t0 = __builtin_amdgcn_readlane(bv, 0), t1 = __builtin_amdgcn_readlane(bv, 1),
                  t2 = __builtin_amdgcn_readlane(bv, 2);
    if ((t0 != pick.pe[0]) | (t1 != pick.pe[1]) | (t2 != pick.pe[2])) {  // uniform; not for a current schedule
      start = (long long)t0 + a.bos;
      n = (long long)t1 - a.eos - start;
      obase = (long long)t2 + a.bos;
      active = is_active();
      if (active) first_pass();
    }
  }
  if constexpr (!cm_on) {
    if (!active) return;  // uniform
  }
  const bool cached = n <= a.row_cap;
  // the bitonic select (one key per thread, from LDS) when every page fits
  // one thread each and k <= 32: no histogram, so no barrier before the rows
  const bool bitonic = cached && n <= T && k <= vtx::kMaxBitonicK;
  uint64_t* sel = reinterpret_cast<uint64_t*>(smem);
  int32_t* rows = reinterpret_cast<int32_t*>(smem + (size_t)vtx::sel_slots(k) * sizeof(uint64_t));
  uint16_t* keys = reinterpret_cast<uint16_t*>(rows + a.row_cap);
  const int32_t* dseg = a.didx + start;
  const uint16_t* qs = a.q + (long long)seg * G * D;
  vtx::Closing<kLocRegs> closing{};
  int n_close = 0;
  if constexpr (cm_on) {
    closing = vtx::closing_build(cma, cm_pos);
    n_close = closing.count;
  }
  // this launch's CMax + CMin: wave w of the workgroup of tile rank r reduces
  // tiles w * grid + r, ... once its own segment is done
  auto cm_tiles = [&]() {
    if constexpr (cm_on)
      vtx::cmean_tiles<LPR, kLocRegs, vtx::kEnvelope>(cma, closing, wave * (int)gridDim.x + pick.tile_rank,
                                                      kWaves * (int)gridDim.x, grp, col);
  };
  if (!active) {  // uniform (only with the in-launch reduce)
    cm_tiles();
    return;
  }
  if (!bitonic) {
    vtx::select_init<T>(sel, k, sh);
    __syncthreads();  // histogram cleared before any wave counts into it
  }

  // ---- scores, page maxima and keys of every middle page
  // page maximum `best` at position p of the segment, row id rid
  auto page_done = [&](long long p, int rid, float best) {
    const uint32_t ab = vtx::f32_to_bf16(best);
    const uint32_t key = vtx::score_key(ab);
    a.aggr[start + p] = (uint16_t)ab;
    if (cached) {
      keys[p] = (uint16_t)key;
      rows[p] = rid;
    }
    if (!bitonic) vtx::select_count<T>(key, sh);
  };
  // A page whose envelopes this launch rewrites (p and rid uniform): scored
  // against the envelopes recomputed from the K tile, stored by lane l.
  auto fresh_page = [&](int l, long long p, int rid) {
    if constexpr (cm_on) {
      vtx::U4 emx, emn;
      vtx::fresh_envelope<LPR>(cma, rid, grp, col, emx, emn);
      float best = -INFINITY;
      for (int g = 0; g < G; ++g) {
        float xg[8];
        vtx::unpack8(vtx::ld16(qs + (long long)g * D + col * 8), xg);
        const uint32_t b = vtx::f32_to_bf16(quest_vec<LPR>(emx, emn, xg));
        if (lane == l) a.sum[(start + p) * G + g] = (uint16_t)b;
        best = fmaxf(best, vtx::bf16_to_f32(b));
      }
      if (lane == l) page_done(p, rid, best);
    }
  };
  // scores of the query heads g0 .. of a page, their maximum into best
  auto heads_done = [&](long long p, int g0, const float (&sc)[kG], float& best) {
#pragma unroll
    for (int gg = 0; gg < kG; ++gg) {
      if (g0 + gg >= G) break;
      const uint32_t b = vtx::f32_to_bf16(sc[gg]);
      a.sum[(start + p) * G + g0 + gg] = (uint16_t)b;
      best = fmaxf(best, vtx::bf16_to_f32(b));
    }
  };
  // query heads g0 .. g0 + kG (heads past G read head G - 1 and are zeroed by
  // a select: no branch around the load, which would make the wave wait for
  // it there)
  auto load_query = [&](int g0, float (&xs)[kG][VPL][8]) {
#pragma unroll
    for (int gg = 0; gg < kG; ++gg)
#pragma unroll
      for (int v = 0; v < VPL; ++v) {
        const bool in = g0 + gg < G;
        float f[8];
        vtx::unpack8(vtx::ld16(qs + (long long)(in ? g0 + gg : G - 1) * D + (v * LPR + col) * 8), f);
#pragma unroll
        for (int e = 0; e < 8; ++e) xs[gg][v][e] = in ? f[e] : 0.f;
      }
  };
  if (piped) {  // uniform
    if constexpr (VPL == 1) {
      float xv[kG][VPL][8];
      load_query(0, xv);
      auto& xs = reinterpret_cast<float(&)[kG][8]>(xv);
      for (long long p0 = (long long)wave * share; p0 < n; p0 += (long long)kWaves * share) {
        const int cnt = (int)min(share, n - p0);
        if (p0 != (long long)wave * share) my_row = lane < cnt ? dseg[p0 + lane] : -1;  // later shares
        int fill = __builtin_amdgcn_readlane(my_row, 0);
        if (fill < 0 || fill >= a.y_rows) fill = 0;
        // the share's pages that are scored afresh, after the others
        uint64_t fresh = 0;
        if constexpr (cm_on)
          if (n_close > 0) fresh = __ballot(vtx::closes_here(cma, closing, lane < cnt ? lane : -1, my_row));
        vtx::QuestRows<LPR, kStep> ba, bb;
        auto issue = [&](int at, vtx::QuestRows<LPR, kStep>& b) {
          vtx::quest_issue<LPR, kStep>(a.ymax, a.ymin, a.y_rows, my_row, fill, at, cnt, grp, col, b);
        };
        auto score = [&](int at, const vtx::QuestRows<LPR, kStep>& b) {
          int r;
          float sc[kG];
          vtx::quest_score<LPR, kStep, kG>(b, xs, at, cnt, grp, col, &r, sc);
          const int rid = __shfl(my_row, (at + r) & (vtx::kWave - 1), vtx::kWave);
          if (r >= 0 && !(fresh >> (at + r) & 1)) {
            float best = -INFINITY;
            heads_done(p0 + at + r, 0, sc, best);
            page_done(p0 + at + r, rid, best);
          }
        };
        issue(0, ba);
        for (int at = 0; at < cnt; at += 2 * kStep) {  // uniform
          issue(at + kStep, bb);
          score(at, ba);
          issue(at + 2 * kStep, ba);
          if (at + kStep < cnt) score(at + kStep, bb);
        }
        for (; fresh; fresh &= fresh - 1) {  // uniform
          const int l = __ffsll((long long)fresh) - 1;
          fresh_page(l, p0 + l, __builtin_amdgcn_readlane(my_row, l));
        }
      }
    }
  } else {
    for (long long p0 = (long long)wave * share; p0 < n; p0 += (long long)kWaves * share) {
      const int cnt = (int)min(share, n - p0);
      if (p0 != (long long)wave * share) my_row = lane < cnt ? dseg[p0 + lane] : -1;  // later passes
      int r = -1;
      float best = -INFINITY;
      for (int g0 = 0; g0 < G; g0 += kG) {
        float xs[kG][VPL][8];
        load_query(g0, xs);
        float sc[kG];
        vtx::quest_pass_multi<LPR, VPL, kPass, kG>(a.ymax, a.ymin, a.y_rows, D, my_row, cnt, xs, grp, col, &r, sc);
        if (r >= 0) heads_done(p0 + r, g0, sc, best);
      }
      const int rid = __shfl(my_row, r < 0 ? 0 : r, vtx::kWave);
      bool done = r < 0;
      if constexpr (cm_on) {
        if (n_close > 0) {  // uniform: stored again by the lane that stored the first scores
          const bool again = vtx::closes_here(cma, closing, r, rid);
          done |= again;
          for (uint64_t m = __ballot(again); m; m &= m - 1) {
            const int l = __ffsll((long long)m) - 1;
            fresh_page(l, p0 + __builtin_amdgcn_readlane(r, l), __builtin_amdgcn_readlane(rid, l));
          }
        }
      }
      if (!done) page_done(p0 + r, rid, best);
    }
  }
  __syncthreads();

  // ---- top-k of the segment: the bitonic select, else the radix select
  // over the counted keys
  if (bitonic) {  // uniform
    const int i = threadIdx.x;
    const uint32_t comp = vtx::bitonic_comp(i < n, i < n ? (uint32_t)keys[i] : 0u, i);
    vtx::select_bitonic<T>(comp, k, bsh, [&](int rk, uint32_t c) { a.sidx[obase + rk] = rows[vtx::bitonic_position(c)]; });
    cm_tiles();
    return;
  }
  if (cached) {
    vtx::select_topk_counted<T>([&](long long i) { return (uint32_t)keys[i]; }, n, k, sel, sh);
  } else {
    const uint16_t* ag = a.aggr + start;
    vtx::select_topk_counted<T>([&](long long i) { return vtx::score_key(ag[i]); }, n, k, sel, sh);
  }
  vtx::select_emit<T>(sel, k, n, [&](int rk, long long pos) { a.sidx[obase + rk] = cached ? rows[pos] : dseg[pos]; });
  cm_tiles();
}

constexpr int kLdsBudget = 56 * 1024;  // dynamic LDS; the select tables take up to ~6 KB more
constexpr int kMaxTopk = 4096;
constexpr int kMaxGroup = 8;

template <int T, int kG>
int launch_dim(const QuestArgs& a, const vtx::CmArgs* cm, int grid, size_t lds, hipStream_t s) {
  const vtx::CmArgs none{};
  if (cm) {  // the in-kernel CMax + CMin: rows of one 16-byte vector per lane
    const bool one = cm->nnz <= vtx::kWave;
    const int32_t nnz = (int32_t)cm->nnz;  // at most vtx::kCmLoc
    switch (a.dim) {
      case 64:
        if (one) quest_fused_kernel<T, 8, 1, kG, 1>
            <<<grid, T, lds, s>>>(a.sched, cm->loc, a.segments, nnz, a, *cm);
        else quest_fused_kernel<T, 8, 1, kG, vtx::kCmLoc / vtx::kWave>
            <<<grid, T, lds, s>>>(a.sched, cm->loc, a.segments, nnz, a, *cm);
        break;
      case 128:
        if (one) quest_fused_kernel<T, 16, 1, kG, 1>
            <<<grid, T, lds, s>>>(a.sched, cm->loc, a.segments, nnz, a, *cm);
        else quest_fused_kernel<T, 16, 1, kG, vtx::kCmLoc / vtx::kWave>
            <<<grid, T, lds, s>>>(a.sched, cm->loc, a.segments, nnz, a, *cm);
        break;
      default: return vtx::fail(VTX_E_INVALID, "indexer_quest_fused: in-kernel page reduce needs head_dim 64 or 128");
    }
    return vtx::check_launch("indexer_quest_fused (with CMax + CMin)");
  }
  switch (a.dim) {
    case 64:
      quest_fused_kernel<T, 8, 1, kG, 0><<<grid, T, lds, s>>>(a.sched, nullptr, a.segments, 0, a, none);
      break;
    case 128:
      quest_fused_kernel<T, 16, 1, kG, 0><<<grid, T, lds, s>>>(a.sched, nullptr, a.segments, 0, a, none);
      break;
    case 256:
      quest_fused_kernel<(T > 512 ? 512 : T), 16, 2, 1, 0>
          <<<grid, (T > 512 ? 512 : T), lds, s>>>(a.sched, nullptr, a.segments, 0, a, none);
      break;
    // wide rows keep their query slice in registers: fewer threads, no spills
    case 512:
      quest_fused_kernel<(T > 512 ? 512 : T), 16, 4, 1, 0>
          <<<grid, (T > 512 ? 512 : T), lds, s>>>(a.sched, nullptr, a.segments, 0, a, none);
      break;
    case 576:
      quest_fused_kernel<256, 8, 9, 1, 0><<<grid, 256, lds, s>>>(a.sched, nullptr, a.segments, 0, a, none);
      break;
    default: return vtx::fail(VTX_E_INVALID, "indexer_quest_fused: head_dim %d not supported", a.dim);
  }
  return vtx::check_launch("indexer_quest_fused");
}

template <int T>
int launch_g(const QuestArgs& a, const vtx::CmArgs* cm, int grid, size_t lds, hipStream_t s) {
  return a.G >= 2 ? launch_dim<T, 2>(a, cm, grid, lds, s) : launch_dim<T, 1>(a, cm, grid, lds, s);
}

}  // namespace

extern "C" int vtx_indexer_quest_fused_supported(int32_t head_dim, int32_t group_size) {
  return (head_dim == 64 || head_dim == 128 || head_dim == 256 || head_dim == 512 || head_dim == 576) &&
         group_size >= 1 && group_size <= kMaxGroup;
}

namespace {

// The decode CMax + CMin a Quest launch may run first (vtx_indexer_quest_fused_cmean).
struct CmeanSpec {
  const uint16_t* k;
  int64_t k_rows;
  int32_t page_size, heads;
  const int64_t* loc;
  int64_t nnz;
};

int quest_impl(const uint16_t* q, int64_t q_rows, int32_t group_size, const uint16_t* ymax, const uint16_t* ymin,
               int64_t y_rows, int32_t head_dim, uint16_t* sum, int64_t sum_rows, uint16_t* aggr, int64_t aggr_len,
               const int32_t* dense_kv_indptr, const int32_t* sparse_kv_indptr, const int32_t* dense_kv_indices,
               int64_t dense_kv_indices_len, int32_t* sparse_kv_indices, int64_t sparse_kv_indices_len,
               int32_t eff_batch_size, int32_t topk_val, int32_t reserved_bos, int32_t reserved_eos,
               int32_t max_num_pages, const CmeanSpec* cms, const int32_t* schedule,
               int64_t schedule_len, void* stream);

}  // namespace

extern "C" int vtx_indexer_quest_fused(const uint16_t* q, int64_t q_rows, int32_t group_size,
                                       const uint16_t* ymax, const uint16_t* ymin, int64_t y_rows,
                                       int32_t head_dim, uint16_t* sum, int64_t sum_rows, uint16_t* aggr,
                                       int64_t aggr_len, const int32_t* dense_kv_indptr,
                                       const int32_t* sparse_kv_indptr, const int32_t* dense_kv_indices,
                                       int64_t dense_kv_indices_len, int32_t* sparse_kv_indices,
                                       int64_t sparse_kv_indices_len, int32_t eff_batch_size, int32_t topk_val,
                                       int32_t reserved_bos, int32_t reserved_eos, int32_t max_num_pages,
                                       const int32_t* schedule, int64_t schedule_len, void* stream) {
  vtx::clear_error();
  return quest_impl(q, q_rows, group_size, ymax, ymin, y_rows, head_dim, sum, sum_rows, aggr, aggr_len,
                    dense_kv_indptr, sparse_kv_indptr, dense_kv_indices, dense_kv_indices_len, sparse_kv_indices,
                    sparse_kv_indices_len, eff_batch_size, topk_val, reserved_bos, reserved_eos, max_num_pages,
                    nullptr, schedule, schedule_len, stream);
}

extern "C" int vtx_indexer_quest_fused_cmean(const uint16_t* q, int64_t q_rows, int32_t group_size,
                                             uint16_t* ymax, uint16_t* ymin, int64_t y_rows, int32_t head_dim,
                                             uint16_t* sum, int64_t sum_rows, uint16_t* aggr, int64_t aggr_len,
                                             const int32_t* dense_kv_indptr, const int32_t* sparse_kv_indptr,
                                             const int32_t* dense_kv_indices, int64_t dense_kv_indices_len,
                                             int32_t* sparse_kv_indices, int64_t sparse_kv_indices_len,
                                             int32_t eff_batch_size, int32_t topk_val, int32_t reserved_bos,
                                             int32_t reserved_eos, int32_t max_num_pages, const uint16_t* k_cache,
                                             int64_t k_rows, int32_t page_size, int32_t num_kv_heads,
                                             const int64_t* loc, int64_t nnz, const int32_t* schedule,
                                             int64_t schedule_len, void* stream) {
  vtx::clear_error();
  if (!k_cache || (nnz > 0 && !loc))
    return vtx::fail(VTX_E_INVALID, "indexer_quest_fused_cmean: null K pool or loc");
  if (page_size < 1 || num_kv_heads < 1 || k_rows < 0 || nnz < 0)
    return vtx::fail(VTX_E_INVALID, "indexer_quest_fused_cmean: bad page-reduce sizes");
  const CmeanSpec cm{k_cache, k_rows, page_size, num_kv_heads, loc, nnz};
  return quest_impl(q, q_rows, group_size, ymax, ymin, y_rows, head_dim, sum, sum_rows, aggr, aggr_len,
                    dense_kv_indptr, sparse_kv_indptr, dense_kv_indices, dense_kv_indices_len, sparse_kv_indices,
                    sparse_kv_indices_len, eff_batch_size, topk_val, reserved_bos, reserved_eos, max_num_pages, &cm,
                    schedule, schedule_len, stream);
}

namespace {

int quest_impl(const uint16_t* q, int64_t q_rows, int32_t group_size, const uint16_t* ymax, const uint16_t* ymin,
               int64_t y_rows, int32_t head_dim, uint16_t* sum, int64_t sum_rows, uint16_t* aggr, int64_t aggr_len,
               const int32_t* dense_kv_indptr, const int32_t* sparse_kv_indptr, const int32_t* dense_kv_indices,
               int64_t dense_kv_indices_len, int32_t* sparse_kv_indices, int64_t sparse_kv_indices_len,
               int32_t eff_batch_size, int32_t topk_val, int32_t reserved_bos, int32_t reserved_eos,
               int32_t max_num_pages, const CmeanSpec* cms, const int32_t* schedule,
               int64_t schedule_len, void* stream) {
  const char* what = "indexer_quest_fused";
  if (eff_batch_size < 0 || reserved_bos < 0 || reserved_eos < 0)
    return vtx::fail(VTX_E_INVALID, "%s: negative size", what);
  if (!vtx_indexer_quest_fused_supported(head_dim, group_size))
    return vtx::fail(VTX_E_INVALID, "%s: head_dim %d with group size %d not supported", what, head_dim,
                     group_size);
  if (topk_val > kMaxTopk) return vtx::fail(VTX_E_INVALID, "%s: topk_val %d exceeds %d", what, topk_val, kMaxTopk);
  if (q_rows < (long long)eff_batch_size * group_size)
    return vtx::fail(VTX_E_INVALID, "%s: %lld query rows for %d segments of %d heads", what, (long long)q_rows,
                     eff_batch_size, group_size);
  // CMax + CMin run inside the launch for rows of one 16-byte vector per lane
  // and decode-sized loc; otherwise as one page-reduce pass of their own, first.
  const bool cm_inside = cms && (head_dim == 64 || head_dim == 128) && cms->nnz <= vtx::kCmLoc;
  if (cms && !cm_inside && cms->nnz > 0) {
    void* const outs[2] = {const_cast<uint16_t*>(ymax), const_cast<uint16_t*>(ymin)};
    const int32_t dtypes[2] = {VTX_DTYPE_BF16, VTX_DTYPE_BF16};
    const int32_t types[2] = {VTX_REDUCE_MAX, VTX_REDUCE_MIN};
    const int rc = vtx_page_reduce_multi(cms->k, cms->k_rows, cms->page_size, head_dim, 2, outs, dtypes, types,
                                         y_rows, cms->loc, cms->nnz, cms->heads, cms->page_size, 1, stream);
    if (rc != VTX_OK) return rc;
  }
  if (eff_batch_size == 0) return VTX_OK;
  if (!q || !ymax || !ymin || !sum || !aggr || !dense_kv_indptr || !sparse_kv_indptr || !dense_kv_indices ||
      !sparse_kv_indices)
    return vtx::fail(VTX_E_INVALID, "%s: null pointer", what);
  if (y_rows <= 0) return vtx::fail(VTX_E_INVALID, "%s: empty envelope pools", what);
  if (!vtx::aligned16(q) || !vtx::aligned16(ymax) || !vtx::aligned16(ymin))
    return vtx::fail(VTX_E_INVALID, "%s: query and envelope rows must be 16-byte aligned", what);
  QuestArgs a;
  a.q = q;
  a.ymax = ymax;
  a.ymin = ymin;
  a.y_rows = y_rows;
  a.sum = sum;
  a.sum_rows = sum_rows;
  a.aggr = aggr;
  a.aggr_len = aggr_len;
  a.dindptr = dense_kv_indptr;
  a.sindptr = sparse_kv_indptr;
  a.didx = dense_kv_indices;
  a.didx_len = dense_kv_indices_len;
  a.sidx = sparse_kv_indices;
  a.sidx_len = sparse_kv_indices_len;
  a.segments = eff_batch_size;
  a.G = group_size;
  a.dim = head_dim;
  a.topk = topk_val > 0 ? topk_val : 0;
  a.bos = reserved_bos;
  a.eos = reserved_eos;
  // a schedule too short for this launch is not used (the kernel would also
  // ignore one whose header names another segment count)
  a.sched = schedule && schedule_len >= vtx::sched_len(1, eff_batch_size) ? schedule : nullptr;
  const long long want = max_num_pages > 0 ? max_num_pages : 0;
  const long long room = (kLdsBudget - (long long)vtx::sel_slots(a.topk) * 8) / 6;  // page id + key per page
  long long cap = want < room ? want : room;
  cap &= ~7LL;
  if (cap < 0) cap = 0;
  a.row_cap = (int32_t)cap;
  const size_t lds = (size_t)vtx::sel_slots(a.topk) * 8 + (size_t)cap * 6;
  hipStream_t s = vtx::as_stream(stream);
  vtx::CmArgs cma{};
  const bool cm_launch = cm_inside && cms->nnz > 0;
  if (cm_launch) {
    cma.x = cms->k;
    cma.x_rows = cms->k_rows;
    cma.rows_per_tile = cms->page_size;
    cma.cols = head_dim;
    cma.out = const_cast<uint16_t*>(ymax);
    cma.out2 = const_cast<uint16_t*>(ymin);
    cma.out_rows = y_rows;
    cma.loc = cms->loc;
    cma.nnz = cms->nnz;
    cma.heads = cms->heads;
    cma.page = cms->page_size;
    cma.page_shift = vtx::log2_exact(cms->page_size);
  }
  const vtx::CmArgs* cmp = cm_launch ? &cma : nullptr;
  switch (vtx::segment_threads(eff_batch_size, max_num_pages, vtx::device_cu_count())) {
    case 256: return launch_g<256>(a, cmp, eff_batch_size, lds, s);
    case 512: return launch_g<512>(a, cmp, eff_batch_size, lds, s);
    default: return launch_g<1024>(a, cmp, eff_batch_size, lds, s);
  }
}

}  // namespace
