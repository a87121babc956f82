// Paged decode attention over a block table for gfx950: the consumer of the
// indexer's sparse block table (or of the dense one, for full attention).
//
// Segment s = b * H + h (request b, kv head h) attends to the tokens of the
// pages kv_indices[kv_indptr[s] .. kv_indptr[s+1]) — each entry a row of the
// K / V pools [rows, P, D] (page * H + h) — all P tokens of every page but
// the last, of which kv_last_page_len[s]; its G query heads (rows s*G + g of
// q [B*H*G, D]) each get
//   o[s*G + g] = sum_t softmax_t(sm_scale * q . K[t]) V[t]      (bf16 out)
// with fp32 scores, an fp32 online softmax and fp32 accumulation.  A segment
// with no tokens writes zeros.
//
// One workgroup per segment, or per chunk of a segment where segments are few
// and long (the chunks' partial outputs then combined by a second launch);
// 8 waves, or 4 for wide G x D.  Three and more query heads take the matrix
// cores (decode_attention_mfma_kernel); what follows describes the VALU kernel
// and holds for both where it speaks of batches and buffers.  The segment's
// page rows are staged in LDS first (one load per page, up to kPageCap
// pages; longer segments read them from the table), so each batch of a
// wave costs one memory round trip: a wave takes every kWaves-th batch of
// kB groups of kRowsPerLoad consecutive tokens (LPR lanes per token, 16-byte
// vectors of K and V; a batch is one contiguous run of rows), and issues the
// next batch's K and V loads
// before it computes on the current one (two register buffers).  It keeps a
// running max and per-lane partial sums (online softmax); the waves'
// (max, sum, accumulator) are merged in LDS.
#include "vtx_device.h"
#include "vtx_host.h"

namespace {

constexpr int kPageCap = 2048;  // page rows staged in LDS

struct AttnArgs {
  const uint16_t* q;
  uint16_t* o;
  const uint16_t* k;
  const uint16_t* v;
  int64_t rows;  // pool rows (page * H + h)
  const int32_t* indptr;
  const int32_t* indices;
  int64_t indices_len;
  const int32_t* last_len;
  int32_t segments, G, D, P;
  int32_t p_shift;  // log2(P), or -1
  float scale;
  // split segments (vtx_paged_decode_attention_split): up to nsplit chunks
  // per segment (chunks_of); ml and acc hold a chunk's (max, sum) and
  // unnormalised output, [segments, nsplit, G(, D)]
  int32_t nsplit, cus, min_avg_tokens;
  int32_t ragged_only;  // split only tables of uneven segments
  float2* ml;
  float* acc;
};

constexpr int kMaxSplit = 128;             // chunks per segment
constexpr int kMaxSplitSegmentsPerCu = 4;  // from so many segments per CU on nothing is split
constexpr int kMinChunkTokens = 128;
constexpr int kFewChunkTokens = 256;

// Chunks of a segment of m pages (1: not split) and the pages of each, from
// the table's total page count: a function of the table alone (the same in
// the attention and the combine kernel, and for two tables that hold the same
// pages in buffers of different capacity).
//
// A table is split when its segments hold min_avg_tokens on average and,
// with half a segment per CU and more, the longest is over 1.3 times the
// average (split_plan says why).  A workgroup takes about 5.5 us + 14 us per
// 1024 tokens (two heads of 128 columns: its dot products, not its loads, set
// that; 1024 threads took as long) until all of them together reach the card's read rate, the combine
// launch 2.5 us.  So a few short segments want one chunk of 128-256 tokens per
// CU (8 segments of 2048 tokens: 11.4 us with chunks of 128, 13.1 with 256; 64
// segments of 1024: 19.0 and 16.0), and long ones four chunks per CU in all,
// which even out ragged lengths without making the chunks short (128 segments
// of 1k to 16k tokens: 107 us, 112 with two or eight and 137 with sixteen).
struct Chunks {
  uint32_t count, pages;
};
// The table's total page count, or 0 where its average is too short to split:
// every thread of both kernels asks this first, of two loads that arrive with
// the segment's own, so that a workgroup of a table that is not split (a short
// one in a large buffer, whose chunks' workgroups are launched all the same)
// does not look for the longest segment.
__device__ __forceinline__ uint32_t split_pages(const AttnArgs& a) {
  const long long all = (long long)a.indptr[a.segments] - a.indptr[0];
  const uint32_t total = all < 0 ? 0u : (uint32_t)(all < a.indices_len ? all : a.indices_len);
  return (unsigned long long)total * a.P < (unsigned long long)a.min_avg_tokens * a.segments ? 0u : total;
}
__device__ __forceinline__ Chunks chunks_of(const AttnArgs& a, uint32_t m, uint32_t longest, uint32_t total) {
  Chunks c{1u, m};
  if (m == 0 || total == 0) return c;
  if (a.ragged_only && 10ull * longest * a.segments <= 13ull * total) return c;
  const uint32_t least = (kMinChunkTokens + a.P - 1) / a.P, few = (kFewChunkTokens + a.P - 1) / a.P;
  uint32_t per = total / a.cus;
  per = per < least ? least : (per > few ? few : per);
  const uint32_t even = (total + 4 * a.cus - 1) / (4 * a.cus);
  per = per < even ? even : per;
  uint32_t n = (m + per - 1) / per;
  n = n > (uint32_t)a.nsplit ? (uint32_t)a.nsplit : n;
  c.pages = (m + n - 1) / n;
  c.count = (m + c.pages - 1) / c.pages;
  return c;
}

// Pages of the table's longest segment (0 where chunks_of does not ask).  Every
// thread of the workgroup calls it; red: LDS, one entry per wave, free again
// after the caller's next barrier.
template <int T>
__device__ __forceinline__ uint32_t longest_segment(const AttnArgs& a, uint32_t* red) {
  if (!a.ragged_only) return 0;  // uniform
  uint32_t mx = 0;
  for (int i = threadIdx.x; i < a.segments; i += T) {
    const int32_t d = (int32_t)((uint32_t)a.indptr[i + 1] - (uint32_t)a.indptr[i]);
    mx = d > 0 && (uint32_t)d > mx ? (uint32_t)d : mx;
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) mx = max(mx, vtx::xshfl(mx, d));
  if (vtx::lane_id() == 0) red[threadIdx.x / vtx::kWave] = mx;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < T / vtx::kWave; ++w) mx = max(mx, red[w]);
  return mx;
}

// What a workgroup attends to: a segment, or one chunk of a split one.
struct Span {
  int seg, chunk, chunks;
  long long start, pages;  // its pages in the table
  int tokens;              // 0: an empty segment
};

// The workgroup's span; false for a chunk past the segment's last.  Every
// thread of the workgroup calls it and gets the same answer.
template <bool kSplit, int T>
__device__ __forceinline__ bool attn_span(const AttnArgs& a, uint32_t* red, Span& sp) {
  const int P = a.P;
  sp.seg = kSplit ? (int)(blockIdx.x % (uint32_t)a.segments) : (int)blockIdx.x;
  sp.chunk = kSplit ? (int)(blockIdx.x / (uint32_t)a.segments) : 0;
  sp.chunks = 1;
  sp.start = a.indptr[sp.seg];
  sp.pages = (long long)a.indptr[sp.seg + 1] - sp.start;
  sp.tokens = 0;
  if (sp.pages > 0 && sp.start >= 0 && sp.start + sp.pages <= a.indices_len && a.rows > 0) {
    int last = a.last_len[sp.seg];
    last = last < 0 ? 0 : (last > P ? P : last);
    const long long t = (sp.pages - 1) * P + last;
    sp.tokens = t < (1LL << 30) ? (int)t : 0;  // (token indices, with the prefetch past the end, fit an int)
    if constexpr (kSplit) {
      const uint32_t total = split_pages(a);
      if (sp.tokens > 0 && total > 0) {  // uniform
        const Chunks c = chunks_of(a, (uint32_t)sp.pages, longest_segment<T>(a, red), total);
        sp.chunks = (int)c.count;
        if (sp.chunk < sp.chunks) {  // this chunk's pages as a segment of their own
          const int p0 = sp.chunk * (int)c.pages;
          const int p1 = min((int)sp.pages, p0 + (int)c.pages);
          sp.tokens = (p1 == (int)sp.pages ? sp.tokens : p1 * P) - p0 * P;
          sp.start += p0;
          sp.pages = p1 - p0;
        }
      }
    }
  }
  return sp.chunk < sp.chunks;
}

// The waves' (max, sum, output) merged, one thread per (g, column): the
// result, or for a split segment the chunk's share for the combine kernel.
template <int kWaves, int kG, int kD, bool kSplit, int T>
__device__ __forceinline__ void attn_merge(const AttnArgs& a, const Span& sp, const float (*s_m)[kG],
                                           const float (*s_l)[kG], const float (*s_acc)[kG][kD]) {
  const int G = a.G;
  for (int idx = threadIdx.x; idx < G * kD; idx += T) {
    const int g = idx / kD;
    const int d = idx - g * kD;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) M = fmaxf(M, s_m[w][g]);
    float L = 0.f, O = 0.f;
    if (M != -INFINITY) {
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        const float f = __expf(s_m[w][g] - M);
        L = fmaf(s_l[w][g], f, L);
        O = fmaf(s_acc[w][g][d], f, O);
      }
    }
    if constexpr (kSplit) {
      if (sp.chunks > 1) {  // uniform
        const long long row = ((long long)sp.seg * a.nsplit + sp.chunk) * G + g;
        a.acc[row * kD + d] = O;
        if (d == 0) a.ml[row] = float2{M, L};
        continue;
      }
    }
    a.o[((long long)sp.seg * G + g) * kD + d] = (uint16_t)vtx::f32_to_bf16(L > 0.f ? O / L : 0.f);
  }
}

// unpack8, or zeros where the token is masked: a weight of 0 does not mask a
// NaN or an infinity in the row that a masked token loaded.  The mask rides on
// the unpacking (a byte permutation instead of the shift, an and): two selects
// per token and no instruction more per value.  Over 45 tables of 64 to 2048
// tokens, time without any masking / with it (mean): one head 0.997, 256 columns and 1
// to 4 heads 0.999, 8 heads 0.98.  Two heads of 64 and 128 columns, whose values
// are unpacked once per head, lose 2 to 7 % to the longer instruction and zero
// the loaded rows of batches with masked tokens behind a branch instead (0.995;
// 0.97 to 0.99 for the others).  Loads from a row of zeros cost up to 4 %, loops
// of their own for batches without masked tokens up to 14 % (code to fetch).
__device__ __forceinline__ void unpack8_or_zero(const vtx::U4& v, bool live, float (&f)[8]) {
  const uint32_t lo = live ? 0x01000c0cu : 0x0c0c0c0cu;  // v_perm_b32: bytes 1 and 0 above two zeros
  const uint32_t hi = live ? 0xffff0000u : 0u;
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = __uint_as_float(__builtin_amdgcn_perm(0u, w[i], lo));
    f[2 * i + 1] = __uint_as_float(w[i] & hi);
  }
}

// Threads per workgroup: 8 waves where a wave's registers fit 128 (rows of
// one 16-byte vector per lane, at most two query heads), else 4.
template <int LPR, int VPL, int kG>
constexpr int attn_threads() {
  return VPL == 1 && kG <= 2 ? 512 : 256;
}
// Token groups per batch (two batches in registers at a time).
template <int VPL, int kG>
constexpr int attn_batch() {
  return VPL == 1 ? (kG == 1 ? 4 : (kG == 2 ? 3 : 2)) : (kG == 1 ? 2 : 1);
}

// With 8 waves, at most 128 registers (four waves per SIMD: two workgroups per CU).
template <int LPR, int VPL, int kG, bool kSplit>
__global__ __launch_bounds__((attn_threads<LPR, VPL, kG>()),
                             (attn_threads<LPR, VPL, kG>() == 512 ? 4 : 1)) void paged_decode_attention_kernel(AttnArgs a) {
  constexpr int T = attn_threads<LPR, VPL, kG>();
  constexpr int kWaves = T / vtx::kWave;
  constexpr int kRowsPerLoad = vtx::kWave / LPR;  // tokens per wave-wide load
  constexpr int kB = attn_batch<VPL, kG>();        // token groups per batch
  constexpr bool kMaskRows = VPL == 1 && kG == 2;  // (unpack8_or_zero says why)
  __shared__ int32_t s_rows[kPageCap];
  __shared__ uint32_t s_red[kWaves];
  __shared__ float s_m[kWaves][kG];
  __shared__ float s_l[kWaves][kG];
  __shared__ float s_acc[kWaves][kG][LPR * VPL * 8];

  const int tid = threadIdx.x;
  const int wave = vtx::uniform(tid / vtx::kWave);
  const int lane = vtx::lane_id();
  const int grp = lane / LPR;
  const int col = lane % LPR;
  const int G = a.G, D = a.D, P = a.P;

  Span sp;
  if (!attn_span<kSplit, T>(a, s_red, sp)) return;  // uniform
  const int seg = sp.seg, T_tok = sp.tokens;
  const long long start = sp.start, m = sp.pages;
  // query slice of this lane (columns (v * LPR + col) * 8 .. + 8), requested
  // first so that it arrives with the page rows; heads past G read head
  // G - 1 and are zeroed by a select (no branch around the load, which would
  // make the wave wait for it there)
  vtx::U4 qraw[kG][VPL];
#pragma unroll
  for (int g = 0; g < kG; ++g)
#pragma unroll
    for (int v = 0; v < VPL; ++v)
      qraw[g][v] = vtx::ld16(a.q + ((long long)seg * G + (g < G ? g : G - 1)) * D + (v * LPR + col) * 8);

  // the segment's page rows (-1: outside the pool)
  const bool staged = m <= kPageCap;
  if (staged && T_tok > 0) {
    for (int i = tid; i < (int)m; i += T) {
      const int r = a.indices[start + i];
      s_rows[i] = (r >= 0 && r < a.rows) ? r : -1;
    }
  }

  float qs[kG][VPL][8];
#pragma unroll
  for (int g = 0; g < kG; ++g)
#pragma unroll
    for (int v = 0; v < VPL; ++v) {
      float f[8];
      vtx::unpack8(qraw[g][v], f);
#pragma unroll
      for (int e = 0; e < 8; ++e) qs[g][v][e] = g < G ? f[e] : 0.f;
    }

  float mx[kG], l[kG], acc[kG][VPL][8];
#pragma unroll
  for (int g = 0; g < kG; ++g) {
    mx[g] = -INFINITY;
    l[g] = 0.f;
#pragma unroll
    for (int v = 0; v < VPL; ++v)
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[g][v][e] = 0.f;
  }
  __syncthreads();  // page rows staged

  const int groups = (T_tok + kRowsPerLoad - 1) / kRowsPerLoad;
  // batches of this wave: groups (wave + kWaves * j) * kB + i, i < kB (a
  // batch is kB consecutive groups: one contiguous run of a page's rows)
  const int batches = (groups + kB - 1) / kB;
  const int nb = batches > wave ? (batches - wave + kWaves - 1) / kWaves : 0;

  // K and V of batch j; tokens past the segment or on rows outside the pool
  // load the pool's first row (a valid address) and are masked off, its values
  // with them: they may be anything, NaN and infinities too
  auto load = [&](int j, vtx::U4 (&kv)[kB][VPL], vtx::U4 (&vv)[kB][VPL], bool (&ok)[kB]) {
#pragma unroll
    for (int i = 0; i < kB; ++i) {
      const int t = ((wave + kWaves * j) * kB + i) * kRowsPerLoad + grp;
      int row = -1, slot = 0;
      if (t < T_tok) {
        const int pg = a.p_shift >= 0 ? t >> a.p_shift : t / P;
        slot = t - pg * P;
        if (staged) {
          row = s_rows[pg];
        } else {
          const int r = a.indices[start + pg];
          row = (r >= 0 && r < a.rows) ? r : -1;
        }
      }
      ok[i] = row >= 0;
      const long long base = ok[i] ? ((long long)row * P + slot) * (long long)D : 0;
#pragma unroll
      for (int v = 0; v < VPL; ++v) {
        kv[i][v] = vtx::ld16_stream(a.k + base + (v * LPR + col) * 8);
        vv[i][v] = vtx::ld16_stream(a.v + base + (v * LPR + col) * 8);
      }
    }
  };
  auto compute = [&](const vtx::U4 (&kv)[kB][VPL], vtx::U4 (&vv)[kB][VPL], const bool (&ok)[kB]) {
    if constexpr (kMaskRows) {
      bool live = true;
#pragma unroll
      for (int i = 0; i < kB; ++i) live = live && ok[i];
      if (__ballot(!live)) {  // uniform: few batches (a segment's last, rows outside the pool)
#pragma unroll
        for (int i = 0; i < kB; ++i)
#pragma unroll
          for (int v = 0; v < VPL; ++v)
            vv[i][v] = vtx::U4{ok[i] ? vv[i][v].x : 0u, ok[i] ? vv[i][v].y : 0u, ok[i] ? vv[i][v].z : 0u,
                               ok[i] ? vv[i][v].w : 0u};
      }
    }
    // scores: every lane of a token's LPR group ends with the full dot
    float sc[kB][kG];
#pragma unroll
    for (int i = 0; i < kB; ++i)
#pragma unroll
      for (int g = 0; g < kG; ++g) {
        float s = vtx::dot_row<VPL>(kv[i], qs[g]);
#pragma unroll
        for (int d = LPR / 2; d >= 1; d >>= 1) s += vtx::xshfl(s, d);
        sc[i][g] = ok[i] ? s * a.scale : -INFINITY;
      }
    // online softmax: the wave's running max covers every token it has seen
#pragma unroll
    for (int g = 0; g < kG; ++g) {
      float bm = sc[0][g];
#pragma unroll
      for (int i = 1; i < kB; ++i) bm = fmaxf(bm, sc[i][g]);
#pragma unroll
      for (int d = LPR; d < vtx::kWave; d <<= 1) bm = fmaxf(bm, vtx::xshfl(bm, d));
      const float nm = fmaxf(mx[g], bm);
      if (nm == -INFINITY) continue;  // nothing seen yet (wave-uniform)
      const float r = __expf(mx[g] - nm);
      l[g] *= r;
#pragma unroll
      for (int v = 0; v < VPL; ++v)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[g][v][e] *= r;
#pragma unroll
      for (int i = 0; i < kB; ++i) {
        const float p = __expf(sc[i][g] - nm);  // 0 for masked tokens
        l[g] += p;
#pragma unroll
        for (int v = 0; v < VPL; ++v) {
          float vf[8];
          unpack8_or_zero(vv[i][v], kMaskRows || ok[i], vf);
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[g][v][e] = fmaf(p, vf[e], acc[g][v][e]);
        }
      }
      mx[g] = nm;
    }
  };

  // two register buffers: batch j + 1's loads are in flight while batch j
  // is computed (the loads are unconditional, so the wait for a buffer is
  // for its own loads only)
  if (nb > 0) {  // uniform over the wave
    vtx::U4 ka[kB][VPL], va[kB][VPL], kb[kB][VPL], vb[kB][VPL];
    bool oka[kB], okb[kB];
    load(0, ka, va, oka);
    for (int j = 0; j < nb; j += 2) {
      load(j + 1, kb, vb, okb);
      compute(ka, va, oka);
      load(j + 2, ka, va, oka);
      if (j + 1 < nb) compute(kb, vb, okb);
    }
  }

  // fold the token groups of the wave (lanes that share col), then the waves
#pragma unroll
  for (int g = 0; g < kG; ++g) {
#pragma unroll
    for (int d = LPR; d < vtx::kWave; d <<= 1) {
      l[g] += vtx::xshfl(l[g], d);
#pragma unroll
      for (int v = 0; v < VPL; ++v)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[g][v][e] += vtx::xshfl(acc[g][v][e], d);
    }
    if (lane == 0) {
      s_m[wave][g] = mx[g];
      s_l[wave][g] = l[g];
    }
    if (grp == 0) {
#pragma unroll
      for (int v = 0; v < VPL; ++v)
#pragma unroll
        for (int e = 0; e < 8; ++e) s_acc[wave][g][(v * LPR + col) * 8 + e] = acc[g][v][e];
    }
  }
  __syncthreads();
  attn_merge<kWaves, kG, LPR * VPL * 8, kSplit, T>(a, sp, s_m, s_l, s_acc);
}

// More than two query heads, rows of 64 or 128 columns, pages of a multiple of
// 16 tokens: the scores on the matrix cores.
//
// With many heads the VALU sets the kernel above's time: dot products with a
// lane tree each and an exponential per token and head in every lane.  Here a
// wave takes 16 consecutive tokens per batch, S^T = K Q^T as kD / 32 steps of
// v_mfma_f32_16x16x32_bf16 (bf16 products, fp32 sums): A holds the tokens' rows
// (lane l: token l % 16, 16 bytes of its row per step), B the query heads
// (lane l: head l % 16, zero past G), and lane l ends with tokens
// 4 (l / 16) + r, r < 4, of head l % 16.  One exponential per lane then serves
// 16 heads.  The probabilities stay in fp32: for P V, lane l takes columns
// (l % 16) * kE .. of V's rows of the same four tokens and reads head g's
// probability from lane g of its 16-lane row (a DPP row broadcast), so P V is
// kE fused multiply-adds per token and head, with no transposition and no
// rounding.  A batch lies in one page, so its row is uniform.
//
// Per layer, D 128, VALU / matrix: 8 heads, 128 segments of 1k to 16k tokens
// 280 / 135 us, 512 of 2048 182 / 90; 4 heads 155 / 121 and 110 / 86, 64 segments
// of 512 tokens 23.5 / 14.2.  Error against 64 bits the same (the result's own
// rounding).  With two heads the VALU keeps up with the card and its wider
// loads (a token's 256 bytes by 16 lanes, here 64 by 4) win: 128 segments of 1k
// to 16k 112 us, 125 here; so 1 and 2 heads stay there.  8 waves instead of 4
// were slower (8 heads' registers leave one such workgroup per CU).
constexpr int kMfmaThreads = 256;
// Waves per SIMD that the registers are limited to.
template <int kG>
constexpr int mfma_waves() {
  return kG <= 4 ? 3 : 2;
}

template <int kG>
__device__ __forceinline__ float row_broadcast(float v, int g) {
  static_assert(kG <= 8, "heads of a row broadcast");
  const int x = (int)__float_as_uint(v);
  int y = 0;
  switch (g) {  // (compile-time constants after unrolling)
    case 0: y = __builtin_amdgcn_update_dpp(0, x, 0x150, 0xf, 0xf, false); break;
    case 1: y = __builtin_amdgcn_update_dpp(0, x, 0x151, 0xf, 0xf, false); break;
    case 2: y = __builtin_amdgcn_update_dpp(0, x, 0x152, 0xf, 0xf, false); break;
    case 3: y = __builtin_amdgcn_update_dpp(0, x, 0x153, 0xf, 0xf, false); break;
    case 4: y = __builtin_amdgcn_update_dpp(0, x, 0x154, 0xf, 0xf, false); break;
    case 5: y = __builtin_amdgcn_update_dpp(0, x, 0x155, 0xf, 0xf, false); break;
    case 6: y = __builtin_amdgcn_update_dpp(0, x, 0x156, 0xf, 0xf, false); break;
    default: y = __builtin_amdgcn_update_dpp(0, x, 0x157, 0xf, 0xf, false); break;
  }
  return __uint_as_float((uint32_t)y);
}

// kE consecutive bf16 values of a V row: 16 bytes (kE 8) or 8 (kE 4).
template <int kE>
struct VRow {
  uint32_t w[kE / 2];
};
template <int kE>
__device__ __forceinline__ VRow<kE> load_v(const uint16_t* p) {
  VRow<kE> r;
  if constexpr (kE == 8) {
    const vtx::U4 t = vtx::ld16_stream(p);
    r.w[0] = t.x;
    r.w[1] = t.y;
    r.w[2] = t.z;
    r.w[3] = t.w;
  } else {
    typedef uint32_t v2u __attribute__((ext_vector_type(2)));
    const v2u t = __builtin_nontemporal_load(reinterpret_cast<const v2u*>(p));
    r.w[0] = t.x;
    r.w[1] = t.y;
  }
  return r;
}

template <int kD, int kG, bool kSplit>
__global__ __launch_bounds__(kMfmaThreads, mfma_waves<kG>()) void decode_attention_mfma_kernel(AttnArgs a) {
  typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  constexpr int T = kMfmaThreads;
  constexpr int kWaves = T / vtx::kWave;
  constexpr int kSteps = kD / 32;  // matrix steps per score
  constexpr int kE = kD / 16;      // V columns per lane
  constexpr int kTok = 16;         // tokens per batch
  __shared__ int32_t s_rows[kPageCap];
  __shared__ uint32_t s_red[kWaves];
  __shared__ float s_m[kWaves][kG];
  __shared__ float s_l[kWaves][kG];
  __shared__ float s_acc[kWaves][kG][kD];

  const int tid = threadIdx.x;
  const int wave = vtx::uniform(tid / vtx::kWave);
  const int lane = vtx::lane_id();
  const int quad = lane / 16;
  const int l16 = lane % 16;
  const int G = a.G, P = a.P;

  Span sp;
  if (!attn_span<kSplit, T>(a, s_red, sp)) return;  // uniform
  const int T_tok = sp.tokens;

  // the query heads as the B operand, requested first
  vtx::U4 qf[kSteps];
#pragma unroll
  for (int s = 0; s < kSteps; ++s)
    qf[s] = vtx::ld16(a.q + ((long long)sp.seg * G + (l16 < G ? l16 : G - 1)) * kD + s * 32 + quad * 8);

  // the segment's page rows (-1: outside the pool)
  const bool staged = sp.pages <= kPageCap;
  if (staged && T_tok > 0) {
    for (int i = tid; i < (int)sp.pages; i += T) {
      const int r = a.indices[sp.start + i];
      s_rows[i] = (r >= 0 && r < a.rows) ? r : -1;
    }
  }
#pragma unroll
  for (int s = 0; s < kSteps; ++s)
    if (l16 >= G) qf[s] = vtx::U4{0u, 0u, 0u, 0u};

  float mx = -INFINITY, l = 0.f;  // head l16; l: the tokens of this lane's quad
  float acc[kG][kE];              // columns l16 * kE + e over the tokens of this lane's quad
#pragma unroll
  for (int g = 0; g < kG; ++g)
#pragma unroll
    for (int e = 0; e < kE; ++e) acc[g][e] = 0.f;
  __syncthreads();  // page rows staged

  // Page rows of this wave's batches j0 .. j0 + 63, one per lane (-1: past the
  // segment or outside the pool).  A page holds a multiple of 16 tokens, so a
  // batch lies in one page and its row is uniform.
  int lane_row = -1;
  auto rows_from = [&](int j0) {
    const int t = (wave + kWaves * (j0 + lane)) * kTok;
    lane_row = -1;
    if (t < T_tok) {
      const int pg = a.p_shift >= 0 ? t >> a.p_shift : t / P;
      if (staged) {
        lane_row = s_rows[pg];
      } else {
        const int r = a.indices[sp.start + pg];
        lane_row = (r >= 0 && r < a.rows) ? r : -1;
      }
    }
  };
  struct Batch {
    vtx::U4 k[kSteps];
    VRow<kE> v[4];
    int tokens;  // of the 16, how many the segment has
  };
  // batch j of this wave: tokens (wave + kWaves * j) * 16 ..  (j in order).
  // All 16 rows are loaded, of the pool's first page for a batch without one
  // (valid addresses: every page has its P >= 16 rows), and masked off.
  auto load = [&](int j, Batch& b) {
    if (j % vtx::kWave == 0) rows_from(j);  // uniform
    const int row = __builtin_amdgcn_readlane(lane_row, j % vtx::kWave);
    const int t0 = (wave + kWaves * j) * kTok;
    const int slot = a.p_shift >= 0 ? t0 & (P - 1) : t0 % P;
    b.tokens = row >= 0 ? min(kTok, T_tok - t0) : 0;
    const long long base = row >= 0 ? ((long long)row * P + slot) * kD : 0;
    const uint16_t* kp = a.k + base + (l16 * kD + quad * 8);
#pragma unroll
    for (int s = 0; s < kSteps; ++s) b.k[s] = vtx::ld16_stream(kp + s * 32);
    const uint16_t* vp = a.v + base + (4 * quad * kD + l16 * kE);
#pragma unroll
    for (int r = 0; r < 4; ++r) b.v[r] = load_v<kE>(vp + r * kD);
  };
  auto compute = [&](Batch& b) {
    f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < kSteps; ++s)
      c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, b.k[s]),
                                                  __builtin_bit_cast(bf16x8, qf[s]), c, 0, 0, 0);
    float p[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) p[r] = 4 * quad + r < b.tokens ? c[r] * a.scale : -INFINITY;
    // online softmax: the running max of head l16 covers every token the wave has seen
    float bm = fmaxf(fmaxf(p[0], p[1]), fmaxf(p[2], p[3]));
    bm = fmaxf(bm, vtx::xshfl(bm, 16));
    bm = fmaxf(bm, vtx::xshfl(bm, 32));
    const float nm = fmaxf(mx, bm);
    if (__ballot(nm > mx && l16 < G)) {  // uniform: a head's maximum grew
      const float f = nm == -INFINITY ? 1.f : __expf(mx - nm);
      l *= f;
#pragma unroll
      for (int g = 0; g < kG; ++g) {
        const float fg = row_broadcast<kG>(f, g);
#pragma unroll
        for (int e = 0; e < kE; ++e) acc[g][e] *= fg;
      }
      mx = nm;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) p[r] = mx == -INFINITY ? 0.f : __expf(p[r] - mx);  // 0 for masked tokens
    l += (p[0] + p[1]) + (p[2] + p[3]);
    if (b.tokens < kTok) {  // uniform: rows past the segment may hold anything, NaN too
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int w = 0; w < kE / 2; ++w) b.v[r].w[w] = 4 * quad + r < b.tokens ? b.v[r].w[w] : 0u;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float vf[kE];
#pragma unroll
      for (int w = 0; w < kE / 2; ++w) {
        vf[2 * w] = vtx::bf16_lo(b.v[r].w[w]);
        vf[2 * w + 1] = vtx::bf16_hi(b.v[r].w[w]);
      }
#pragma unroll
      for (int g = 0; g < kG; ++g) {
        const float pg = row_broadcast<kG>(p[r], g);
#pragma unroll
        for (int e = 0; e < kE; ++e) acc[g][e] = fmaf(pg, vf[e], acc[g][e]);
      }
    }
  };
  // two register buffers, as in paged_decode_attention_kernel
  const int batches = (T_tok + kTok - 1) / kTok;
  const int nb = batches > wave ? (batches - wave + kWaves - 1) / kWaves : 0;
  if (nb > 0) {  // uniform over the wave
    Batch ba, bb;
    load(0, ba);
    for (int j = 0; j < nb; j += 2) {
      load(j + 1, bb);
      compute(ba);
      load(j + 2, ba);
      if (j + 1 < nb) compute(bb);
    }
  }

  // fold the quads of the wave, then the waves
#pragma unroll
  for (int d = 16; d < vtx::kWave; d <<= 1) {
    l += vtx::xshfl(l, d);
#pragma unroll
    for (int g = 0; g < kG; ++g)
#pragma unroll
      for (int e = 0; e < kE; ++e) acc[g][e] += vtx::xshfl(acc[g][e], d);
  }
  if (lane < kG) {
    s_m[wave][lane] = mx;
    s_l[wave][lane] = l;
  }
  if (quad == 0) {
#pragma unroll
    for (int g = 0; g < kG; ++g)
#pragma unroll
      for (int e = 0; e < kE; ++e) s_acc[wave][g][l16 * kE + e] = acc[g][e];
  }
  __syncthreads();
  attn_merge<kWaves, kG, kD, kSplit, T>(a, sp, s_m, s_l, s_acc);
}

// Outputs of the split segments: one workgroup per (segment, query head)
// weighs its chunks' partial outputs, wave w those of chunks w, w + kCombineWaves,
// ... (lane l of the wave holds the (max, sum) of the l-th of them); the waves'
// (max, sum, output) are merged in LDS.
constexpr int kCombineWaves = 4;
static_assert(kMaxSplit <= kCombineWaves * vtx::kWave, "one lane per chunk");
template <int kD>
__global__ __launch_bounds__(kCombineWaves * vtx::kWave) void attention_combine_kernel(AttnArgs a) {
  constexpr int kCols = kD / vtx::kWave;
  constexpr int kAhead = 8;  // chunks loaded before any is added
  __shared__ uint32_t s_red[kCombineWaves];
  __shared__ float s_m[kCombineWaves];
  __shared__ float s_l[kCombineWaves];
  __shared__ float s_o[kCombineWaves][kD];
  const long long row = blockIdx.x;
  const int seg = (int)(row / a.G);
  const int g = (int)(row % a.G);
  const int wave = vtx::uniform(threadIdx.x / vtx::kWave);
  const int lane = vtx::lane_id();
  const long long start = a.indptr[seg];
  const long long m = (long long)a.indptr[seg + 1] - start;
  const int32_t last = a.last_len[seg];
  if (!(m > 0 && start >= 0 && start + m <= a.indices_len && a.rows > 0)) return;  // uniform, as the returns below
  const long long tok = (m - 1) * a.P + (last < 0 ? 0 : (last > a.P ? a.P : last));
  const uint32_t total = split_pages(a);
  if (tok <= 0 || tok >= (1LL << 30) || total == 0) return;
  const uint32_t longest = longest_segment<kCombineWaves * vtx::kWave>(a, s_red);
  const int all = (int)chunks_of(a, (uint32_t)m, longest, total).count;
  if (all <= 1) return;  // written by its workgroup
  // this wave's chunks (none: wave 0's first again, with weight 0)
  const int n = all > wave ? (all - wave + kCombineWaves - 1) / kCombineWaves : 0;
  auto at = [&](int i) {  // row of the i-th of them in ml and acc
    const int c = i < n ? wave + kCombineWaves * i : 0;
    return ((long long)seg * a.nsplit + c) * a.G + g;
  };
  const float2 ml = a.ml[at(lane)];
  float M = lane < n ? ml.x : -INFINITY;
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) M = fmaxf(M, vtx::xshfl(M, d));
  const float w = lane < n && M != -INFINITY ? __expf(ml.x - M) : 0.f;
  const float L = vtx::wave_sum(w * ml.y);
  float O[kCols];
#pragma unroll
  for (int j = 0; j < kCols; ++j) O[j] = 0.f;
  for (int i0 = 0; i0 < n; i0 += kAhead) {
    float v[kAhead][kCols];
#pragma unroll
    for (int i = 0; i < kAhead; ++i)
#pragma unroll
      for (int j = 0; j < kCols; ++j) v[i][j] = a.acc[at(i0 + i) * kD + j * vtx::kWave + lane];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const float f = i0 + i < n ? __uint_as_float(vtx::lane_value(__float_as_uint(w), i0 + i)) : 0.f;
#pragma unroll
      for (int j = 0; j < kCols; ++j) O[j] = i0 + i < n ? fmaf(v[i][j], f, O[j]) : O[j];
    }
  }
  if (lane == 0) {
    s_m[wave] = M;
    s_l[wave] = L;
  }
#pragma unroll
  for (int j = 0; j < kCols; ++j) s_o[wave][j * vtx::kWave + lane] = O[j];
  __syncthreads();
  for (int d = threadIdx.x; d < kD; d += kCombineWaves * vtx::kWave) {
    float MM = -INFINITY;
#pragma unroll
    for (int v = 0; v < kCombineWaves; ++v) MM = fmaxf(MM, s_m[v]);
    float LL = 0.f, OO = 0.f;
    if (MM != -INFINITY) {
#pragma unroll
      for (int v = 0; v < kCombineWaves; ++v) {
        const float f = __expf(s_m[v] - MM);
        LL = fmaf(s_l[v], f, LL);
        OO = fmaf(s_o[v][d], f, OO);
      }
    }
    a.o[row * kD + d] = (uint16_t)vtx::f32_to_bf16(LL > 0.f ? OO / LL : 0.f);
  }
}

// Three and more heads of 64 or 128 columns in pages of a multiple of 16 tokens
// take the matrix cores' kernel (why: there), the rest the VALU's.
template <int kD, int kG>
int launch_one(const AttnArgs& a, hipStream_t s) {
  constexpr int LPR = kD == 64 ? 8 : 16, VPL = kD / (LPR * 8);
  constexpr int T = attn_threads<LPR, VPL, kG>();
  const bool split = a.nsplit > 1;
  const int grid = a.segments * a.nsplit;
  bool matrix = false;
  if constexpr (kD <= 128 && kG >= 4) {
    matrix = a.P % 16 == 0;
    if (matrix && split) decode_attention_mfma_kernel<kD, kG, true><<<grid, kMfmaThreads, 0, s>>>(a);
    else if (matrix) decode_attention_mfma_kernel<kD, kG, false><<<grid, kMfmaThreads, 0, s>>>(a);
  }
  if (!matrix && split) paged_decode_attention_kernel<LPR, VPL, kG, true><<<grid, T, 0, s>>>(a);
  else if (!matrix) paged_decode_attention_kernel<LPR, VPL, kG, false><<<grid, T, 0, s>>>(a);
  if (split) attention_combine_kernel<kD><<<a.segments * a.G, kCombineWaves * vtx::kWave, 0, s>>>(a);
  return vtx::check_launch("paged_decode_attention");
}

template <int kD>
int launch_g(const AttnArgs& a, hipStream_t s) {
  if (a.G <= 1) return launch_one<kD, 1>(a, s);
  if (a.G <= 2) return launch_one<kD, 2>(a, s);
  if (a.G <= 4) return launch_one<kD, 4>(a, s);
  return launch_one<kD, 8>(a, s);
}

}  // namespace

extern "C" int vtx_paged_decode_attention_supported(int32_t head_dim, int32_t group_size) {
  return (head_dim == 64 || head_dim == 128 || head_dim == 256) && group_size >= 1 && group_size <= 8;
}

namespace {

// How a call may split its segments: up to nsplit chunks each (1: not at
// all), in tables whose segments hold min_avg_tokens on average.
struct SplitPlan {
  int32_t nsplit, cus, min_avg_tokens, ragged_only;
};

// Fewer than half a segment per CU leave the chip idle: splitting pays where a
// whole segment takes longer than the extra workgroups and the combine launch.
// A whole segment's time per token follows its dot products and its rows: with
// one and two heads 5.5 us + D / 128 * (6 + 4 G) us per 1024 tokens, and a split
// table of S segments takes about 11 to 17 us, so the line lies at 512 + 8 S
// tokens for two heads of 128 columns and in that proportion for the others.
// Whole / split, 8 segments: D 128, 2 heads 13.2 / 12.1 us at 544 tokens, 21.1 /
// 12.3 at 1056; 1 head 10.6 / 11.2 and 15.9 / 11.1; D 64, 1 head 8.4 / 10.5,
// 10.8 / 10.6 and (2112) 15.9 / 11.1.  16 segments: D 64, 1 head 8.6 / 13.3, 10.9
// / 14.0 and 16.3 / 15.1.  52 of 1024 tokens: D 64, 1 head 11.0 / 16.0; D 128 16.8
// / 17.5.  Three and more heads (4 heads, 52 segments of 1024: 40.5 whole on the
// VALU, 17.8) and rows of 256 columns split from 384 + 8 S tokens on.  With more segments a table gains by evening out its lengths
// (128 segments of 1k to 16k tokens: 219 -> 108 us; 256 of 0.5k to 8k: 128 ->
// 109), and one of equal lengths only pays for the combine launch (128 of 2048:
// 32.3 us, 34.2 with it; 240 of 2048, 1 head: 42.4 and 44.5, D 64 24.3 and 26.7),
// so the line lies where that is a few percent.
//
// The host knows the buffer's capacity, the kernels its contents: a short table in
// a large buffer (32k tokens per segment) pays for the chunks' workgroups, which
// leave at once, and for the second launch.  Two heads of 128 columns, alone / in
// such a buffer: 8 to 128 segments of 64 tokens 5.6 to 5.8 / 7.1 to 7.6 us, of 512
// 11.3 to 11.7 / 12.3 to 13.1; 256 of 64 6.3 / 8.7, 512 of 256 13.9 / 15.9, 1000 of
// 256 22.9 / 26.2 and of 1024 60.5 / 60.6.
SplitPlan split_plan(long long segments, long long indices_len, int32_t page_size, int32_t group_size,
                     int32_t head_dim) {
  const int cus = vtx::device_cu_count();
  SplitPlan p{1, 1, 0, 0};
  if (cus <= 0 || segments <= 0 || segments >= kMaxSplitSegmentsPerCu * (long long)cus) return p;
  p.cus = cus;
  p.ragged_only = 2 * segments >= cus;
  const bool narrow = group_size <= 2 && head_dim <= 128;
  long long least = !p.ragged_only ? (narrow ? 512 : 384) + 8 * segments
                                   : (segments >= cus ? 4096 : (narrow ? 3072 : 2048));
  if (narrow) least = least * 896 / (head_dim * (3 + 2 * group_size));  // (1 for two heads of 128 columns)
  p.min_avg_tokens = (int32_t)least;
  // (a table that cannot hold this average is not split whatever it holds)
  if (indices_len * page_size < least * segments) return p;
  // chunks of a segment: as many as even out the longest, and no more than a
  // table of this capacity can need (chunks_of cuts no chunk below its minimum
  // but the last, so this bound changes no table's chunks)
  const long long min_pages = (kMinChunkTokens + page_size - 1) / page_size;
  long long n = (8LL * cus + segments - 1) / segments;
  n = n > kMaxSplit ? kMaxSplit : n;
  const long long need = (indices_len + min_pages - 1) / min_pages;
  p.nsplit = (int32_t)(n > need ? need : n);
  return p;
}

int attention_impl(const char* what, const uint16_t* q, uint16_t* o, const uint16_t* k_cache,
                   const uint16_t* v_cache, int64_t cache_rows, const int32_t* kv_indptr, const int32_t* kv_indices,
                   int64_t kv_indices_len, const int32_t* kv_last_page_len, int32_t batch_size, int32_t num_kv_heads,
                   int32_t group_size, int32_t head_dim, int32_t page_size, float sm_scale, float* workspace,
                   int64_t workspace_len, void* stream) {
  if (batch_size < 0 || num_kv_heads < 1 || page_size < 1 || cache_rows < 0 || kv_indices_len < 0)
    return vtx::fail(VTX_E_INVALID, "%s: bad sizes", what);
  if (!vtx_paged_decode_attention_supported(head_dim, group_size))
    return vtx::fail(VTX_E_INVALID, "%s: head_dim %d with %d query heads per kv head not supported", what,
                     head_dim, group_size);
  const long long segments = (long long)batch_size * num_kv_heads;
  if (segments == 0) return VTX_OK;
  if (segments > 0x7fffffffLL) return vtx::fail(VTX_E_INVALID, "%s: too many segments", what);
  if (!q || !o || !k_cache || !v_cache || !kv_indptr || !kv_last_page_len || (kv_indices_len > 0 && !kv_indices))
    return vtx::fail(VTX_E_INVALID, "%s: null pointer", what);
  if (!vtx::aligned16(q) || !vtx::aligned16(k_cache) || !vtx::aligned16(v_cache))
    return vtx::fail(VTX_E_INVALID, "%s: q, k_cache and v_cache must be 16-byte aligned", what);
  AttnArgs a;
  a.q = q;
  a.o = o;
  a.k = k_cache;
  a.v = v_cache;
  a.rows = cache_rows;
  a.indptr = kv_indptr;
  a.indices = kv_indices;
  a.indices_len = kv_indices_len;
  a.last_len = kv_last_page_len;
  a.segments = (int32_t)segments;
  a.G = group_size;
  a.D = head_dim;
  a.P = page_size;
  a.p_shift = vtx::log2_exact(page_size);
  a.scale = sm_scale;
  a.nsplit = 1;
  a.cus = 1;
  a.min_avg_tokens = 0;
  a.ragged_only = 0;
  a.ml = nullptr;
  a.acc = nullptr;
  if (workspace) {
    const SplitPlan p = split_plan(segments, kv_indices_len, page_size, group_size, head_dim);
    const long long rows = segments * p.nsplit * group_size;
    if (p.nsplit > 1) {
      if (workspace_len < rows * (head_dim + 2) || !vtx::aligned16(workspace))
        return vtx::fail(VTX_E_INVALID, "%s: workspace of %lld floats (16-byte aligned) needed, got %lld", what,
                         rows * (long long)(head_dim + 2), (long long)workspace_len);
      a.nsplit = p.nsplit;
      a.cus = p.cus;
      a.min_avg_tokens = p.min_avg_tokens;
      a.ragged_only = p.ragged_only;
      a.acc = workspace;
      a.ml = reinterpret_cast<float2*>(workspace + rows * head_dim);
    }
  }
  hipStream_t s = vtx::as_stream(stream);
  switch (head_dim) {
    case 64: return launch_g<64>(a, s);
    case 128: return launch_g<128>(a, s);
    default: return launch_g<256>(a, s);
  }
}

}  // namespace

extern "C" int vtx_paged_decode_attention(const uint16_t* q, uint16_t* o, const uint16_t* k_cache,
                                          const uint16_t* v_cache, int64_t cache_rows, const int32_t* kv_indptr,
                                          const int32_t* kv_indices, int64_t kv_indices_len,
                                          const int32_t* kv_last_page_len, int32_t batch_size,
                                          int32_t num_kv_heads, int32_t group_size, int32_t head_dim,
                                          int32_t page_size, float sm_scale, void* stream) {
  vtx::clear_error();
  return attention_impl("paged_decode_attention", q, o, k_cache, v_cache, cache_rows, kv_indptr, kv_indices,
                        kv_indices_len, kv_last_page_len, batch_size, num_kv_heads, group_size, head_dim, page_size,
                        sm_scale, nullptr, 0, stream);
}

extern "C" int64_t vtx_paged_decode_attention_workspace_len(int32_t batch_size, int32_t num_kv_heads,
                                                            int32_t group_size, int32_t head_dim, int32_t page_size,
                                                            int64_t kv_indices_len) {
  if (batch_size < 0 || num_kv_heads < 1 || page_size < 1 || kv_indices_len < 0 ||
      !vtx_paged_decode_attention_supported(head_dim, group_size))
    return 0;
  const long long segments = (long long)batch_size * num_kv_heads;
  const SplitPlan p = split_plan(segments, kv_indices_len, page_size, group_size, head_dim);
  return p.nsplit > 1 ? segments * p.nsplit * group_size * (head_dim + 2) : 0;
}

extern "C" int vtx_paged_decode_attention_split(const uint16_t* q, uint16_t* o, const uint16_t* k_cache,
                                                const uint16_t* v_cache, int64_t cache_rows,
                                                const int32_t* kv_indptr, const int32_t* kv_indices,
                                                int64_t kv_indices_len, const int32_t* kv_last_page_len,
                                                int32_t batch_size, int32_t num_kv_heads, int32_t group_size,
                                                int32_t head_dim, int32_t page_size, float sm_scale,
                                                float* workspace, int64_t workspace_len, void* stream) {
  vtx::clear_error();
  return attention_impl("paged_decode_attention", q, o, k_cache, v_cache, cache_rows, kv_indptr, kv_indices,
                        kv_indices_len, kv_last_page_len, batch_size, num_kv_heads, group_size, head_dim, page_size,
                        sm_scale, workspace, workspace_len, stream);
}
