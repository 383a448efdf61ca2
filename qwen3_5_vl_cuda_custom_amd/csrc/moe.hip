// Sparse-MoE kernels.
//
//  q3_moe_route     router probabilities -> top-k -> renormalise, one wave per
//                   token: fp32 softmax over the (bf16) logits, k rounds of a
//                   wave arg-max (larger probability wins, lower expert index
//                   among equals), weights = p / sum(p_selected) cast to bf16.
//  q3_moe_experts   dispatch + expert MLPs + combine for routed tokens:
//                     1. count      block per expert: #(token, slot) pairs
//                     2. scan       one block: expert offsets and the m-tile table
//                     3. scatter    block per expert: its pairs in ascending
//                                   token order (a block-wide ballot prefix sum)
//                     4. GEMM 1     grouped MFMA GEMM, gathered token rows x
//                                   gate/up of the pair's expert, SwiGLU epilogue
//                     5. GEMM 2     grouped MFMA GEMM x down, epilogue
//                                   bf16(bf16(y) * routing weight)
//                     6. combine    one wave per token: its k expert rows added
//                                   in ascending expert order with a bf16
//                                   rounding after each add (the order and
//                                   rounding of a per-expert bf16 index_add),
//                                   optionally plus a residual
//                   At most 32 tokens (a decode step): one-block dispatch and
//                   weight-streaming kernels instead of 1 to 5.
//  q3_index_add     deterministic target[idx[i]] += src[i]: bucket the sources
//                   by target, then each target adds its sources in ascending
//                   source order in fp32 and rounds once.
#include <algorithm>

#include <climits>
#include <type_traits>

#include "gemm_bwd.h"
#include "gemm_kernels.h"

using namespace q3;

namespace {

// Expert GEMM tiles: 256 rows x 256 weight rows (SwiGLU: 128 gate/up output
// columns), 8 waves, 64-wide K stages in 2 X and 3 W slots (the whole 160 KB of
// LDS). Every expert's weights stream from HBM exactly once per layer, so W is
// issued two stages ahead. Measured at T=4096, H=2048, I=768, E=128, top-8
// (random routing, 193 m-tiles): gate/up 274 us, down 184 us, against 312 and
// 182 us for 320-row tiles with 2 W slots (one m-tile per expert but 1.42x the
// time per tile wave); with 256 rows per expert, 232 and 156 against 328 and 183.
constexpr int kMoeBM = 256;
constexpr int kMoeBN = 256;
constexpr int kMoeNSTW = 3;

// ------------------------------------------------------------------ routing
// partials (split-K router, q3_moe_router): the logits are first summed from
// nsplit fp32 planes of (T, E), in plane order, rounded once to bf16 and
// written to `logits_out`; the routing then uses those bf16 values.
template <int MAXV>
__global__ __launch_bounds__(256) void moe_route_kernel(const bf16* __restrict__ logits, int* __restrict__ top_idx,
                                                        bf16* __restrict__ top_w, float* __restrict__ top_p,
                                                        int T, int E, int k, int norm,
                                                        const float* __restrict__ partials, int nsplit,
                                                        bf16* __restrict__ logits_out) {
  const int lane = threadIdx.x & 63;
  const int t = (int)(((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6);
  if (t >= T) return;
  const bf16* lr = logits + (int64_t)t * E;
  float v[MAXV];
  bool live[MAXV];
  float mx = -INFINITY;
  if (partials) {
    const int64_t plane = (int64_t)T * E;
#pragma unroll
    for (int i = 0; i < MAXV; ++i) {
      const int e = lane + 64 * i;
      live[i] = e < E;
      float acc = 0.f;
      for (int z = 0; z < nsplit; ++z) acc += live[i] ? partials[z * plane + (int64_t)t * E + e] : 0.f;
      const bf16 b = f2bf(acc);
      if (live[i]) logits_out[(int64_t)t * E + e] = b;
      v[i] = live[i] ? bf2f(b) : -INFINITY;
    }
  } else {
#pragma unroll
    for (int i = 0; i < MAXV; ++i) {
      const int e = lane + 64 * i;
      live[i] = e < E;
      v[i] = live[i] ? bf2f(lr[e]) : -INFINITY;
    }
  }
#pragma unroll
  for (int i = 0; i < MAXV; ++i) mx = fmaxf(mx, v[i]);
  mx = wave_max(mx);
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    v[i] = live[i] ? expf(v[i] - mx) : 0.f;
    s += v[i];
  }
  s = wave_sum(s);
  const float inv = 1.0f / s;
#pragma unroll
  for (int i = 0; i < MAXV; ++i) v[i] *= inv;
  // Top-k by threshold (the same k entries in the same order as k rounds of a
  // wave arg-max, without their shuffle chains). Probabilities are >= +0, so
  // they order as their bit patterns: thr = the k-th largest key, found by a
  // binary search over the bits with ballot counts. The entries above thr and
  // the lowest-index entries equal to it make the k; each then takes its place
  // (larger first, lower expert index among equals) by comparing itself with
  // the selected entries one at a time.
  uint32_t key[MAXV];
#pragma unroll
  for (int i = 0; i < MAXV; ++i) key[i] = __float_as_uint(v[i]);
  uint32_t thr = 0;
  for (int bit = 30; bit >= 0; --bit) {
    const uint32_t cand = thr | (1u << bit);
    int c = 0;
#pragma unroll
    for (int i = 0; i < MAXV; ++i) c += __builtin_popcountll(__ballot(live[i] && key[i] >= cand));
    if (c >= k) thr = cand;
  }
  int need = k;  // entries equal to thr that are taken, lowest index first
#pragma unroll
  for (int i = 0; i < MAXV; ++i) need -= __builtin_popcountll(__ballot(live[i] && key[i] > thr));
  bool sel[MAXV];
  int eq_before = 0;
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const uint64_t eq = __ballot(live[i] && key[i] == thr);
    const int below = eq_before + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(eq >> 32),
                                                                  __builtin_amdgcn_mbcnt_lo((uint32_t)eq, 0u));
    sel[i] = live[i] && (key[i] > thr || (key[i] == thr && below < need));
    eq_before += __builtin_popcountll(eq);
  }
  int pos[MAXV];
#pragma unroll
  for (int i = 0; i < MAXV; ++i) pos[i] = 0;
#pragma unroll
  for (int j = 0; j < MAXV; ++j) {
    uint64_t m = __ballot(sel[j]);
    while (m) {
      const int l = __builtin_ctzll(m);
      m &= m - 1;
      const uint32_t ky = (uint32_t)__builtin_amdgcn_readlane((int)key[j], l);
      const int ey = l + 64 * j;
#pragma unroll
      for (int i = 0; i < MAXV; ++i) pos[i] += (ky > key[i] || (ky == key[i] && ey < lane + 64 * i)) ? 1 : 0;
    }
  }
  // Renormalise: the sum runs over the selected values in selection order.
  float sel_sum = 0.f;
  for (int r = 0; r < k; ++r) {
    uint32_t vr = 0;
#pragma unroll
    for (int j = 0; j < MAXV; ++j) {
      const uint64_t m = __ballot(sel[j] && pos[j] == r);
      if (m) vr = (uint32_t)__builtin_amdgcn_readlane((int)key[j], __builtin_ctzll(m));
    }
    sel_sum += __uint_as_float(vr);
  }
#pragma unroll
  for (int i = 0; i < MAXV; ++i)
    if (sel[i]) {
      const int64_t o = (int64_t)t * k + pos[i];
      top_idx[o] = lane + 64 * i;
      top_w[o] = f2bf(norm ? v[i] / sel_sum : v[i]);
      if (top_p) top_p[o] = v[i];
    }
}

// ------------------------------------------------------------------ permute
// Workspace carve-out (all int32 unless noted):
//   hist[chunks][E], cstart[chunks][E], counts[E], offsets[E + 1],
//   tile_table[max_tiles], n_tiles[1],
//   sorted_token[P], sorted_w (bf16)[P], pos_of[P]   (P = T * k)
struct MoeWs {
  int* hist;    // (chunks, E) entries per chunk and expert
  int* cstart;  // (chunks, E) first row of the chunk's entries in each expert's block
  int* counts;
  int* offsets;
  int* tile_table;
  int* n_tiles;
  int* sorted_token;
  bf16* sorted_w;
  int* pos_of;
  bf16* act;     // (P, I)
  bf16* y_perm;  // (P, H)
  int* chunk_table;  // decode (moe_gemv_kernel): 16-row chunks of the experts' rows
  int* n_chunks;
};

constexpr int kMoeChunk = 64;  // tokens per dispatch chunk (one wave)

// Wave per 64-token chunk: number of (token, slot) entries of the chunk per
// expert (ids outside [0, E) are never dispatched).
__global__ __launch_bounds__(64) void moe_hist_kernel(const int* __restrict__ top_idx, int T, int k, int E,
                                                      int* __restrict__ hist) {
  extern __shared__ int s_cnt[];  // E counters
  const int c = blockIdx.x, lane = threadIdx.x;
  for (int e = lane; e < E; e += 64) s_cnt[e] = 0;
  __syncthreads();
  const int t = c * kMoeChunk + lane;
  if (t < T)
    for (int s = 0; s < k; ++s) {
      const int e = top_idx[(int64_t)t * k + s];
      if (e >= 0 && e < E) atomicAdd(&s_cnt[e], 1);
    }
  __syncthreads();
  for (int e = lane; e < E; e += 64) hist[(int64_t)c * E + e] = s_cnt[e];
}

// Exclusive scan of a[0, n) in LDS by one wave (lane l takes a contiguous
// run of ceil(n / 64) entries); returns the total to every lane.
__device__ int wave_excl_scan(int* a, int n) {
  const int lane = threadIdx.x & 63;
  const int per = (n + 63) / 64, b0 = lane * per;
  int loc = 0;
  for (int i = 0; i < per; ++i)
    if (b0 + i < n) loc += a[b0 + i];
  int incl = loc;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(incl, o, 64);
    if (lane >= o) incl += v;
  }
  int run = incl - loc;
  for (int i = 0; i < per; ++i)
    if (b0 + i < n) {
      const int x = a[b0 + i];
      a[b0 + i] = run;
      run += x;
    }
  return __shfl(incl, 63, 64);
}

// One block of 1024 threads: per-expert counts and offsets (exclusive scan),
// each chunk's first position per expert, and the m-tile table of the grouped
// GEMMs (tiles of kMoeBM rows, expert-major). Thread (g, e) sums the chunk
// range g of expert e (G = 1024 / E ranges; independent loads), so the chunk
// prefix per expert is a short scan over the ranges; the two scans over the
// experts run on one wave each (with a block-wide scan over 1024 threads,
// ~40 barriers, the dispatch took 21.7 us at C4 against 18.7).
__global__ __launch_bounds__(1024) void moe_plan_kernel(const int* __restrict__ hist, int NC, int E,
                                                        int* __restrict__ counts, int* __restrict__ offsets,
                                                        int* __restrict__ cstart, int* __restrict__ tile_table,
                                                        int* __restrict__ n_tiles) {
  __shared__ int s_off[2048], s_til[2048], s_part[1024], s_tot[2];
  const int tid = threadIdx.x;
  const int G = E <= 1024 ? 1024 / E : 1;  // chunk ranges per expert
  // Partial sums (for E > 1024 one range per expert, thread strides over experts).
  for (int e0 = 0; e0 < E; e0 += 1024 / G) {
    const int e = e0 + tid % (1024 / G), g = tid / (1024 / G);
    const bool act = e < E && g < G;
    int sum = 0;
    if (act) {
      const int c0 = (int)((int64_t)g * NC / G), c1 = (int)((int64_t)(g + 1) * NC / G);
#pragma unroll 8
      for (int ci = c0; ci < c1; ++ci) sum += hist[(int64_t)ci * E + e];
    }
    if (G > 1) {
      if (act) s_part[g * E + e] = sum;
    } else if (act) {
      s_off[e] = sum;
    }
  }
  __syncthreads();
  if (G > 1) {
    for (int e = tid; e < E; e += 1024) {
      int run = 0;
      for (int g = 0; g < G; ++g) {
        const int v = s_part[g * E + e];
        s_part[g * E + e] = run;  // exclusive prefix over ranges
        run += v;
      }
      s_off[e] = run;
    }
    __syncthreads();
  }
  for (int e = tid; e < E; e += 1024) {
    counts[e] = s_off[e];
    s_til[e] = (s_off[e] + kMoeBM - 1) / kMoeBM;
  }
  __syncthreads();
  // The two scans over the experts, one wave each.
  if (tid < 64) {
    const int tot = wave_excl_scan(s_off, E);
    if (tid == 0) s_tot[0] = tot;
  } else if (tid < 128) {
    const int tot = wave_excl_scan(s_til, E);
    if (tid == 64) s_tot[1] = tot;
  }
  __syncthreads();
  const int rows = s_tot[0], tiles = s_tot[1];
  for (int e = tid; e < E; e += 1024) {
    const int off = s_off[e];
    offsets[e] = off;
    const int end = e + 1 < E ? s_off[e + 1] : rows;
    int tt = s_til[e];
    for (int m = off; m < end; m += kMoeBM) tile_table[tt++] = (e << 20) | m;
  }
  // Chunk starts: range g of expert e begins at off_e + (rows of ranges < g).
  for (int e0 = 0; e0 < E; e0 += 1024 / G) {
    const int e = e0 + tid % (1024 / G), g = tid / (1024 / G);
    if (e >= E || g >= G) continue;
    int run = s_off[e] + (G > 1 ? s_part[g * E + e] : 0);
    const int c0 = (int)((int64_t)g * NC / G), c1 = (int)((int64_t)(g + 1) * NC / G);
    for (int ci = c0; ci < c1; ++ci) {
      cstart[(int64_t)ci * E + e] = run;
      run += hist[(int64_t)ci * E + e];
    }
  }
  if (tid == 0) {
    offsets[E] = rows;
    *n_tiles = tiles;
  }
}

// Wave per chunk: every (token, slot) entry of an expert gets the next row of
// that expert's block, in (token, slot) order: the order of nonzero() on the
// (T, k) routing matrix. An id outside [0, E) gets no row: its pos_of entry is
// -1 with mark_unplaced, else left as it is. Lane l of every wave holds token
// l's k expert ids in registers and the chunk's histogram and start rows sit in
// LDS; the block's waves split the experts, and per expert present in the chunk
// one ballot per slot counts the entries of the lanes below.
constexpr int kPlaceWaves = 8;  // waves per chunk; wave w places experts e = w (mod 8)

template <int KMAX>
__global__ __launch_bounds__(kPlaceWaves * 64) void moe_place_kernel(const int* __restrict__ top_idx,
                                                       const bf16* __restrict__ top_w, int T, int k, int E,
                                                       const int* __restrict__ hist, const int* __restrict__ cstart,
                                                       int* __restrict__ sorted_token, bf16* __restrict__ sorted_w,
                                                       int* __restrict__ pos_of, bool mark_unplaced) {
  extern __shared__ int s_row[];  // [0, E): the chunk's counts, [E, 2E): its start rows
  const int c = blockIdx.x, lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int e = threadIdx.x; e < E; e += kPlaceWaves * 64) {
    s_row[e] = hist[(int64_t)c * E + e];
    s_row[E + e] = cstart[(int64_t)c * E + e];
  }
  const int t = c * kMoeChunk + lane;
  int ex[KMAX];
  bf16 wv[KMAX];
#pragma unroll
  for (int s = 0; s < KMAX; ++s) {
    const bool ok = t < T && s < k;
    ex[s] = ok ? top_idx[(int64_t)t * k + s] : -1;
    wv[s] = ok ? top_w[(int64_t)t * k + s] : bf16{};
  }
  __syncthreads();
  int dst[KMAX];  // row of each slot's entry (-1: not dispatched)
#pragma unroll
  for (int s = 0; s < KMAX; ++s) dst[s] = -1;
  for (int e = wave; e < E; e += kPlaceWaves) {
    if (s_row[e] == 0) continue;  // uniform
    // Entries of lower lanes (earlier tokens) with expert e: per slot, the
    // ballot's set bits below this lane.
    int below = 0;
#pragma unroll
    for (int s = 0; s < KMAX; ++s) {
      const uint64_t m = __ballot(ex[s] == e);
      below += __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
    }
    int pos = s_row[E + e] + below;
#pragma unroll
    for (int s = 0; s < KMAX; ++s)
      if (ex[s] == e) dst[s] = pos++;
  }
  // One store per slot and array, all lanes together (a slot's row was set
  // by the wave that owns its expert; wave 0 marks the entries without a row).
#pragma unroll
  for (int s = 0; s < KMAX; ++s) {
    if (dst[s] >= 0) {
      sorted_token[dst[s]] = t;
      sorted_w[dst[s]] = wv[s];
      pos_of[(int64_t)t * k + s] = dst[s];
    } else if (mark_unplaced && wave == 0 && t < T && s < k && (ex[s] < 0 || ex[s] >= E)) {
      pos_of[(int64_t)t * k + s] = -1;
    }
  }
}

// One wave per token: add its k expert rows in ascending expert order.
template <int VPL>
__global__ __launch_bounds__(256) void moe_combine_kernel(const int* __restrict__ top_idx,
                                                          const int* __restrict__ pos_of,
                                                          const bf16* __restrict__ y_perm,
                                                          const bf16* __restrict__ residual, bf16* __restrict__ out,
                                                          int T, int k, int H, int E) {
  const int lane = threadIdx.x & 63;
  const int t = (int)(((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6);
  if (t >= T) return;
  int ex[32], ps[32];
  int kk = 0;  // slots with a valid expert id (others were never dispatched)
  for (int s = 0; s < k; ++s) {
    const int e = top_idx[(int64_t)t * k + s];
    const int pp = pos_of[(int64_t)t * k + s];
    if (e < 0 || e >= E || pp < 0 || pp >= T * k) continue;
    ex[kk] = e;
    ps[kk] = pp;
    ++kk;
  }
  k = kk;
  // insertion sort by expert id
  for (int i = 1; i < k; ++i) {
    const int e = ex[i], p = ps[i];
    int j = i - 1;
    while (j >= 0 && ex[j] > e) {
      ex[j + 1] = ex[j];
      ps[j + 1] = ps[j];
      --j;
    }
    ex[j + 1] = e;
    ps[j + 1] = p;
  }
  // lane owns vectors lane + 64 * i of 8 bf16
  const int nvec = H / 8;
  for (int i = 0; i < VPL; ++i) {
    const int vi = lane + 64 * i;
    if (vi >= nvec) break;
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < k; ++s) {
      const bf16x8 yv = reinterpret_cast<const bf16x8*>(y_perm + (int64_t)ps[s] * H)[vi];
#pragma unroll
      for (int q = 0; q < 8; ++q) acc[q] = bf2f(f2bf(acc[q] + bf2f(yv[q])));
    }
    bf16x8 o;
    if (residual) {
      const bf16x8 rv = reinterpret_cast<const bf16x8*>(residual + (int64_t)t * H)[vi];
#pragma unroll
      for (int q = 0; q < 8; ++q) o[q] = f2bf(acc[q] + bf2f(rv[q]));
    } else {
#pragma unroll
      for (int q = 0; q < 8; ++q) o[q] = f2bf(acc[q]);
    }
    reinterpret_cast<bf16x8*>(out + (int64_t)t * H)[vi] = o;
  }
}

// Combine, wide form (k <= 8, H = 8 * blockDim.x): one block per token,
// thread j owns columns [8j, 8j + 8). The token's valid slots are ranked by
// expert id in registers (ties by slot), every thread issues its k row loads
// at once, then adds them in rank order with the same per-add bf16 rounding.
template <int KMAX>
__global__ __launch_bounds__(1024) void moe_combine_wide_kernel(const int* __restrict__ top_idx,
                                                                const int* __restrict__ pos_of,
                                                                const bf16* __restrict__ y_perm,
                                                                const bf16* __restrict__ residual,
                                                                bf16* __restrict__ out, int T, int k, int H, int E) {
  const int t = blockIdx.x;
  const int j = threadIdx.x;
  int e[KMAX], p[KMAX];
#pragma unroll
  for (int s = 0; s < KMAX; ++s) {
    int ee = INT_MAX, pp = -1;
    if (s < k) {
      ee = top_idx[(int64_t)t * k + s];
      pp = pos_of[(int64_t)t * k + s];
      if (ee < 0 || ee >= E || pp < 0 || pp >= T * k) {  // never dispatched
        ee = INT_MAX;
        pp = -1;
      }
    }
    e[s] = ee;
    p[s] = pp;
  }
  // rank[s]: slots before s in (expert, slot) order; invalid slots rank last
  int ps[KMAX];
#pragma unroll
  for (int r = 0; r < KMAX; ++r) ps[r] = -1;
#pragma unroll
  for (int s = 0; s < KMAX; ++s) {
    int rank = 0;
#pragma unroll
    for (int q = 0; q < KMAX; ++q) rank += (e[q] < e[s]) || (e[q] == e[s] && q < s);
#pragma unroll
    for (int r = 0; r < KMAX; ++r)
      if (rank == r) ps[r] = p[s];
  }
  bf16x8 yv[KMAX];
#pragma unroll
  for (int r = 0; r < KMAX; ++r)
    yv[r] = ps[r] >= 0 ? reinterpret_cast<const bf16x8*>(y_perm + (int64_t)ps[r] * H)[j] : bf16x8{};
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int r = 0; r < KMAX; ++r)
    if (ps[r] >= 0)
#pragma unroll
      for (int q = 0; q < 8; ++q) acc[q] = bf2f(f2bf(acc[q] + bf2f(yv[r][q])));
  bf16x8 o;
  if (residual) {
    const bf16x8 rv = reinterpret_cast<const bf16x8*>(residual + (int64_t)t * H)[j];
#pragma unroll
    for (int q = 0; q < 8; ++q) o[q] = f2bf(acc[q] + bf2f(rv[q]));
  } else {
#pragma unroll
    for (int q = 0; q < 8; ++q) o[q] = f2bf(acc[q]);
  }
  reinterpret_cast<bf16x8*>(out + (int64_t)t * H)[j] = o;
}

// ------------------------------------------------------------------ decode
// A decode step routes at most 32 tokens, so an expert gets a few rows and its
// products are a stream of its weights. The tile GEMMs (256-row tiles) leave
// the last wave of tiles nearly empty there (82 experts x 8 down tiles: 2.6
// waves) and stage and multiply 256 rows for one or two; moe_gemv_kernel
// instead deals (16-row chunk of an expert, 32 weight rows) units evenly over
// 256 blocks, and the dispatch of at most 1024 entries is one block's work.
constexpr int kSmallT = 32, kSmallP = 1024, kSmallK = 2048;
bool moe_small(int64_t T, int64_t H, int64_t I, int64_t k) {
  return T <= kSmallT && T * k <= kSmallP && H <= kSmallK && I <= kSmallK;
}

// One block: counts, offsets, every entry's row (ascending (token, slot) per
// expert: the entries before it with the same expert, counted by a scan of the
// list in LDS) and the 16-row chunks (expert << 20 | first row), expert-major.
__global__ __launch_bounds__(kSmallP) void moe_dispatch_small_kernel(const int* __restrict__ top_idx,
                                                                     const bf16* __restrict__ top_w, int P, int k,
                                                                     int E, MoeWs w) {
  __shared__ __attribute__((aligned(16))) int s_e[kSmallP];
  extern __shared__ int s_int[];  // counts -> offsets (E + 1), chunk counts -> offsets (E + 1)
  int* s_off = s_int;
  int* s_ch = s_int + E + 1;
  const int i = threadIdx.x;
  for (int e = i; e <= E; e += kSmallP) s_off[e] = s_ch[e] = 0;
  int e = -1;
  if (i < P) {
    e = top_idx[i];
    if (e < 0 || e >= E) e = -1;  // never dispatched
  }
  s_e[i] = e;
  __syncthreads();
  if (e >= 0) atomicAdd(&s_off[e], 1);
  __syncthreads();
  for (int x = i; x < E; x += kSmallP) s_ch[x] = (s_off[x] + 15) / 16;
  __syncthreads();
  if (i < 64) wave_excl_scan(s_off, E + 1);
  else if (i < 128) wave_excl_scan(s_ch, E + 1);
  int rank = 0;
  const int4* e4 = reinterpret_cast<const int4*>(s_e);
#pragma unroll 8
  for (int j = 0; j < (P + 3) / 4; ++j) {
    const int4 v = e4[j];
    rank += (4 * j < i && v.x == e) + (4 * j + 1 < i && v.y == e) + (4 * j + 2 < i && v.z == e) +
            (4 * j + 3 < i && v.w == e);
  }
  __syncthreads();
  if (i < P) {
    const int pos = e >= 0 ? s_off[e] + rank : -1;
    w.pos_of[i] = pos;
    if (pos >= 0) {
      w.sorted_token[pos] = i / k;
      w.sorted_w[pos] = top_w[i];
    }
  }
  for (int x = i; x <= E; x += kSmallP) {
    w.offsets[x] = s_off[x];
    if (x < E)
      for (int c = s_ch[x]; c < s_ch[x + 1]; ++c) w.chunk_table[c] = (x << 20) | (s_off[x] + 16 * (c - s_ch[x]));
  }
  if (i == 0) *w.n_chunks = s_ch[E];
}

struct MoeGemvP {
  const bf16 *X, *W, *rowscale;  // X rows (through `gather` when set), W (E, rows, K)
  bf16* C;                       // (P, N)
  const int *gather, *chunk_table, *n_chunks, *offsets;
  int N, K, ldx, x_rows;         // N: output columns (SWIGLU: I, W has 2 I rows)
};

// C[row] = X[row] . W[e]^T of at most 16 rows per chunk. A unit is 32 weight
// rows (SWIGLU: 16 gate rows and the 16 up rows of the same columns, else 32
// consecutive ones): waves 0, 1 take the first 16 rows, waves 2, 3 the other
// 16, each wave one half of K, so its X fragments stay in registers while the
// expert lasts (NST stages of 128 k, 4 fragments each). A wave streams its
// weights through a private LDS ring of kRing stages (16 rows x 128 k, 4 KB) by
// non-temporal direct-to-LDS loads that run on across units, no barrier in
// between; the halves (and gate and up) meet in LDS once per unit, two buffers
// in turn. A stage is issued into the slot that the step before has read, so the
// issue first waits for that step's LDS reads (its MFMAs wait for them as well). Chunk c of a stage row r sits at slot c ^ r (conflict-free fragment
// reads). SPLIT false (K <= 1024, plain): a unit is 64 rows, each wave takes 16
// of them over all of K and stores them alone, with no exchange or barrier.
// Bound by the weight stream: 16
// tokens, top-8 of 128 experts, H = 2048, I = 768 (about 82 experts, 775 MB):
// gate/up 110 -> 83 us (6.2 TB/s), down 59 -> 47 us against the tile GEMMs.
template <bool SWIGLU, int NST, bool SPLIT>
__global__ __launch_bounds__(256) void moe_gemv_kernel(const MoeGemvP p) {
  constexpr int kRing = 8, kStage = 16 * 128;
  __shared__ __attribute__((aligned(1024))) bf16 ring[4 * kRing * kStage];
  __shared__ __attribute__((aligned(16))) floatx4 s_part[2][SPLIT ? 4 : 1][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  static_assert(SPLIT || !SWIGLU, "gate and up meet in the exchange");
  constexpr int kUnit = SPLIT ? 32 : 64;  // weight rows per unit (SWIGLU: 16 of each matrix)
  const int grp = SPLIT ? wave >> 1 : wave, kh = SPLIT ? wave & 1 : 0, l16 = lane & 15, q4 = lane >> 4;
  const int N = p.N, K = p.K;
  const int NG = SWIGLU ? (N + 15) / 16 : (N + kUnit - 1) / kUnit;
  const int wrows = SWIGLU ? 2 * N : N;
  const int64_t U = (int64_t)*p.n_chunks * NG;
  const int u0 = (int)(U * blockIdx.x / gridDim.x), u1 = (int)(U * (blockIdx.x + 1) / gridDim.x);
  if (u0 >= u1) return;
  const int kbeg = kh * NST * 128;
  const uint32_t lring = q3::lds_addr(ring + wave * kRing * kStage);

  // Issue cursor: stage `is` of unit `iu` (chunk ic, group ig).
  int iu = u0, is = 0, ic = u0 / NG, ig = u0 - ic * NG, slot_i = 0;
  int ie = __builtin_amdgcn_readfirstlane(p.chunk_table[ic]) >> 20;
  const int lrow = lane >> 4;
  auto issue = [&]() {
    const bool live = iu < u1;
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(p.W + (int64_t)ie * wrows * K, (int64_t)wrows * K * 2);
    const int r0 = SWIGLU ? (grp ? N : 0) + 16 * ig : kUnit * ig + 16 * grp;
    const int rlim = (SWIGLU ? 16 * ig : r0) + 16 <= N ? 16 : N - (SWIGLU ? 16 * ig : r0);  // live rows (may be <= 0)
    const uint32_t dst = lring + (uint32_t)(slot_i * kStage * 2);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot's last fragment reads have returned
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 4 * i + lrow, k = kbeg + is * 128 + ((l16 ^ r) << 3);
      const bool ok = live && r < rlim && k < K;
      dma16_nt(rs, ok ? (uint32_t)(((r0 + r) * K + k) * 2) : kOOB, dst + (uint32_t)(i * 1024));
    }
    slot_i = slot_i + 1 == kRing ? 0 : slot_i + 1;
    if (++is == NST) {
      is = 0;
      ++iu;
      if (++ig == NG && iu < u1) {
        ig = 0;
        ie = __builtin_amdgcn_readfirstlane(p.chunk_table[++ic]) >> 20;
      }
    }
  };
#pragma unroll
  for (int j = 0; j < kRing - 1; ++j) issue();

  const __amdgpu_buffer_rsrc_t xrs = make_rsrc(p.X, (int64_t)p.x_rows * p.ldx * 2);
  bf16x8 xf[NST * 4];
  float rs = 1.f;  // this lane's row scale (loaded with the rows: a load in the epilogue would drain the ring)
  int cc = -1, row0 = 0, rows = 0, slot_c = 0;
  for (int u = u0; u < u1; ++u) {
    const int c = u / NG, g = u - c * NG;
    if (c != cc) {  // this chunk's rows as B fragments: lane l holds row l % 16, k 8 (l / 16) .. + 7 of each 32
      cc = c;
      const int entry = __builtin_amdgcn_readfirstlane(p.chunk_table[c]);
      row0 = entry & 0xFFFFF;
      rows = min(16, __builtin_amdgcn_readfirstlane(p.offsets[(entry >> 20) + 1]) - row0);
      const bool live = l16 < rows;
      const int src = live ? (p.gather ? p.gather[row0 + l16] : row0 + l16) : 0;
      if constexpr (!SWIGLU) rs = live ? bf2f(p.rowscale[row0 + l16]) : 0.f;
      const uint32_t x0 = live ? (uint32_t)(src * p.ldx * 2) : kOOB;
#pragma unroll
      for (int s = 0; s < NST * 4; ++s) {
        const int k = kbeg + s * 32 + 8 * q4;
        xf[s] = buffer_load16(xrs, k < K ? x0 + (uint32_t)(k * 2) : kOOB);
      }
    }
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < NST; ++s) {
      issue();
      vm_wait<(kRing - 1) * 4>();  // the oldest stage has landed
      const bf16* st = ring + (wave * kRing + slot_c) * kStage + l16 * 128;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(st + (((4 * ks + q4) ^ l16) << 3));
        acc = mfma16x16x32(a, xf[4 * s + ks], acc);
      }
      slot_c = slot_c + 1 == kRing ? 0 : slot_c + 1;
    }
    // register r of lane (q4, l16): weight row 4 q4 + r, token row l16
    const int buf = u & 1;
    if constexpr (SPLIT) {
      s_part[buf][wave][lane] = acc;
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
    if (kh == 0 && (!SWIGLU || grp == 0) && l16 < rows) {
      floatx4 a = acc;
      if constexpr (SPLIT) a += s_part[buf][wave + 1][lane];
      const int n = SWIGLU ? 16 * g + 4 * q4 : kUnit * g + 16 * grp + 4 * q4;
      bf16x4 o;
      if constexpr (SWIGLU) {
        const floatx4 b = s_part[buf][2][lane] + s_part[buf][3][lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = f2bf(silu_mul(a[e], b[e]));
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = f2bf(bf2f(f2bf(a[e])) * rs);
      }
      if (n < N) *reinterpret_cast<bf16x4*>(p.C + (int64_t)(row0 + l16) * N + n) = o;  // N is a multiple of 8
    }
  }
  vm_wait<0>();  // no load may still target this block's LDS when the wave retires
}

template <bool SWIGLU, bool SPLIT>
int launch_moe_gemv_t(const MoeGemvP& p, hipStream_t st) {
  const int n = (int)q3_cdiv(p.K, SPLIT ? 256 : 128);  // stages of 128 k per wave
  auto run = [&](auto stages) {
    hipLaunchKernelGGL((moe_gemv_kernel<SWIGLU, decltype(stages)::value, SPLIT>), dim3(256), dim3(256), 0, st, p);
  };
  if constexpr (SWIGLU || !SPLIT) {  // (the plain split form starts at K > 1024)
    if (n == 1) run(std::integral_constant<int, 1>{});
    if (n == 2) run(std::integral_constant<int, 2>{});
    if (n == 3) run(std::integral_constant<int, 3>{});
    if (n == 4) run(std::integral_constant<int, 4>{});
  }
  if (n == 5 || n == 6) run(std::integral_constant<int, 6>{});
  if (n > 6) run(std::integral_constant<int, 8>{});
  Q3_LAUNCH_CHECK();
  return Q3_OK;
}
template <bool SWIGLU>
int launch_moe_gemv(const MoeGemvP& p, hipStream_t st) {
  if constexpr (!SWIGLU) {
    if (p.K <= 1024) return launch_moe_gemv_t<SWIGLU, false>(p, st);
  }
  return launch_moe_gemv_t<SWIGLU, true>(p, st);
}

int64_t align256(int64_t x) { return (x + 255) / 256 * 256; }

int64_t moe_ws_layout(int64_t T, int64_t H, int64_t I, int64_t E, int64_t k, MoeWs* ws, char* base) {
  const int64_t P = T * k;
  const int64_t max_tiles = q3_cdiv(P, kMoeBM) + E;
  int64_t off = 0;
  auto take = [&](int64_t bytes) {
    char* p = base ? base + off : nullptr;
    off += align256(bytes);
    return p;
  };
  MoeWs w{};
  const int64_t NC = q3_cdiv(T, kMoeChunk);
  w.hist = reinterpret_cast<int*>(take(NC * E * 4));
  w.cstart = reinterpret_cast<int*>(take(NC * E * 4));
  w.counts = reinterpret_cast<int*>(take(E * 4));
  w.offsets = reinterpret_cast<int*>(take((E + 1) * 4));
  w.tile_table = reinterpret_cast<int*>(take(max_tiles * 4));
  w.n_tiles = reinterpret_cast<int*>(take(4));
  w.sorted_token = reinterpret_cast<int*>(take(P * 4));
  w.sorted_w = reinterpret_cast<bf16*>(take(P * 2));
  w.pos_of = reinterpret_cast<int*>(take(P * 4));
  w.act = reinterpret_cast<bf16*>(take(P * I * 2));
  w.y_perm = reinterpret_cast<bf16*>(take(P * H * 2));
  if (moe_small(T, H, I, k)) {
    w.chunk_table = reinterpret_cast<int*>(take((E + P / 16 + 1) * 4));
    w.n_chunks = reinterpret_cast<int*>(take(4));
  }
  if (ws) *ws = w;
  return off;
}

// Workspace of the dispatch alone (q3_moe_permute): the per-chunk tables,
// counts and the m-tile table; the sorted list, weights and positions go to
// the caller's buffers.
int64_t moe_permute_ws_layout(int64_t T, int64_t E, int64_t k, MoeWs* ws, char* base) {
  const int64_t P = T * k;
  const int64_t max_tiles = q3_cdiv(P, kMoeBM) + E;
  int64_t off = 0;
  auto take = [&](int64_t bytes) {
    char* p = base ? base + off : nullptr;
    off += align256(bytes);
    return p;
  };
  MoeWs w{};
  const int64_t NC = q3_cdiv(T, kMoeChunk);
  w.hist = reinterpret_cast<int*>(take(NC * E * 4));
  w.cstart = reinterpret_cast<int*>(take(NC * E * 4));
  w.counts = reinterpret_cast<int*>(take(E * 4));
  w.tile_table = reinterpret_cast<int*>(take(max_tiles * 4));
  w.n_tiles = reinterpret_cast<int*>(take(4));
  if (ws) *ws = w;
  return off;
}

// Dispatch: per-expert counts and offsets, the m-tile table, and every
// (token, slot) entry's row in expert-major, (token, slot)-ascending order
// (the order of the reference's per-expert nonzero(), modules/moe.py:75).
int moe_dispatch(const int* top_idx, const bf16* top_w, int64_t T, int64_t k, int64_t E, const MoeWs& w,
                 hipStream_t st, bool mark_unplaced = false) {
  const int NC = (int)q3_cdiv(T, kMoeChunk);
  hipLaunchKernelGGL(moe_hist_kernel, dim3((unsigned)NC), dim3(64), E * sizeof(int), st, top_idx, (int)T, (int)k,
                     (int)E, w.hist);
  hipLaunchKernelGGL(moe_plan_kernel, dim3(1), dim3(1024), 0, st, w.hist, NC, (int)E, w.counts, w.offsets, w.cstart,
                     w.tile_table, w.n_tiles);
  const dim3 place_blk(kPlaceWaves * 64);
  const size_t place_lds = 2 * E * sizeof(int);
  if (k <= 8)
    hipLaunchKernelGGL(moe_place_kernel<8>, dim3((unsigned)NC), place_blk, place_lds, st, top_idx, top_w, (int)T,
                       (int)k, (int)E, w.hist, w.cstart, w.sorted_token, w.sorted_w, w.pos_of, mark_unplaced);
  else
    hipLaunchKernelGGL(moe_place_kernel<32>, dim3((unsigned)NC), place_blk, place_lds, st, top_idx, top_w, (int)T,
                       (int)k, (int)E, w.hist, w.cstart, w.sorted_token, w.sorted_w, w.pos_of, mark_unplaced);
  Q3_LAUNCH_CHECK();
  return Q3_OK;
}

// ------------------------------------------------------------------ index_add
__global__ void fill_int_kernel(int* p, int64_t n, int v) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

__global__ void ia_count_kernel(const int64_t* __restrict__ idx, int64_t ns, int64_t nt, int* __restrict__ counts,
                                int* __restrict__ bad) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < ns; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t t = idx[i];
    if (t < 0 || t >= nt) {
      atomicOr(bad, 1);
      continue;
    }
    atomicAdd(&counts[t], 1);
  }
}

__global__ void ia_scan_kernel(const int* __restrict__ counts, int64_t nt, int* __restrict__ starts) {
  // Single block, 256 threads: chunked scan.
  __shared__ int s[256];
  __shared__ int carry;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (int64_t c0 = 0; c0 < nt; c0 += 256) {
    const int64_t i = c0 + threadIdx.x;
    const int v = i < nt ? counts[i] : 0;
    s[threadIdx.x] = v;
    __syncthreads();
    for (int o = 1; o < 256; o <<= 1) {
      const int a = (threadIdx.x >= (unsigned)o) ? s[threadIdx.x - o] : 0;
      __syncthreads();
      s[threadIdx.x] += a;
      __syncthreads();
    }
    if (i < nt) starts[i] = carry + s[threadIdx.x] - v;
    __syncthreads();
    if (threadIdx.x == 255) carry += s[255];
    __syncthreads();
  }
  if (threadIdx.x == 0) starts[nt] = carry;
}

__global__ void ia_scatter_kernel(const int64_t* __restrict__ idx, int64_t ns, int64_t nt,
                                  const int* __restrict__ starts, int* __restrict__ fill, int* __restrict__ bucket) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < ns; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t t = idx[i];
    if (t < 0 || t >= nt) continue;
    const int slot = atomicAdd(&fill[t], 1);
    bucket[starts[t] + slot] = (int)i;
  }
}

// One wave per target row. Its sources are added in ascending source index,
// in fp32 starting from the target value, with one rounding at the end (the
// order and precision of torch's CPU index_add_). The bucket (unordered after
// the atomic scatter) is rank-sorted in LDS when it holds <= kIaLds entries;
// longer buckets take the next-smallest index by repeated wave minima.
constexpr int kIaLds = 1024;

template <typename T>
__global__ __launch_bounds__(256) void ia_accumulate_kernel(T* __restrict__ target, const T* __restrict__ src,
                                                            const int* __restrict__ starts,
                                                            const int* __restrict__ bucket, int64_t nt, int64_t D) {
  __shared__ int s_raw[4][kIaLds];
  __shared__ int s_sorted[4][kIaLds];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int64_t t = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  if (t >= nt) return;
  const int b0 = starts[t], c = starts[t + 1] - b0;
  if (c == 0) return;
  T* tr = target + t * D;
  if (c <= kIaLds) {
    for (int j = lane; j < c; j += 64) s_raw[wave][j] = bucket[b0 + j];
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    for (int j = lane; j < c; j += 64) {
      const int v = s_raw[wave][j];
      int rank = 0;
      for (int q = 0; q < c; ++q) rank += s_raw[wave][q] < v;  // source indices are distinct
      s_sorted[wave][rank] = v;
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    for (int64_t d = lane; d < D; d += 64) {
      float acc = to_f<T>(tr[d]);
      for (int n = 0; n < c; ++n) acc += to_f<T>(src[(int64_t)s_sorted[wave][n] * D + d]);
      tr[d] = from_f<T>(acc);
    }
    return;
  }
  for (int64_t d0 = 0; d0 < D; d0 += 64) {
    const int64_t d = d0 + lane;
    float acc = d < D ? to_f<T>(tr[d]) : 0.f;
    int prev = -1;
    for (int n = 0; n < c; ++n) {
      int best = 0x7fffffff;
      for (int j = lane; j < c; j += 64) {
        const int v = bucket[b0 + j];
        if (v > prev && v < best) best = v;
      }
#pragma unroll
      for (int o = 32; o >= 1; o >>= 1) best = min(best, __shfl_xor(best, o, 64));
      prev = best;
      if (d < D) acc += to_f<T>(src[(int64_t)best * D + d]);
    }
    if (d < D) tr[d] = from_f<T>(acc);
  }
}

template <typename T>
int index_add_t(void* target, const void* src, const int64_t* idx, int64_t ns, int64_t nt, int64_t D, char* ws,
                int* status, hipStream_t st) {
  int* counts = reinterpret_cast<int*>(ws);
  int* fill = counts + nt;
  int* starts = fill + nt;
  int* bucket = starts + nt + 1;
  int* bad = status ? status : bucket + ns;  // the caller's status word is sticky: never cleared here
  const unsigned fb = (unsigned)std::min<int64_t>(q3_cdiv(2 * nt + 1, 256), 1024);
  hipLaunchKernelGGL(fill_int_kernel, dim3(fb), dim3(256), 0, st, counts, 2 * nt, 0);
  if (!status) hipLaunchKernelGGL(fill_int_kernel, dim3(1), dim3(64), 0, st, bad, (int64_t)1, 0);
  const unsigned sb = (unsigned)std::max<int64_t>(1, std::min<int64_t>(q3_cdiv(ns, 256), 1024));
  hipLaunchKernelGGL(ia_count_kernel, dim3(sb), dim3(256), 0, st, idx, ns, nt, counts, bad);
  hipLaunchKernelGGL(ia_scan_kernel, dim3(1), dim3(256), 0, st, counts, nt, starts);
  hipLaunchKernelGGL(ia_scatter_kernel, dim3(sb), dim3(256), 0, st, idx, ns, nt, starts, fill, bucket);
  hipLaunchKernelGGL(ia_accumulate_kernel<T>, dim3((unsigned)q3_cdiv(nt, 4)), dim3(256), 0, st,
                     static_cast<T*>(target), static_cast<const T*>(src), starts, bucket, nt, D);
  Q3_LAUNCH_CHECK();
  return Q3_OK;
}

}  // namespace

namespace {

// Splits over K of the router GEMM (q3_moe_router): enough (T/128 x E/128)
// tiles x splits to give every CU one (at most 256), each split a multiple of
// 64 columns dividing H (a 2048-wide router at 4096 tokens: 32 tiles x 8
// splits of 256).
int router_splits(int64_t T, int64_t H, int64_t E) {
  const int64_t tiles = q3_cdiv(T, 128) * q3_cdiv(E, 128);
  int best = 1;
  for (int s = 2; s <= 64; ++s)
    if (tiles * s <= 256 && H % s == 0 && (H / s) % 64 == 0) best = s;
  return best;
}

int launch_route(const bf16* lg, int* top_idx, bf16* tw, float* top_p, int64_t T, int64_t E, int64_t k, int norm,
                 const float* partials, int ns, bf16* lg_out, hipStream_t st) {
  const unsigned blocks = (unsigned)q3_cdiv(T, 4);
  if (E <= 64)
    hipLaunchKernelGGL(moe_route_kernel<1>, dim3(blocks), dim3(256), 0, st, lg, top_idx, tw, top_p, (int)T, (int)E,
                       (int)k, norm, partials, ns, lg_out);
  else if (E <= 128)
    hipLaunchKernelGGL(moe_route_kernel<2>, dim3(blocks), dim3(256), 0, st, lg, top_idx, tw, top_p, (int)T, (int)E,
                       (int)k, norm, partials, ns, lg_out);
  else if (E <= 256)
    hipLaunchKernelGGL(moe_route_kernel<4>, dim3(blocks), dim3(256), 0, st, lg, top_idx, tw, top_p, (int)T, (int)E,
                       (int)k, norm, partials, ns, lg_out);
  else
    hipLaunchKernelGGL(moe_route_kernel<8>, dim3(blocks), dim3(256), 0, st, lg, top_idx, tw, top_p, (int)T, (int)E,
                       (int)k, norm, partials, ns, lg_out);
  Q3_LAUNCH_CHECK();
  return Q3_OK;
}

int launch_combine(const int* top_idx, const int* pos_of, const bf16* y_perm, const bf16* res, bf16* o, int64_t T,
                   int64_t H, int64_t E, int64_t k, hipStream_t st) {
  const int vpl = (int)q3_cdiv(H / 8, 64);
  const unsigned cb = (unsigned)q3_cdiv(T, 4);
  if (k <= 8 && H % 8 == 0 && H / 8 <= 1024) {
    hipLaunchKernelGGL(moe_combine_wide_kernel<8>, dim3((unsigned)T), dim3((unsigned)(H / 8)), 0, st, top_idx,
                       pos_of, y_perm, res, o, (int)T, (int)k, (int)H, (int)E);
  } else if (vpl <= 4)
    hipLaunchKernelGGL(moe_combine_kernel<4>, dim3(cb), dim3(256), 0, st, top_idx, pos_of, y_perm, res, o, (int)T,
                       (int)k, (int)H, (int)E);
  else if (vpl <= 8)
    hipLaunchKernelGGL(moe_combine_kernel<8>, dim3(cb), dim3(256), 0, st, top_idx, pos_of, y_perm, res, o, (int)T,
                       (int)k, (int)H, (int)E);
  else
    hipLaunchKernelGGL(moe_combine_kernel<64>, dim3(cb), dim3(256), 0, st, top_idx, pos_of, y_perm, res, o, (int)T,
                       (int)k, (int)H, (int)E);
  Q3_LAUNCH_CHECK();
  return Q3_OK;
}

// ------------------------------------------------------------------ training
// The routed experts with a backward, for all experts at once. Rows are the
// (token, slot) entries in expert-major order (P = T k), as the inference path.
//   forward   gu = x[token] . gate_up[e]^T     a = bf16(silu(g) u)
//             out = sum over the token's experts of bf16(bf16(a . down[e]^T) w)
//   backward  dh = dout[token] . down[e]       dw = sum_i dh silu(g) u
//             dgu = swiglu'(g, u) (w dh)       aw = bf16(silu(g) u w)
//             dx[t] = sum over its rows of dgu . gate_up[e]   (fp32, rounded once)
//             dgate_up[e] = dgu_e^T . x[token]_e    ddown[e] = dout[token]_e^T . aw_e
// The products are grouped MFMA GEMMs on the weights as they are stored: dh
// and dxp read an expert's matrix with the reduction as its rows, the weight
// gradients reduce over an expert's row range (gemm_bwd.h). Entries whose id
// lies outside [0, E) (the top-k of a NaN row) have no row: the dispatched
// rows are the first offsets[E] of P, nothing is read of the others. Bound by the
// weights: gate_up and down are read twice and their gradients written once.
// Built as a loop over the experts from the single ops instead, every expert's
// slice gradient filled and added a tensor of all experts: T = 2048, H = 2048,
// I = 768, E = 128, top-8 forward + backward 170 ms, ~6000 launches; here 1.36 ms.
struct MoeTrainState {
  int* offsets;
  int* tile_table;
  int* n_tiles;
  int* sorted_token;
  bf16* sorted_w;
  int* pos_of;
  bf16* gu;  // (P, 2I)
};

int64_t moe_train_state_layout(int64_t T, int64_t I, int64_t E, int64_t k, MoeTrainState* out, char* base) {
  const int64_t P = T * k;
  int64_t off = 0;
  auto take = [&](int64_t bytes) {
    char* p = base ? base + off : nullptr;
    off += align256(bytes);
    return p;
  };
  MoeTrainState w{};
  w.offsets = reinterpret_cast<int*>(take((E + 1) * 4));
  w.tile_table = reinterpret_cast<int*>(take((q3_cdiv(P, kMoeBM) + E) * 4));
  w.n_tiles = reinterpret_cast<int*>(take(4));
  w.sorted_token = reinterpret_cast<int*>(take(P * 4));
  w.sorted_w = reinterpret_cast<bf16*>(take(P * 2));
  w.pos_of = reinterpret_cast<int*>(take(P * 4));
  w.gu = reinterpret_cast<bf16*>(take(P * 2 * I * 2));
  if (out) *out = w;
  return off;
}

// The forward's scratch, then the backward's (never needed at the same time).
struct MoeTrainWs {
  int *hist, *cstart, *counts;
  bf16 *act, *y_perm;                         // forward: (P, I), (P, H)
  bf16 *dh, *dgu, *aw, *dxp, *xg, *dog;       // backward: (P, I), (P, 2I), (P, I), 3 x (P, H)
  float* dw;                                  // backward: (P)
};

int64_t moe_train_ws_layout(int64_t T, int64_t H, int64_t I, int64_t E, int64_t k, bool backward, MoeTrainWs* out,
                            char* base) {
  const int64_t P = T * k;
  int64_t off = 0;
  auto take = [&](int64_t bytes) {
    char* p = base ? base + off : nullptr;
    off += align256(bytes);
    return p;
  };
  MoeTrainWs w{};
  if (!backward) {
    const int64_t NC = q3_cdiv(T, kMoeChunk);
    w.hist = reinterpret_cast<int*>(take(NC * E * 4));
    w.cstart = reinterpret_cast<int*>(take(NC * E * 4));
    w.counts = reinterpret_cast<int*>(take(E * 4));
    w.act = reinterpret_cast<bf16*>(take(P * I * 2));
    w.y_perm = reinterpret_cast<bf16*>(take(P * H * 2));
  } else {
    w.dh = reinterpret_cast<bf16*>(take(P * I * 2));
    w.dgu = reinterpret_cast<bf16*>(take(P * 2 * I * 2));
    w.aw = reinterpret_cast<bf16*>(take(P * I * 2));
    w.dxp = reinterpret_cast<bf16*>(take(P * H * 2));
    w.xg = reinterpret_cast<bf16*>(take(P * H * 2));
    w.dog = reinterpret_cast<bf16*>(take(P * H * 2));
    w.dw = reinterpret_cast<float*>(take(P * 4));
  }
  if (out) *out = w;
  return off;
}

// a = bf16(silu(g) u) of the (P, 2I) gate | up rows, 8 columns per thread.
__device__ __forceinline__ float moe_act(float g, float u) { return g / (1.0f + expf(-g)) * u; }

__global__ __launch_bounds__(256) void moe_act_kernel(const bf16* __restrict__ gu, bf16* __restrict__ act,
                                                      const int* __restrict__ n_rows, int I) {
  const int c8 = I / 8;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)*n_rows * c8) return;
  const int64_t row = i / c8;
  const int c = (int)(i - row * c8) * 8;
  const bf16x8 g = *reinterpret_cast<const bf16x8*>(gu + row * 2 * I + c);
  const bf16x8 u = *reinterpret_cast<const bf16x8*>(gu + row * 2 * I + I + c);
  bf16x8 o;
#pragma unroll
  for (int q = 0; q < 8; ++q) o[q] = f2bf(moe_act(bf2f(g[q]), bf2f(u[q])));
  *reinterpret_cast<bf16x8*>(act + row * I + c) = o;
}

// One wave per row: dgu, aw and dw of the header above.
__global__ __launch_bounds__(256) void moe_act_bwd_kernel(const bf16* __restrict__ gu, const bf16* __restrict__ dh,
                                                          const bf16* __restrict__ sorted_w, bf16* __restrict__ dgu,
                                                          bf16* __restrict__ aw, float* __restrict__ dw,
                                                          const int* __restrict__ n_rows, int I) {
  const int lane = threadIdx.x & 63;
  const int64_t row = ((int64_t)blockIdx.x * 256 + threadIdx.x) >> 6;
  if (row >= *n_rows) return;
  const float w = bf2f(sorted_w[row]);
  float acc = 0.f;
  for (int c = lane * 8; c < I; c += 512) {
    const bf16x8 g8 = *reinterpret_cast<const bf16x8*>(gu + row * 2 * I + c);
    const bf16x8 u8 = *reinterpret_cast<const bf16x8*>(gu + row * 2 * I + I + c);
    const bf16x8 d8 = *reinterpret_cast<const bf16x8*>(dh + row * I + c);
    bf16x8 dg, du, a8;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const float g = bf2f(g8[q]), u = bf2f(u8[q]), d = bf2f(d8[q]);
      const float s = 1.0f / (1.0f + expf(-g));
      const float a = moe_act(g, u);  // unrounded: aw and dw round once, not after the forward's rounding
      acc += d * a;
      a8[q] = f2bf(a * w);
      dg[q] = f2bf(d * w * u * s * (1.0f + g * (1.0f - s)));
      du[q] = f2bf(d * w * g * s);
    }
    *reinterpret_cast<bf16x8*>(dgu + row * 2 * I + c) = dg;
    *reinterpret_cast<bf16x8*>(dgu + row * 2 * I + I + c) = du;
    *reinterpret_cast<bf16x8*>(aw + row * I + c) = a8;
  }
  acc = wave_sum(acc);
  if (lane == 0) dw[row] = acc;
}

// Rows of two (T, H) matrices gathered by the sorted token list: xg = x[token], dog = dout[token].
__global__ __launch_bounds__(256) void moe_gather2_kernel(const bf16* __restrict__ x, const bf16* __restrict__ dout,
                                                          const int* __restrict__ token, bf16* __restrict__ xg,
                                                          bf16* __restrict__ dog, const int* __restrict__ n_rows,
                                                          int H) {
  const int c8 = H / 8;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)*n_rows * c8) return;
  const int64_t row = i / c8;
  const int c = (int)(i - row * c8) * 8;
  const int64_t src = (int64_t)token[row] * H + c, dst = row * H + c;
  const bf16x8 a = *reinterpret_cast<const bf16x8*>(x + src), b = *reinterpret_cast<const bf16x8*>(dout + src);
  *reinterpret_cast<bf16x8*>(xg + dst) = a;
  *reinterpret_cast<bf16x8*>(dog + dst) = b;
}

// dx[t] = the sum of the token's rows of dxp in slot order (fp32, rounded
// once); dtop_w[t, s] = dw of the slot's row. A block per token.
__global__ __launch_bounds__(256) void moe_combine_bwd_kernel(const int* __restrict__ pos_of,
                                                              const bf16* __restrict__ dxp,
                                                              const float* __restrict__ dw, bf16* __restrict__ dx,
                                                              bf16* __restrict__ dtop_w, int64_t P, int k, int H) {
  const int64_t t = blockIdx.x;
  const int* pos = pos_of + t * k;
  if (dtop_w && (int)threadIdx.x < k) {
    const int p = pos[threadIdx.x];
    dtop_w[t * k + threadIdx.x] = f2bf(p >= 0 && p < P ? dw[p] : 0.f);
  }
  if (!dx) return;
  for (int c = threadIdx.x * 8; c < H; c += 256 * 8) {
    float acc[8] = {};
#pragma unroll 8
    for (int s = 0; s < k; ++s) {
      const int p = pos[s];
      if (p < 0 || p >= P) continue;
      const bf16x8 v = *reinterpret_cast<const bf16x8*>(dxp + (int64_t)p * H + c);
#pragma unroll
      for (int q = 0; q < 8; ++q) acc[q] += bf2f(v[q]);
    }
    bf16x8 o;
#pragma unroll
    for (int q = 0; q < 8; ++q) o[q] = f2bf(acc[q]);
    *reinterpret_cast<bf16x8*>(dx + t * H + c) = o;
  }
}

// Grouped product C[row] = X[row or gather[row]] . W[e] over the tile table:
// W[e] (N, K) as stored, or with WT (K, N).
template <int EPI, bool WT>
int launch_grouped(const bf16* X, const bf16* W, bf16* C, const bf16* rowscale, int64_t P, int64_t N, int64_t K,
                   const int* gather, int64_t m_src, const int* tile_table, const int* offsets, const int* n_tiles,
                   int64_t E, hipStream_t st) {
  GemmParams p{};
  p.X = X;
  p.W = W;
  p.C = C;
  p.rowscale = rowscale;
  p.M = (int)P;
  p.N = (int)N;
  p.K = (int)K;
  p.ldx = K;
  p.ldw = WT ? N : K;
  p.ldc = N;
  p.gather = gather;
  p.M_src = (int)m_src;
  p.tile_table = tile_table;
  p.group_end = offsets + 1;
  p.n_tiles_total = n_tiles;
  p.expert_stride_w = N * K;
  const int64_t tiles = (q3_cdiv(P, kMoeBM) + E) * q3_cdiv(N, kMoeBN);
  hipLaunchKernelGGL((gemm_bf16_dma_kernel<kMoeBM, kMoeBN, 2, 4, EPI, true, 2, 64, kMoeNSTW, WT, false, WT>),
                     dim3((unsigned)(q3_cdiv(tiles, 8) * 8)), dim3(512), 0, st, p);
  Q3_LAUNCH_CHECK();
  return Q3_OK;
}

// What the training path takes (the caller keeps the per-expert loop for the rest).
int moe_train_check(int64_t T, int64_t H, int64_t I, int64_t E, int64_t k) {
  Q3_REQUIRE(T >= 0 && H >= 8 && I >= 8 && E >= 1 && k >= 1 && k <= E, Q3_ERR_SHAPE);
  Q3_REQUIRE(H % 8 == 0 && I % 8 == 0 && k <= 32 && E < 2048 && T * k < (1 << 20), Q3_ERR_UNSUPPORTED);
  Q3_REQUIRE((T * k + 512) * std::max(2 * I, H) * 2 < (1ll << 31) && (2 * I + 512) * H * 2 < (1ll << 31),
             Q3_ERR_UNSUPPORTED);
  return Q3_OK;
}

}  // namespace

extern "C" {

// logits (T, E) bf16 -> top_idx (T, k) int32, top_w (T, k) bf16 (renormalised
// when norm != 0), top_p (T, k) fp32 selected probabilities (optional).
int q3_moe_route(const void* logits, int* top_idx, void* top_w, float* top_p, int64_t T, int64_t E, int64_t k,
                 int norm, void* stream) {
  Q3_REQUIRE(logits && top_idx && top_w, Q3_ERR_NULL);
  Q3_REQUIRE(T >= 0 && E >= 1 && k >= 1 && k <= E, Q3_ERR_SHAPE);
  Q3_REQUIRE(E <= 512 && k <= 32, Q3_ERR_UNSUPPORTED);
  if (T == 0) return Q3_OK;
  return launch_route(static_cast<const bf16*>(logits), top_idx, static_cast<bf16*>(top_w), top_p, T, E, k, norm,
                      nullptr, 0, nullptr, static_cast<hipStream_t>(stream));
}

int64_t q3_moe_router_workspace_bytes(int64_t T, int64_t H, int64_t E) {
  if (T <= 0 || H <= 0 || E <= 0) return 0;
  return (int64_t)router_splits(T, H, E) * T * E * 4;
}

int q3_moe_router(const void* x, const void* gate_w, void* logits, int* top_idx, void* top_w, float* top_p,
                  int64_t T, int64_t H, int64_t E, int64_t k, int norm, void* workspace, int64_t workspace_bytes,
                  void* stream) {
  Q3_REQUIRE(x && gate_w && logits && top_idx && top_w, Q3_ERR_NULL);
  Q3_REQUIRE(T >= 0 && H >= 1 && E >= 1 && k >= 1 && k <= E, Q3_ERR_SHAPE);
  Q3_REQUIRE(E <= 512 && k <= 32, Q3_ERR_UNSUPPORTED);
  Q3_REQUIRE(H % 8 == 0 && q3_aligned(x, 16) && q3_aligned(gate_w, 16), Q3_ERR_ALIGN);
  Q3_REQUIRE(T * H * 2 < 0x7fffffffLL && E * H * 2 < 0x7fffffffLL, Q3_ERR_UNSUPPORTED);
  if (T == 0) return Q3_OK;
  const int ns = router_splits(T, H, E);
  const int64_t ks = H / ns;
  Q3_REQUIRE(workspace != nullptr && workspace_bytes >= (int64_t)ns * T * E * 4, Q3_ERR_WORKSPACE);
  Q3_REQUIRE(q3_aligned(workspace, 16), Q3_ERR_ALIGN);
  hipStream_t st = static_cast<hipStream_t>(stream);
  // Split z: X and W columns [z ks, (z + 1) ks) -> fp32 plane z of (T, E).
  GemmParams p{};
  p.X = static_cast<const bf16*>(x);
  p.W = static_cast<const bf16*>(gate_w);
  p.C = static_cast<bf16*>(workspace);
  p.M = (int)T;
  p.N = (int)E;
  p.K = (int)ks;
  p.ldx = H;
  p.ldw = H;
  p.ldc = E;
  p.bsX = ks;
  p.bsW = ks;
  p.bsC = T * E;
  p.group_m = 8;
  p.seg.n = 1;
  p.seg.w[0] = p.W;
  const int64_t tiles = q3_cdiv(T, 128) * q3_cdiv(E, 128);
  hipLaunchKernelGGL((gemm_bf16_dma_kernel<128, 128, 2, 2, kEpiStoreF32, false, 4, 64, 5>),
                     dim3((unsigned)tiles, 1, (unsigned)ns), dim3(256), 0, st, p);
  Q3_LAUNCH_CHECK();
  return launch_route(static_cast<const bf16*>(logits), top_idx, static_cast<bf16*>(top_w), top_p, T, E, k, norm,
                      static_cast<const float*>(workspace), ns, static_cast<bf16*>(logits), st);
}

int64_t q3_moe_experts_workspace_bytes(int64_t T, int64_t H, int64_t I, int64_t E, int64_t k) {
  if (T <= 0 || H <= 0 || I <= 0 || E <= 0 || k <= 0) return 0;
  return moe_ws_layout(T, H, I, E, k, nullptr, nullptr);
}

// x (T, H) bf16; gate_up (E, 2I, H); down (E, H, I); top_idx (T, k) int32;
// top_w (T, k) bf16; out (T, H) bf16 = sum over the token's experts of
// w * down(swiglu(gate_up x)) (+ residual (T, H) when given).
int q3_moe_experts(const void* x, const void* gate_up, const void* down, const int* top_idx, const void* top_w,
                   const void* residual, void* out, int64_t T, int64_t H, int64_t I, int64_t E, int64_t k,
                   void* workspace, int64_t workspace_bytes, void* stream) {
  Q3_REQUIRE(x && gate_up && down && top_idx && top_w && out, Q3_ERR_NULL);
  Q3_REQUIRE(T >= 0 && H >= 8 && I >= 8 && E >= 1 && k >= 1 && k <= E, Q3_ERR_SHAPE);
  Q3_REQUIRE(H % 8 == 0 && I % 8 == 0 && k <= 32 && E < 2048 && T * k < (1 << 20), Q3_ERR_UNSUPPORTED);
  Q3_REQUIRE(q3_aligned(x, 16) && q3_aligned(gate_up, 16) && q3_aligned(down, 16) && q3_aligned(out, 16) &&
                 (!residual || q3_aligned(residual, 16)),
             Q3_ERR_ALIGN);
  if (T == 0) return Q3_OK;
  Q3_REQUIRE(workspace && workspace_bytes >= q3_moe_experts_workspace_bytes(T, H, I, E, k), Q3_ERR_WORKSPACE);
  hipStream_t st = static_cast<hipStream_t>(stream);
  MoeWs w{};
  moe_ws_layout(T, H, I, E, k, &w, static_cast<char*>(workspace));
  const int64_t P = T * k;
  const int64_t max_tiles = q3_cdiv(P, kMoeBM) + E;
  if (moe_small(T, H, I, k)) {  // decode: the weights as an even stream
    hipLaunchKernelGGL(moe_dispatch_small_kernel, dim3(1), dim3(kSmallP), 2 * (E + 1) * sizeof(int), st,
                       top_idx, static_cast<const bf16*>(top_w), (int)P, (int)k, (int)E, w);
    Q3_LAUNCH_CHECK();
    MoeGemvP g{static_cast<const bf16*>(x), static_cast<const bf16*>(gate_up), nullptr, w.act, w.sorted_token,
               w.chunk_table, w.n_chunks, w.offsets, (int)I, (int)H, (int)H, (int)T};
    int rc = launch_moe_gemv<true>(g, st);
    if (rc != Q3_OK) return rc;
    g = {w.act, static_cast<const bf16*>(down), w.sorted_w, w.y_perm, nullptr, w.chunk_table, w.n_chunks, w.offsets,
         (int)H, (int)I, (int)I, (int)P};
    if ((rc = launch_moe_gemv<false>(g, st)) != Q3_OK) return rc;
    return launch_combine(top_idx, w.pos_of, w.y_perm, static_cast<const bf16*>(residual), static_cast<bf16*>(out), T,
                          H, E, k, st);
  }
  {
    const int rc = moe_dispatch(top_idx, static_cast<const bf16*>(top_w), T, k, E, w, st);
    if (rc != Q3_OK) return rc;
  }

  // GEMM 1: act[pos] = swiglu(x[token(pos)] . gate_up[e]^T)
  {
    GemmParams p{};
    p.X = static_cast<const bf16*>(x);
    p.W = static_cast<const bf16*>(gate_up);           // gate rows [0, I)
    p.W2 = static_cast<const bf16*>(gate_up) + I * H;  // up rows [I, 2I)
    p.C = w.act;
    p.M = (int)P;
    p.N = (int)I;
    p.K = (int)H;
    p.ldx = H;
    p.ldw = H;
    p.ldc = I;
    p.gather = w.sorted_token;
    p.M_src = (int)T;
    p.tile_table = w.tile_table;
    p.group_end = w.offsets + 1;
    p.n_tiles_total = w.n_tiles;
    p.expert_stride_w = 2 * I * H;
    const int64_t ntn = q3_cdiv(I, kMoeBN / 2);
    // Grid: a multiple of 8 (the kernel deals the valid tiles out per XCD).
    hipLaunchKernelGGL((gemm_bf16_dma_kernel<kMoeBM, kMoeBN, 2, 4, kEpiSwiGLU, true, 2, 64, kMoeNSTW>),
                       dim3((unsigned)(q3_cdiv(max_tiles * ntn, 8) * 8)),
                       dim3(512), 0, st, p);
    Q3_LAUNCH_CHECK();
  }
  // GEMM 2: y_perm[pos] = bf16(bf16(act[pos] . down[e]^T) * w[pos])
  {
    GemmParams p{};
    p.X = w.act;
    p.W = static_cast<const bf16*>(down);
    p.C = w.y_perm;
    p.rowscale = w.sorted_w;
    p.M = (int)P;
    p.N = (int)H;
    p.K = (int)I;
    p.ldx = I;
    p.ldw = I;
    p.ldc = H;
    p.gather = nullptr;
    p.tile_table = w.tile_table;
    p.group_end = w.offsets + 1;
    p.n_tiles_total = w.n_tiles;
    p.expert_stride_w = H * I;
    const int64_t ntn = q3_cdiv(H, kMoeBN);
    hipLaunchKernelGGL((gemm_bf16_dma_kernel<kMoeBM, kMoeBN, 2, 4, kEpiRowScale, true, 2, 64, kMoeNSTW>),
                       dim3((unsigned)(q3_cdiv(max_tiles * ntn, 8) * 8)), dim3(512), 0, st, p);
    Q3_LAUNCH_CHECK();
  }
  return launch_combine(top_idx, w.pos_of, w.y_perm, static_cast<const bf16*>(residual), static_cast<bf16*>(out), T, H,
                        E, k, st);
}

int64_t q3_moe_train_state_bytes(int64_t T, int64_t H, int64_t I, int64_t E, int64_t k) {
  if (T <= 0 || moe_train_check(T, H, I, E, k) != Q3_OK) return 0;
  return moe_train_state_layout(T, I, E, k, nullptr, nullptr);
}

int64_t q3_moe_train_workspace_bytes(int64_t T, int64_t H, int64_t I, int64_t E, int64_t k, int backward) {
  if (T <= 0 || moe_train_check(T, H, I, E, k) != Q3_OK) return 0;
  return moe_train_ws_layout(T, H, I, E, k, backward != 0, nullptr, nullptr);
}

int q3_moe_train_forward(const void* x, const void* gate_up, const void* down, const int* top_idx, const void* top_w,
                         void* out, int64_t T, int64_t H, int64_t I, int64_t E, int64_t k, void* state,
                         int64_t state_bytes, void* workspace, int64_t workspace_bytes, void* stream) {
  Q3_REQUIRE(x && gate_up && down && top_idx && top_w && out, Q3_ERR_NULL);
  int rc = moe_train_check(T, H, I, E, k);
  if (rc != Q3_OK) return rc;
  Q3_REQUIRE(q3_aligned(x, 16) && q3_aligned(gate_up, 16) && q3_aligned(down, 16) && q3_aligned(out, 16), Q3_ERR_ALIGN);
  if (T == 0) return Q3_OK;
  Q3_REQUIRE(state && state_bytes >= q3_moe_train_state_bytes(T, H, I, E, k) && workspace &&
                 workspace_bytes >= q3_moe_train_workspace_bytes(T, H, I, E, k, 0),
             Q3_ERR_WORKSPACE);
  Q3_REQUIRE(q3_aligned(state, 256) && q3_aligned(workspace, 256), Q3_ERR_ALIGN);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t P = T * k;
  MoeTrainState s{};
  MoeTrainWs w{};
  moe_train_state_layout(T, I, E, k, &s, static_cast<char*>(state));
  moe_train_ws_layout(T, H, I, E, k, false, &w, static_cast<char*>(workspace));
  MoeWs d{};
  d.hist = w.hist;
  d.cstart = w.cstart;
  d.counts = w.counts;
  d.offsets = s.offsets;
  d.tile_table = s.tile_table;
  d.n_tiles = s.n_tiles;
  d.sorted_token = s.sorted_token;
  d.sorted_w = s.sorted_w;
  d.pos_of = s.pos_of;
  if ((rc = moe_dispatch(top_idx, static_cast<const bf16*>(top_w), T, k, E, d, st, true)) != Q3_OK) return rc;
  if ((rc = launch_grouped<kEpiStore, false>(static_cast<const bf16*>(x), static_cast<const bf16*>(gate_up), s.gu,
                                             nullptr, P, 2 * I, H, s.sorted_token, T, s.tile_table, s.offsets,
                                             s.n_tiles, E, st)) != Q3_OK)
    return rc;
  hipLaunchKernelGGL(moe_act_kernel, dim3((unsigned)q3_cdiv(P * (I / 8), 256)), dim3(256), 0, st, s.gu, w.act,
                     s.offsets + E, (int)I);
  Q3_LAUNCH_CHECK();
  if ((rc = launch_grouped<kEpiRowScale, false>(w.act, static_cast<const bf16*>(down), w.y_perm, s.sorted_w, P, H, I,
                                                nullptr, 0, s.tile_table, s.offsets, s.n_tiles, E, st)) != Q3_OK)
    return rc;
  return launch_combine(top_idx, s.pos_of, w.y_perm, nullptr, static_cast<bf16*>(out), T, H, E, k, st);
}

int q3_moe_train_backward(const void* x, const void* gate_up, const void* down, const void* grad_out, void* grad_x,
                          void* grad_gate_up, void* grad_down, void* grad_top_w, int64_t T, int64_t H, int64_t I,
                          int64_t E, int64_t k, const void* state, int64_t state_bytes, void* workspace,
                          int64_t workspace_bytes, void* stream) {
  Q3_REQUIRE(x && gate_up && down && grad_out, Q3_ERR_NULL);
  int rc = moe_train_check(T, H, I, E, k);
  if (rc != Q3_OK) return rc;
  Q3_REQUIRE(q3_aligned(x, 16) && q3_aligned(gate_up, 16) && q3_aligned(down, 16) && q3_aligned(grad_out, 16) &&
                 q3_aligned(grad_x, 16) && q3_aligned(grad_gate_up, 16) && q3_aligned(grad_down, 16),
             Q3_ERR_ALIGN);
  if (T == 0) return Q3_OK;
  Q3_REQUIRE(state && state_bytes >= q3_moe_train_state_bytes(T, H, I, E, k) && workspace &&
                 workspace_bytes >= q3_moe_train_workspace_bytes(T, H, I, E, k, 1),
             Q3_ERR_WORKSPACE);
  Q3_REQUIRE(q3_aligned(state, 256) && q3_aligned(workspace, 256), Q3_ERR_ALIGN);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t P = T * k;
  MoeTrainState s{};
  MoeTrainWs w{};
  moe_train_state_layout(T, I, E, k, &s, static_cast<char*>(const_cast<void*>(state)));
  moe_train_ws_layout(T, H, I, E, k, true, &w, static_cast<char*>(workspace));
  const bf16* dout = static_cast<const bf16*>(grad_out);
  if ((rc = launch_grouped<kEpiStore, true>(dout, static_cast<const bf16*>(down), w.dh, nullptr, P, I, H,
                                            s.sorted_token, T, s.tile_table, s.offsets, s.n_tiles, E, st)) != Q3_OK)
    return rc;
  hipLaunchKernelGGL(moe_act_bwd_kernel, dim3((unsigned)q3_cdiv(P, 4)), dim3(256), 0, st, s.gu, w.dh, s.sorted_w,
                     w.dgu, w.aw, w.dw, s.offsets + E, (int)I);
  Q3_LAUNCH_CHECK();
  if (grad_x) {
    if ((rc = launch_grouped<kEpiStore, true>(w.dgu, static_cast<const bf16*>(gate_up), w.dxp, nullptr, P, H, 2 * I,
                                              nullptr, 0, s.tile_table, s.offsets, s.n_tiles, E, st)) != Q3_OK)
      return rc;
  }
  if (grad_x || grad_top_w) {
    hipLaunchKernelGGL(moe_combine_bwd_kernel, dim3((unsigned)T), dim3(256), 0, st, s.pos_of, w.dxp, w.dw,
                       static_cast<bf16*>(grad_x), static_cast<bf16*>(grad_top_w), P, (int)k, (int)H);
    Q3_LAUNCH_CHECK();
  }
  if (grad_gate_up || grad_down) {
    hipLaunchKernelGGL(moe_gather2_kernel, dim3((unsigned)q3_cdiv(P * (H / 8), 256)), dim3(256), 0, st,
                       static_cast<const bf16*>(x), dout, s.sorted_token, w.xg, w.dog, s.offsets + E, (int)H);
    Q3_LAUNCH_CHECK();
  }
  if (grad_gate_up) {
    if ((rc = q3::gemm_tn_ranges(w.dgu, w.xg, grad_gate_up, 2 * I, H, P, s.offsets, E, st)) != Q3_OK) return rc;
  }
  if (grad_down) return q3::gemm_tn_ranges(w.dog, w.aw, grad_down, H, I, P, s.offsets, E, st);
  return Q3_OK;
}

int64_t q3_moe_permute_workspace_bytes(int64_t T, int64_t E, int64_t k) {
  if (T <= 0 || E <= 0 || k <= 0) return 0;
  return moe_permute_ws_layout(T, E, k, nullptr, nullptr);
}

// The dispatch of q3_moe_experts on its own: offsets (E + 1) int32,
// sorted_token / sorted_w (T * k) (int32 / bf16) and pos_of (T, k) int32.
int q3_moe_permute(const int* top_idx, const void* top_w, int* offsets, int* sorted_token, void* sorted_w,
                   int* pos_of, int64_t T, int64_t E, int64_t k, void* workspace, int64_t workspace_bytes,
                   void* stream) {
  Q3_REQUIRE(top_idx && top_w && offsets && sorted_token && sorted_w && pos_of, Q3_ERR_NULL);
  Q3_REQUIRE(T >= 0 && E >= 1 && k >= 1 && k <= E, Q3_ERR_SHAPE);
  Q3_REQUIRE(k <= 32 && E < 2048 && T * k < (1 << 20), Q3_ERR_UNSUPPORTED);
  if (T == 0) return Q3_OK;
  Q3_REQUIRE(workspace && workspace_bytes >= q3_moe_permute_workspace_bytes(T, E, k), Q3_ERR_WORKSPACE);
  MoeWs w{};
  moe_permute_ws_layout(T, E, k, &w, static_cast<char*>(workspace));
  w.offsets = offsets;
  w.sorted_token = sorted_token;
  w.sorted_w = static_cast<bf16*>(sorted_w);
  w.pos_of = pos_of;
  return moe_dispatch(top_idx, static_cast<const bf16*>(top_w), T, k, E, w, static_cast<hipStream_t>(stream));
}

int64_t q3_index_add_workspace_bytes(int64_t n_src, int64_t n_target) {
  if (n_src < 0 || n_target < 0) return 0;
  return (3 * n_target + 1 + n_src + 1) * (int64_t)sizeof(int);
}

// target (n_target, D) += rows of src (n_src, D) at idx (n_src) int64, in place.
// Source rows whose index is outside [0, n_target) are skipped, and bit 0 of
// *status (a device int, when given) is set: the check costs the host nothing.
int q3_index_add(void* target, const void* src, const int64_t* idx, int64_t n_src, int64_t n_target, int64_t D,
                 int dtype, void* workspace, int64_t workspace_bytes, int* status, void* stream) {
  Q3_REQUIRE(target && (src || n_src == 0) && (idx || n_src == 0), Q3_ERR_NULL);
  Q3_REQUIRE(n_src >= 0 && n_target >= 0 && D >= 0, Q3_ERR_SHAPE);
  Q3_REQUIRE(n_src < (1ll << 31) && n_target < (1ll << 31), Q3_ERR_UNSUPPORTED);
  if (n_src == 0 || n_target == 0 || D == 0) return Q3_OK;
  Q3_REQUIRE(workspace && workspace_bytes >= q3_index_add_workspace_bytes(n_src, n_target), Q3_ERR_WORKSPACE);
  hipStream_t st = static_cast<hipStream_t>(stream);
  char* ws = static_cast<char*>(workspace);
  if (dtype == Q3_BF16) return index_add_t<bf16>(target, src, idx, n_src, n_target, D, ws, status, st);
  if (dtype == Q3_F32) return index_add_t<float>(target, src, idx, n_src, n_target, D, ws, status, st);
  return Q3_ERR_DTYPE;
}

}  // extern "C"
