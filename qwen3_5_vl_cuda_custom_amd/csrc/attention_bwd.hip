// Flash-attention backward (replaces flash_attention_backward of
// csrc/flash_attention_op.cpp:15, csrc/flash_attention_op.cu:235-390): the
// gradients of O = softmax(scale * Q K^T [+ causal mask]) V with GQA, from the
// forward's row log-sum-exp, without materialising the attention matrix.
//
//   Dv[i]   = sum_d dO[i, d] O[i, d]
//   P[i, j] = exp(scale * q_i . k_j - lse[i])        (0 where masked)
//   dV[j]  += P[i, j] dO[i]           dP[i, j] = dO[i] . v_j
//   dS[i, j] = P[i, j] (dP[i, j] - Dv[i])
//   dK[j]  += scale * dS[i, j] q_i    dQ[i]  += scale * dS[i, j] k_j
//
// Two passes keep every sum in a fixed order (no atomics, bitwise reproducible
// results): a key-parallel kernel owns 64 keys of one KV head and walks the
// query rows of all the query heads that share the KV head (GQA), summing dK
// and dV in registers; a query-parallel kernel owns 64 query rows and walks
// the keys, summing dQ. Both recompute P from Q, K and the log-sum-exp. Four
// lanes share a row (key or query), a quarter of its dims each (consecutive ones,
// so a lane reads the staged rows by 16-byte LDS loads), dot products are
// summed over the four lanes with two shuffles. fp32 math for bf16 and fp32
// tensors; head_dim up to 128. The causal mask is top-left aligned (query i
// sees keys 0..i), as the forward's.
//
// bf16 tensors of the forward's MFMA head dims run the same two passes on the
// matrix cores (namespace bmf below); fp32 tensors and other head dims run the
// SIMT kernels that come first.
#include "gemm_tile.h"
#include "q3_common.h"

namespace {

constexpr int kBT = 256;      // threads per block
constexpr int kRowsPB = 64;   // keys (dK/dV) or queries (dQ) per block: 4 lanes each
constexpr int kTile = 16;     // rows of the other side staged in LDS per step
constexpr int kIlp = 2;       // rows of a step in flight per thread: with the 16-byte LDS reads, batch 4, 4 / 2 heads,
                              // 512 x 64 fp32 903 -> 752 us (797 with one row, 747 with 4 rows, which spill nothing
                              // but cost occupancy: 2 x 1024 tokens of 128 5036, 4875, 5141 us for 1, 2, 4)
constexpr int kMaxD = 128;
// Whether a last, partial tile takes all kTile steps (rows past the end are not live). Its own rows only, in a second
// loop: 33 rows of 40 dims 49 -> 38 us, 500 of 64 458 -> 425; with 24 dims per lane the second loop costs more than
// it saves (400 rows of 72 543 -> 561).
template <int DS>
constexpr bool kWholeTiles = DS == 24;

struct BwdParams {
  const void *q, *k, *v, *o, *dout;
  const float* lse;
  float* dvec;
  void *dq, *dk, *dv;
  int B, Hq, Hkv, Sq, Sk, D, groups;
  float scale;
  int causal;
};

__device__ __forceinline__ float quad_sum(float v) {
  v += __shfl_xor(v, 1, 64);
  v += __shfl_xor(v, 2, 64);
  return v;
}

// Dv[row] = dO[row] . O[row], one wave per row.
template <typename T>
__global__ __launch_bounds__(kBT) void attn_bwd_dvec_kernel(const BwdParams p, int64_t rows) {
  const int lane = threadIdx.x & 63;
  const int64_t row = ((int64_t)blockIdx.x * kBT + threadIdx.x) >> 6;
  if (row >= rows) return;
  const T* o = static_cast<const T*>(p.o) + row * p.D;
  const T* g = static_cast<const T*>(p.dout) + row * p.D;
  float acc = 0.f;
  for (int d = lane; d < p.D; d += 64) acc += to_f<T>(o[d]) * to_f<T>(g[d]);
  acc = wave_sum(acc);
  if (lane == 0) p.dvec[row] = acc;
}

// dK, dV: block (key tile, b * Hkv + kv head).
template <typename T, int DS>
__global__ __launch_bounds__(kBT) void attn_bwd_dkdv_kernel(const BwdParams p) {
  constexpr int kDP = 4 * DS;  // staged row width: D rounded up to the four lanes' dims
  static_assert(kDP <= kMaxD, "head_dim <= 128");
  __shared__ float s_q[kTile][kMaxD];
  __shared__ float s_do[kTile][kMaxD];
  __shared__ float s_lse[kTile], s_dv[kTile];
  const int tid = threadIdx.x, part = tid & 3;
  const int bh = blockIdx.y, b = bh / p.Hkv, kvh = bh % p.Hkv;
  const int j0 = blockIdx.x * kRowsPB;
  const int j = j0 + (tid >> 2);
  const int D = p.D;
  const bool jv = j < p.Sk;
  const int64_t kv_base = ((int64_t)b * p.Hkv + kvh) * p.Sk;
  const T* kp = static_cast<const T*>(p.k) + (kv_base + (jv ? j : 0)) * D;
  const T* vp = static_cast<const T*>(p.v) + (kv_base + (jv ? j : 0)) * D;
  float kr[DS], vr[DS], dk[DS], dv[DS];
#pragma unroll
  for (int t = 0; t < DS; ++t) {
    const int d = part * DS + t;
    kr[t] = (jv && d < D) ? to_f<T>(kp[d]) : 0.f;
    vr[t] = (jv && d < D) ? to_f<T>(vp[d]) : 0.f;
    dk[t] = 0.f;
    dv[t] = 0.f;
  }
  const int i_begin = p.causal ? j0 : 0;          // no earlier query sees any of the block's keys
  for (int g = 0; g < p.groups; ++g) {
    const int h = kvh * p.groups + g;
    const int64_t q_base = ((int64_t)b * p.Hq + h) * p.Sq;
    for (int i0 = i_begin; i0 < p.Sq; i0 += kTile) {
      __syncthreads();  // the previous tile's readers are done
      // rows past Sq and dims in [D, 4 * DS) are staged as zeros (every word a lane reads is written)
      for (int e = tid; e < kTile * kDP; e += kBT) {
        const int r = e / kDP, d = e % kDP, i = i0 + r;
        const bool ok = i < p.Sq && d < D;
        s_q[r][d] = ok ? to_f<T>(static_cast<const T*>(p.q)[(q_base + i) * D + d]) : 0.f;
        s_do[r][d] = ok ? to_f<T>(static_cast<const T*>(p.dout)[(q_base + i) * D + d]) : 0.f;
      }
      if (tid < kTile) {
        const int i = i0 + tid;
        s_lse[tid] = i < p.Sq ? p.lse[q_base + i] : 0.f;
        s_dv[tid] = i < p.Sq ? p.dvec[q_base + i] : 0.f;
      }
      __syncthreads();
      // kIlp rows at a time: their dot products, exchanges and exponentials are independent chains
      auto rows = [&](int r0) {
        float s[kIlp], dp[kIlp];
#pragma unroll
        for (int u = 0; u < kIlp; ++u) {
          s[u] = dp[u] = 0.f;
#pragma unroll
          for (int t = 0; t < DS; ++t) {
            s[u] += s_q[r0 + u][part * DS + t] * kr[t];
            dp[u] += s_do[r0 + u][part * DS + t] * vr[t];
          }
        }
#pragma unroll
        for (int u = 0; u < kIlp; ++u) {
          s[u] = quad_sum(s[u]);
          dp[u] = quad_sum(dp[u]);
        }
#pragma unroll
        for (int u = 0; u < kIlp; ++u) {
          const int r = r0 + u, i = i0 + r;
          const bool live = jv && i < p.Sq && (!p.causal || j <= i);
          const float pr = live ? expf(p.scale * s[u] - s_lse[r]) : 0.f;
          const float ds = pr * (dp[u] - s_dv[r]);
#pragma unroll
          for (int t = 0; t < DS; ++t) {
            dv[t] += pr * s_do[r][part * DS + t];
            dk[t] += ds * s_q[r][part * DS + t];
          }
        }
      };
      if (kWholeTiles<DS> || p.Sq - i0 >= kTile)
        for (int r0 = 0; r0 < kTile; r0 += kIlp) rows(r0);
      else
        for (int r0 = 0; r0 < p.Sq - i0; r0 += kIlp) rows(r0);
    }
  }
  if (!jv) return;
  T* dkp = static_cast<T*>(p.dk) + (kv_base + j) * D;
  T* dvp = static_cast<T*>(p.dv) + (kv_base + j) * D;
#pragma unroll
  for (int t = 0; t < DS; ++t) {
    const int d = part * DS + t;
    if (d < D) {
      dkp[d] = from_f<T>(dk[t] * p.scale);
      dvp[d] = from_f<T>(dv[t]);
    }
  }
}

// dQ: block (query tile, b * Hq + head).
template <typename T, int DS>
__global__ __launch_bounds__(kBT) void attn_bwd_dq_kernel(const BwdParams p) {
  constexpr int kDP = 4 * DS;
  static_assert(kDP <= kMaxD, "head_dim <= 128");
  __shared__ float s_k[kTile][kMaxD];
  __shared__ float s_v[kTile][kMaxD];
  const int tid = threadIdx.x, part = tid & 3;
  const int bh = blockIdx.y, b = bh / p.Hq, h = bh % p.Hq;
  const int kvh = h / p.groups;
  const int i0 = blockIdx.x * kRowsPB;
  const int i = i0 + (tid >> 2);
  const int D = p.D;
  const bool iv = i < p.Sq;
  const int64_t q_row = ((int64_t)b * p.Hq + h) * p.Sq + (iv ? i : 0);
  const T* qp = static_cast<const T*>(p.q) + q_row * D;
  const T* gp = static_cast<const T*>(p.dout) + q_row * D;
  float qr[DS], gr[DS], dq[DS];
#pragma unroll
  for (int t = 0; t < DS; ++t) {
    const int d = part * DS + t;
    qr[t] = (iv && d < D) ? to_f<T>(qp[d]) : 0.f;
    gr[t] = (iv && d < D) ? to_f<T>(gp[d]) : 0.f;
    dq[t] = 0.f;
  }
  const float lse = iv ? p.lse[q_row] : 0.f;
  const float dvi = iv ? p.dvec[q_row] : 0.f;
  const int64_t kv_base = ((int64_t)b * p.Hkv + kvh) * p.Sk;
  // keys past the block's last query are masked for every row of the block
  const int j_end = p.causal ? min(p.Sk, min(i0 + kRowsPB, p.Sq)) : p.Sk;
  for (int j0 = 0; j0 < j_end; j0 += kTile) {
    __syncthreads();
    for (int e = tid; e < kTile * kDP; e += kBT) {
      const int r = e / kDP, d = e % kDP, j = j0 + r;
      const bool ok = j < p.Sk && d < D;
      s_k[r][d] = ok ? to_f<T>(static_cast<const T*>(p.k)[(kv_base + j) * D + d]) : 0.f;
      s_v[r][d] = ok ? to_f<T>(static_cast<const T*>(p.v)[(kv_base + j) * D + d]) : 0.f;
    }
    __syncthreads();
    auto rows = [&](int r0) {
      float s[kIlp], dp[kIlp];
#pragma unroll
      for (int u = 0; u < kIlp; ++u) {
        s[u] = dp[u] = 0.f;
#pragma unroll
        for (int t = 0; t < DS; ++t) {
          s[u] += qr[t] * s_k[r0 + u][part * DS + t];
          dp[u] += gr[t] * s_v[r0 + u][part * DS + t];
        }
      }
#pragma unroll
      for (int u = 0; u < kIlp; ++u) {
        s[u] = quad_sum(s[u]);
        dp[u] = quad_sum(dp[u]);
      }
#pragma unroll
      for (int u = 0; u < kIlp; ++u) {
        const int r = r0 + u, j = j0 + r;
        const bool live = iv && j < j_end && (!p.causal || j <= i);
        const float pr = live ? expf(p.scale * s[u] - lse) : 0.f;
        const float ds = pr * (dp[u] - dvi);
#pragma unroll
        for (int t = 0; t < DS; ++t) dq[t] += ds * s_k[r][part * DS + t];
      }
    };
    if (kWholeTiles<DS> || j_end - j0 >= kTile)
      for (int r0 = 0; r0 < kTile; r0 += kIlp) rows(r0);
    else
      for (int r0 = 0; r0 < j_end - j0; r0 += kIlp) rows(r0);
  }
  if (!iv) return;
  T* dqp = static_cast<T*>(p.dq) + q_row * D;
#pragma unroll
  for (int t = 0; t < DS; ++t) {
    const int d = part * DS + t;
    if (d < D) dqp[d] = from_f<T>(dq[t] * p.scale);
  }
}

template <typename T, int DS>
int attn_bwd_t(const BwdParams& p, hipStream_t st) {
  const int64_t rows = (int64_t)p.B * p.Hq * p.Sq;
  hipLaunchKernelGGL(attn_bwd_dvec_kernel<T>, dim3((unsigned)q3_cdiv(rows, kBT / 64)), dim3(kBT), 0, st, p, rows);
  Q3_LAUNCH_CHECK();
  if (p.Sk > 0) {
    hipLaunchKernelGGL((attn_bwd_dkdv_kernel<T, DS>), dim3((unsigned)q3_cdiv(p.Sk, kRowsPB), (unsigned)(p.B * p.Hkv)),
                       dim3(kBT), 0, st, p);
    Q3_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL((attn_bwd_dq_kernel<T, DS>), dim3((unsigned)q3_cdiv(p.Sq, kRowsPB), (unsigned)(p.B * p.Hq)),
                     dim3(kBT), 0, st, p);
  Q3_LAUNCH_CHECK();
  return Q3_OK;
}

template <typename T>
int attn_bwd_d(const BwdParams& p, hipStream_t st) {
  if (p.D <= 32) return attn_bwd_t<T, 8>(p, st);
  if (p.D <= 64) return attn_bwd_t<T, 16>(p, st);
  if (p.D <= 96) return attn_bwd_t<T, 24>(p, st);
  return attn_bwd_t<T, 32>(p, st);
}

// ----------------------------------------------------------------- MFMA (bf16)
// A block is 4 waves of 32 rows of its own side (keys for dK/dV, queries for
// dQ) that share 32-row tiles of the other side through an LDS ring filled by
// direct-to-LDS loads. A wave keeps its rows' operands as B fragments in
// registers and forms, per tile, S and dP with the tile's rows as A operand:
// lane l then holds column l % 32 (its own row) and registers the tile's rows,
// so P and dS go straight from the accumulators into the B operand of the
// second products, whose A operand (dO^T, Q^T or K^T) is read transposed by
// ds_read_b64_tr_b16 in the same row order:
//   dkdv:  dV^T += dO^T P,  dK^T += Q^T dS      (rows of Q and dO per tile)
//   dq:    dQ^T += K^T dS^T                     (rows of K and V per tile)
// P and dS stay 32-bit values: each is split into two bf16 terms, hi = bf16(x)
// and lo = bf16(x - hi) (P: hi cut downwards), and the second products run once
// per term into the same fp32 accumulator. hi + lo carries 16 significant bits,
// so what the split drops (2^-17 of each term, P 2^-16) is far below the one
// rounding of the bf16 outputs (2^-9); a single bf16 term would not be. The
// gradients' distance to float64 equals the SIMT kernels' to four digits (dq,
// dk, dv at S = 2048, D = 128: 0.00204, 0.00198, 0.00166). Infinities in dO stay
// infinities, see split8.
//
// LDS rows are 128 elements whatever D is; chunk c (16 bytes) of row r sits at
// slot c ^ swz(r) with swz(r) = the two bit pairs of r % 16 swapped: 16
// consecutive rows take 16 distinct slots (the row fragment reads) and rows
// 4 i .. 4 i + 3 fall into distinct 64-byte quarters (the transposed reads),
// so one copy of a tile serves both without bank conflicts. Chunks at or past
// D load as zeros.
//
// What bounds it: per 32 x 32 tile a dkdv wave issues 16 + 4 OT x 2 MFMAs (48
// at D = 128, 1536 cycles) beside ~200 VALU operations (exponentials, the
// splits); two waves per SIMD (<= 256 registers) let one wave's MFMAs run
// under the other's VALU work. Measured against the SIMT kernels: causal
// S = 2048, 32 / 8 heads of 128: dK/dV 8797 -> 169 us, dQ 4447 -> 113 us;
// 4 x 784 patches, 16 heads of 72: 1588 -> 69 and 843 -> 50 us.
namespace bmf {

constexpr int kRow = 128;             // elements per LDS row
constexpr int kT32 = 32;              // rows per tile
constexpr int kTileE = kT32 * kRow;   // elements per tile
constexpr int kStg = 4;               // ring depth: tile t + 3 is requested in step t
constexpr int kOwn = 128;             // own-side rows per block (4 waves of 32)
constexpr float kLog2e = 1.4426950408889634f;

typedef short short4v __attribute__((ext_vector_type(4)));
typedef short short8v __attribute__((ext_vector_type(8)));

__device__ __forceinline__ int swz(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }
__device__ __forceinline__ int off(int r, int c) { return r * kRow + ((c ^ swz(r)) << 3); }

__device__ __forceinline__ short4v read_tr16(const bf16* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (short4v __attribute__((address_space(3)))*)(reinterpret_cast<uintptr_t>(p)));
}

// 4 bytes per lane from the buffer at `voff` into LDS at `lds_byte` + 4 * lane.
__device__ __forceinline__ void dma4(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t lds_byte) {
  const uint32_t m0v = __builtin_amdgcn_readfirstlane(lds_byte);
  asm volatile("s_mov_b32 m0, %1\n\tbuffer_load_dword %0, %2, 0 offen lds" ::"v"(voff), "s"(m0v), "s"(r)
               : "memory");
}

struct Str {
  int64_t b, h, s;  // element strides of (batch, head, row); rows are contiguous
};

struct P {
  const bf16 *q, *k, *v, *o, *dout;
  const float* lse;
  float* stats;   // (B * Hq, n_qt, 64): per 32-query tile the rows' lse * log2(e), then their Dv
  float* part;    // hs > 1: fp32 partials (hs, 2, B * Hkv, Sk, D): dK then dV of each head split
  bf16 *dq, *dk, *dv;
  int B, Hq, Hkv, Sq, Sk, groups, n_qt, hs;
  float scale, scale_log2;
  int causal;
  Str sq, sk, sv, so, sg, sdq, sdk, sdv;  // q, k, v, o, dout and the gradients
};

// Blocks in order of falling work (causal), dealt back and forth over the
// chip's 256 CUs: with two blocks per CU the pairs then carry equal work.
__device__ __forceinline__ int snake(int b, int n) {
  const int r = b >> 8;
  if ((r & 1) == 0) return b;
  const int lo = r << 8, hi = min(lo + 255, n - 1);
  return hi - (b - lo);
}

// dS as two bf16 terms. An infinite x is its high term: x - bf16(x) is then NaN, which the clamp turns into a finite
// number (of a finite x the difference is below 2^119, and passes).
__device__ __forceinline__ void split8(const float* x, bf16x8& hi, bf16x8& lo) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    hi[i] = f2bf(x[i]);
    lo[i] = f2bf(__builtin_amdgcn_fmed3f(x[i] - bf2f(hi[i]), -0x1p119f, 0x1p119f));
  }
}
// P >= 0 as two bf16 terms, split downwards with a low term that is positive for every P > 0 (2^-23 P is added to
// it), so that P times an infinite dO is infinite, as in one product.
__device__ __forceinline__ void split8_down(const float* x, bf16x8& hi, bf16x8& lo) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float h = __uint_as_float(__float_as_uint(x[i]) & 0xffff0000u);
    hi[i] = f2bf(h);
    lo[i] = f2bf(fmaf(x[i], 1.0f + 0x1p-23f, -h));
  }
}

// A fragment (32 output rows d = 32 t.., k = rows 16 j + {4 h .. + 3, 8 + 4 h ..}) of a tile, transposed.
__device__ __forceinline__ bf16x8 frag_t(const bf16* tile, int o0, int o1) {
  const short4v a = read_tr16(tile + o0), b = read_tr16(tile + o1);
  const short8v v = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  return __builtin_bit_cast(bf16x8, v);
}

// Row statistics in tile order: lse * log2(e) and Dv = dO . O; rows past Sq get
// an lse that makes every P of theirs 0. 16 lanes per row, 16-byte loads (a
// wave per row with 2-byte loads took 20.9 us at 65,536 rows of 128).
template <int D>
__global__ __launch_bounds__(256) void stats_kernel(const P p) {
  const int64_t row = ((int64_t)blockIdx.x * 256 + threadIdx.x) >> 4;
  const int part = threadIdx.x & 15;
  const int64_t rows_p = (int64_t)p.n_qt * kT32;
  const int64_t bh = row / rows_p;
  const int i = (int)(row - bh * rows_p);
  if (bh >= (int64_t)p.B * p.Hq) return;
  float acc = 0.f;
  if (i < p.Sq && part * 8 < D) {
    const int64_t b = bh / p.Hq, h = bh - b * p.Hq;
    const bf16x8 o = *reinterpret_cast<const bf16x8*>(p.o + b * p.so.b + h * p.so.h + i * p.so.s + part * 8);
    const bf16x8 g = *reinterpret_cast<const bf16x8*>(p.dout + b * p.sg.b + h * p.sg.h + i * p.sg.s + part * 8);
#pragma unroll
    for (int e = 0; e < 8; ++e) acc = fmaf(bf2f(o[e]), bf2f(g[e]), acc);
  }
  acc = group_sum<16>(acc);
  if (part == 0) {
    float* st = p.stats + (bh * p.n_qt + (i >> 5)) * 64 + (i & 31);
    st[0] = i < p.Sq ? p.lse[bh * p.Sq + i] * kLog2e : 1.0e30f;
    st[32] = i < p.Sq ? acc : 0.f;
  }
}

// dK, dV of 128 keys of one KV head over the query heads of one head split.
template <int D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void dkdv_kernel(const P p) {
  constexpr int KSTEPS = (D + 15) / 16, OT = (D + 31) / 32;
  constexpr int PERW = 5;  // direct-to-LDS loads per wave per tile: 2 Q, 2 dO, the statistics
  __shared__ __attribute__((aligned(1024))) bf16 ring[kStg * 2 * kTileE];
  __shared__ __attribute__((aligned(1024))) float s_stat[kStg * 64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, h = lane >> 5;

  // key tiles x (batch, KV head, head split); the first key tiles meet the most queries
  const int nblk = (int)gridDim.x;
  const int blk = p.causal ? snake((int)blockIdx.x, nblk) : (int)blockIdx.x;
  const int nh = p.B * p.Hkv * p.hs;
  const int kt = blk / nh;
  int r = blk - kt * nh;
  const int sp = r % p.hs;
  r /= p.hs;
  const int kvh = r % p.Hkv, b = r / p.Hkv;
  const int gper = p.groups / p.hs;
  const int h0 = kvh * p.groups + sp * gper;  // first query head of the split
  const int j0 = kt * kOwn, kw0 = j0 + 32 * wave, key = kw0 + l32;
  const int64_t kv_row = ((int64_t)b * p.Hkv + kvh) * p.Sk;

  // K and V rows of the wave as B fragments
  bf16x8 kf[KSTEPS], vf[KSTEPS];
  {
    const int64_t row = key < p.Sk ? key : 0;
    const bf16* kr = p.k + b * p.sk.b + kvh * p.sk.h + row * p.sk.s;
    const bf16* vr = p.v + b * p.sv.b + kvh * p.sv.h + row * p.sv.s;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      const bool ok = key < p.Sk && ks * 16 + 8 * h < D;
      kf[ks] = ok ? *reinterpret_cast<const bf16x8*>(kr + ks * 16 + 8 * h) : bf16x8{};
      vf[ks] = ok ? *reinterpret_cast<const bf16x8*>(vr + ks * 16 + 8 * h) : bf16x8{};
    }
  }
  floatx16 dk[OT], dv[OT];
#pragma unroll
  for (int t = 0; t < OT; ++t) dk[t] = dv[t] = floatx16{};

  const int t_first = p.causal ? min(j0 / kT32, p.n_qt) : 0;  // earlier queries see none of the block's keys
  const int per_head = p.n_qt - t_first;
  const int n = per_head * gper;

  const uint32_t lring = q3::lds_addr(ring), lstat = q3::lds_addr(s_stat);
  const int cs = lane & 15;
  const int sq2 = (int)p.sq.s * 2, sg2 = (int)p.sg.s * 2;  // host: Sq * stride * 2 < 2^31
  int ig = 0, it = t_first;  // (head of the split, tile) the next issue takes
  auto issue = [&](int step) {
    const int slot = step % kStg;
    const bool live = step < n;
    const int64_t hd = h0 + (live ? ig : 0);
    const __amdgpu_buffer_rsrc_t qrs =
        q3::make_rsrc(p.q + b * p.sq.b + hd * p.sq.h, ((int64_t)(p.Sq - 1) * p.sq.s + D) * 2);
    const __amdgpu_buffer_rsrc_t grs =
        q3::make_rsrc(p.dout + b * p.sg.b + hd * p.sg.h, ((int64_t)(p.Sq - 1) * p.sg.s + D) * 2);
    const __amdgpu_buffer_rsrc_t srs =
        q3::make_rsrc(p.stats + ((int64_t)b * p.Hq + hd) * p.n_qt * 64, (int64_t)p.n_qt * 256);
    const uint32_t lq = lring + (uint32_t)(slot * 2 * kTileE * 2);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int rr = 8 * wave + 4 * i + (lane >> 4);
      const int c = cs ^ swz(rr);
      const bool ok = live && c * 8 < D;  // rows past Sq lie past the resources' ends
      const uint32_t at = (uint32_t)((8 * wave + 4 * i) * kRow * 2);
      q3::dma16(qrs, ok ? (uint32_t)((it * kT32 + rr) * sq2 + c * 16) : q3::kOOB, lq + at);
      q3::dma16(grs, ok ? (uint32_t)((it * kT32 + rr) * sg2 + c * 16) : q3::kOOB, lq + kTileE * 2 + at);
    }
    // every wave writes the same 64 floats: one load per wave keeps the counts equal
    dma4(srs, live ? (uint32_t)(it * 256 + lane * 4) : q3::kOOB, lstat + (uint32_t)(slot * 256));
    if (live && ++it == p.n_qt) {
      it = t_first;
      ++ig;
    }
  };

  int ro[KSTEPS];  // row fragment offsets
#pragma unroll
  for (int ks = 0; ks < KSTEPS; ++ks) ro[ks] = off(l32, 2 * ks + h);
  const int g16 = (lane >> 4) & 1, rr4 = (lane & 15) >> 2, qq = lane & 3;
  int to[OT][2];  // transposed fragment offsets of rows 4 h + rr4 and 8 + 4 h + rr4 (16 rows on: + 16 kRow)
#pragma unroll
  for (int t = 0; t < OT; ++t) {
    const int d = 32 * t + 16 * g16 + 4 * qq;
    to[t][0] = off(4 * h + rr4, d >> 3) + (d & 7);
    to[t][1] = off(8 + 4 * h + rr4, d >> 3) + (d & 7);
  }

#pragma unroll
  for (int s = 0; s < kStg - 1; ++s) issue(s);
  int ct = t_first;
  const float c2 = p.scale_log2;
  for (int t = 0; t < n; ++t) {
    q3::vm_wait<(kStg - 2) * PERW>();  // this wave's part of tile t has landed
    __syncthreads();                   // every wave's has; the slot of tile t - 1 is free
    issue(t + kStg - 1);
    const int slot = t % kStg, i0 = ct * kT32;
    if (++ct == p.n_qt) ct = t_first;
    if (p.causal && i0 + kT32 - 1 < kw0) continue;  // wave-uniform: every query of the tile precedes the keys
    const bf16* sq = ring + slot * 2 * kTileE;
    const bf16* sg = sq + kTileE;
    const float* st = s_stat + slot * 64;
    floatx16 s = floatx16{}, dp = floatx16{};
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      s = mfma32x32x16(*reinterpret_cast<const bf16x8*>(sq + ro[ks]), kf[ks], s);
      dp = mfma32x32x16(*reinterpret_cast<const bf16x8*>(sg + ro[ks]), vf[ks], dp);
    }
    const bool diag = p.causal && i0 < kw0 + 31;  // wave-uniform: some query of the tile precedes some key
    float pr[16], ds[16];
#pragma unroll
    for (int bq = 0; bq < 4; ++bq) {
      const floatx4 l = *reinterpret_cast<const floatx4*>(st + 8 * bq + 4 * h);
      const floatx4 d4 = *reinterpret_cast<const floatx4*>(st + 32 + 8 * bq + 4 * h);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int x = 4 * bq + e;
        float pe = __builtin_amdgcn_exp2f(fmaf(s[x], c2, -l[e]));
        if (diag && i0 + 8 * bq + 4 * h + e < key) pe = 0.f;
        pr[x] = pe;
        ds[x] = pe * (dp[x] - d4[e]);
      }
    }
    bf16x8 ph[2], pl[2], dh[2], dl[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      split8_down(pr + 8 * j, ph[j], pl[j]);
      split8(ds + 8 * j, dh[j], dl[j]);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int x = 0; x < OT; ++x) {
        const bf16x8 g = frag_t(sg + 16 * j * kRow, to[x][0], to[x][1]);
        dv[x] = mfma32x32x16(g, ph[j], dv[x]);
        dv[x] = mfma32x32x16(g, pl[j], dv[x]);
        const bf16x8 q = frag_t(sq + 16 * j * kRow, to[x][0], to[x][1]);
        dk[x] = mfma32x32x16(q, dh[j], dk[x]);
        dk[x] = mfma32x32x16(q, dl[j], dk[x]);
      }
  }
  q3::vm_wait<0>();  // no load may still target this block's LDS when the wave retires
  if (key >= p.Sk) return;
  if (p.hs == 1) {
    bf16* ko = p.dk + b * p.sdk.b + kvh * p.sdk.h + key * p.sdk.s;
    bf16* vo = p.dv + b * p.sdv.b + kvh * p.sdv.h + key * p.sdv.s;
#pragma unroll
    for (int t = 0; t < OT; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d = 32 * t + 8 * g + 4 * h;
        if (d < D) {
          bf16x4 a, c;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            a[e] = f2bf(dk[t][4 * g + e] * p.scale);
            c[e] = f2bf(dv[t][4 * g + e]);
          }
          *reinterpret_cast<bf16x4*>(ko + d) = a;
          *reinterpret_cast<bf16x4*>(vo + d) = c;
        }
      }
  } else {
    const int64_t plane = (int64_t)p.B * p.Hkv * p.Sk * D;
    float* ko = p.part + (int64_t)sp * 2 * plane + (kv_row + key) * D;
    float* vo = ko + plane;
#pragma unroll
    for (int t = 0; t < OT; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d = 32 * t + 8 * g + 4 * h;
        if (d < D) {
          floatx4 a, c;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            a[e] = dk[t][4 * g + e];
            c[e] = dv[t][4 * g + e];
          }
          *reinterpret_cast<floatx4*>(ko + d) = a;
          *reinterpret_cast<floatx4*>(vo + d) = c;
        }
      }
  }
}

// dK, dV = the head splits' partials in split order, rounded once. n4: floatx4 elements of one plane, d4 of one row.
__global__ __launch_bounds__(256) void dkdv_reduce_kernel(const P p, int64_t n4, int d4) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= 2 * n4) return;
  const floatx4* src = reinterpret_cast<const floatx4*>(p.part) + i;
  floatx4 a = src[0];
  for (int s = 1; s < p.hs; ++s) a += src[(int64_t)s * 2 * n4];
  const bool is_v = i >= n4;
  const float f = is_v ? 1.0f : p.scale;
  bf16x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = f2bf(a[e] * f);
  const int64_t r = (is_v ? i - n4 : i) / d4, bh = r / p.Sk, b = bh / p.Hkv;
  const int c = (int)((is_v ? i - n4 : i) - r * d4);
  const Str st = is_v ? p.sdv : p.sdk;
  bf16* out = (is_v ? p.dv : p.dk) + b * st.b + (bh - b * p.Hkv) * st.h + (r - bh * p.Sk) * st.s + c * 4;
  *reinterpret_cast<bf16x4*>(out) = o;
}

// dQ of 128 queries of one head.
template <int D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void dq_kernel(const P p) {
  constexpr int KSTEPS = (D + 15) / 16, OT = (D + 31) / 32;
  constexpr int PERW = 4;
  __shared__ __attribute__((aligned(1024))) bf16 ring[kStg * 2 * kTileE];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, h = lane >> 5;

  const int nblk = (int)gridDim.x;
  const int blk = p.causal ? snake((int)blockIdx.x, nblk) : (int)blockIdx.x;
  const int nh = p.B * p.Hq;
  const int n_own = nblk / nh;
  const int qt = p.causal ? n_own - 1 - blk / nh : blk / nh;  // the last queries see the most keys
  const int bh = blk % nh, b = bh / p.Hq, kvh = (bh % p.Hq) / p.groups;
  const int q0 = qt * kOwn, qw0 = q0 + 32 * wave, qi = qw0 + l32;
  const int hq = bh - b * p.Hq;

  bf16x8 qf[KSTEPS], gf[KSTEPS];
  {
    const int64_t row = qi < p.Sq ? qi : 0;
    const bf16* qr = p.q + b * p.sq.b + hq * p.sq.h + row * p.sq.s;
    const bf16* gr = p.dout + b * p.sg.b + hq * p.sg.h + row * p.sg.s;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      const bool ok = qi < p.Sq && ks * 16 + 8 * h < D;
      qf[ks] = ok ? *reinterpret_cast<const bf16x8*>(qr + ks * 16 + 8 * h) : bf16x8{};
      gf[ks] = ok ? *reinterpret_cast<const bf16x8*>(gr + ks * 16 + 8 * h) : bf16x8{};
    }
  }
  float lse2 = 1.0e30f, dvi = 0.f;
  if (qi < p.Sq) {
    const float* st = p.stats + ((int64_t)bh * p.n_qt + (qi >> 5)) * 64 + (qi & 31);
    lse2 = st[0];
    dvi = st[32];
  }
  floatx16 dq[OT];
#pragma unroll
  for (int t = 0; t < OT; ++t) dq[t] = floatx16{};

  const int klimit = p.causal ? min(p.Sk, min(q0 + kOwn, p.Sq)) : p.Sk;
  const int n = (klimit + kT32 - 1) / kT32;
  const uint32_t lring = q3::lds_addr(ring);
  const int cs = lane & 15;
  const __amdgpu_buffer_rsrc_t krs =
      q3::make_rsrc(p.k + b * p.sk.b + kvh * p.sk.h, ((int64_t)(p.Sk - 1) * p.sk.s + D) * 2);
  const __amdgpu_buffer_rsrc_t vrs =
      q3::make_rsrc(p.v + b * p.sv.b + kvh * p.sv.h, ((int64_t)(p.Sk - 1) * p.sv.s + D) * 2);
  const int sk2 = (int)p.sk.s * 2, sv2 = (int)p.sv.s * 2;  // host: Sk * stride * 2 < 2^31
  auto issue = [&](int t) {
    const uint32_t lk = lring + (uint32_t)((t % kStg) * 2 * kTileE * 2);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int rr = 8 * wave + 4 * i + (lane >> 4);
      const int c = cs ^ swz(rr);
      const bool ok = t < n && c * 8 < D;
      const uint32_t at = (uint32_t)((8 * wave + 4 * i) * kRow * 2);
      q3::dma16(krs, ok ? (uint32_t)((t * kT32 + rr) * sk2 + c * 16) : q3::kOOB, lk + at);
      q3::dma16(vrs, ok ? (uint32_t)((t * kT32 + rr) * sv2 + c * 16) : q3::kOOB, lk + kTileE * 2 + at);
    }
  };
  int ro[KSTEPS];
#pragma unroll
  for (int ks = 0; ks < KSTEPS; ++ks) ro[ks] = off(l32, 2 * ks + h);
  const int g16 = (lane >> 4) & 1, rr4 = (lane & 15) >> 2, qq = lane & 3;
  int to[OT][2];
#pragma unroll
  for (int t = 0; t < OT; ++t) {
    const int d = 32 * t + 16 * g16 + 4 * qq;
    to[t][0] = off(4 * h + rr4, d >> 3) + (d & 7);
    to[t][1] = off(8 + 4 * h + rr4, d >> 3) + (d & 7);
  }
#pragma unroll
  for (int s = 0; s < kStg - 1; ++s) issue(s);
  const float c2 = p.scale_log2;
  for (int t = 0; t < n; ++t) {
    q3::vm_wait<(kStg - 2) * PERW>();
    __syncthreads();
    issue(t + kStg - 1);
    const int k0 = t * kT32;
    if (p.causal && k0 > qw0 + 31) continue;  // wave-uniform: every key of the tile follows the wave's queries
    const bf16* sk = ring + (t % kStg) * 2 * kTileE;
    const bf16* sv = sk + kTileE;
    floatx16 s = floatx16{}, dp = floatx16{};
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      s = mfma32x32x16(*reinterpret_cast<const bf16x8*>(sk + ro[ks]), qf[ks], s);
      dp = mfma32x32x16(*reinterpret_cast<const bf16x8*>(sv + ro[ks]), gf[ks], dp);
    }
    const bool edge = (p.causal && k0 + kT32 - 1 > qw0) || k0 + kT32 > p.Sk;  // wave-uniform
    float ds[16];
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      const int j = k0 + 8 * (x >> 2) + 4 * h + (x & 3);
      float pe = __builtin_amdgcn_exp2f(fmaf(s[x], c2, -lse2));
      if (edge && (j >= p.Sk || (p.causal && j > qi))) pe = 0.f;
      ds[x] = pe * (dp[x] - dvi);
    }
    bf16x8 dh[2], dl[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) split8(ds + 8 * j, dh[j], dl[j]);
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int x = 0; x < OT; ++x) {
        const bf16x8 a = frag_t(sk + 16 * j * kRow, to[x][0], to[x][1]);
        dq[x] = mfma32x32x16(a, dh[j], dq[x]);
        dq[x] = mfma32x32x16(a, dl[j], dq[x]);
      }
  }
  q3::vm_wait<0>();
  if (qi >= p.Sq) return;
  bf16* qo = p.dq + b * p.sdq.b + hq * p.sdq.h + qi * p.sdq.s;
#pragma unroll
  for (int t = 0; t < OT; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d = 32 * t + 8 * g + 4 * h;
      if (d < D) {
        bf16x4 a;
#pragma unroll
        for (int e = 0; e < 4; ++e) a[e] = f2bf(dq[t][4 * g + e] * p.scale);
        *reinterpret_cast<bf16x4*>(qo + d) = a;
      }
    }
}

// How many blocks share a KV head's query heads: with one block per (key tile,
// KV head) an 8-KV-head layer of 2048 keys has 128 blocks for 512 slots (two
// per CU), so the group's heads are split until the slots are filled; each
// split then leaves fp32 partials that dkdv_reduce_kernel sums.
int64_t head_splits(int64_t B, int64_t Hkv, int64_t groups, int64_t Sk) {
  int64_t hs = 1;
  while (q3_cdiv(Sk, kOwn) * B * Hkv * hs < 512 && groups % (2 * hs) == 0) hs *= 2;
  return hs;
}
int64_t stats_bytes(int64_t B, int64_t Hq, int64_t Sq) { return B * Hq * q3_cdiv(Sq, kT32) * 256; }
int64_t part_bytes(int64_t B, int64_t Hkv, int64_t hs, int64_t Sk, int64_t D) {
  return hs > 1 ? hs * 2 * B * Hkv * Sk * D * 4 : 0;
}
bool head_dim_ok(int64_t D) { return D == 64 || D == 72 || D == 80 || D == 96 || D == 128; }

template <int D>
int launch_d(const P& p, hipStream_t st) {
  const int64_t rows = (int64_t)p.B * p.Hq * p.n_qt * kT32;
  hipLaunchKernelGGL(stats_kernel<D>, dim3((unsigned)q3_cdiv(rows, 16)), dim3(256), 0, st, p);
  Q3_LAUNCH_CHECK();
  const int64_t nk = q3_cdiv(p.Sk, kOwn) * p.B * p.Hkv * p.hs, nq = q3_cdiv(p.Sq, kOwn) * p.B * p.Hq;
  hipLaunchKernelGGL(dkdv_kernel<D>, dim3((unsigned)nk), dim3(256), 0, st, p);
  Q3_LAUNCH_CHECK();
  if (p.hs > 1) {
    const int64_t n4 = (int64_t)p.B * p.Hkv * p.Sk * D / 4;
    hipLaunchKernelGGL(dkdv_reduce_kernel, dim3((unsigned)q3_cdiv(2 * n4, 256)), dim3(256), 0, st, p, n4,
                       D / 4);
    Q3_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(dq_kernel<D>, dim3((unsigned)nq), dim3(256), 0, st, p);
  Q3_LAUNCH_CHECK();
  return Q3_OK;
}

int launch(const P& p, int D, hipStream_t st) {
  if (D == 64) return launch_d<64>(p, st);
  if (D == 72) return launch_d<72>(p, st);
  if (D == 80) return launch_d<80>(p, st);
  if (D == 96) return launch_d<96>(p, st);
  return launch_d<128>(p, st);
}

// 16-byte loads (aligned bases, strides in multiples of 8; 8-byte stores), 32-bit byte offsets within a head, and a
// workspace that holds the row statistics. strides: (b, h, s) of q, k, v, o, grad_out, grad_q, grad_k, grad_v.
bool takes(const void* q, const void* k, const void* v, const void* o, const void* g, const void* dq, const void* dk,
           const void* dv, int64_t B, int64_t Hq, int64_t Hkv, int64_t Sq, int64_t Sk, int64_t D,
           const int64_t* strides, int dtype, const void* ws, int64_t ws_bytes) {
  if (dtype != Q3_BF16 || !head_dim_ok(D) || Sk < 1 || ws_bytes < stats_bytes(B, Hq, Sq) || !q3_aligned(ws, 16))
    return false;
  for (const void* x : {q, k, v, o, g})
    if (!q3_aligned(x, 16)) return false;
  for (const void* x : {dq, dk, dv})
    if (!q3_aligned(x, 8)) return false;
  for (int i = 0; i < 24; ++i)
    if (strides[i] % 8 != 0 || strides[i] < 0) return false;
  for (int t = 0; t < 8; ++t)
    if (strides[3 * t + 2] < D) return false;  // row r of a tile past the last one is past the resource's end
  const int64_t lim = 1ll << 31;
  for (int t : {0, 1, 2, 4})
    if (((t == 1 || t == 2 ? Sk : Sq) + kT32) * strides[3 * t + 2] * 2 >= lim) return false;
  return q3_cdiv(Sk, kOwn) * B * Hq < lim && q3_cdiv(Sq, kOwn) * B * Hq < lim;
}

int run(const void* q, const void* k, const void* v, const void* o, const float* lse, const void* g, void* dq,
        void* dk, void* dv, int64_t B, int64_t Hq, int64_t Hkv, int64_t Sq, int64_t Sk, int64_t D,
        const int64_t* strides, float scale, int is_causal, void* ws, int64_t ws_bytes, hipStream_t st) {
  P m{};
  m.q = static_cast<const bf16*>(q);
  m.k = static_cast<const bf16*>(k);
  m.v = static_cast<const bf16*>(v);
  m.o = static_cast<const bf16*>(o);
  m.dout = static_cast<const bf16*>(g);
  m.lse = lse;
  m.stats = static_cast<float*>(ws);
  m.part = m.stats + stats_bytes(B, Hq, Sq) / 4;
  m.dq = static_cast<bf16*>(dq);
  m.dk = static_cast<bf16*>(dk);
  m.dv = static_cast<bf16*>(dv);
  m.B = (int)B;
  m.Hq = (int)Hq;
  m.Hkv = (int)Hkv;
  m.Sq = (int)Sq;
  m.Sk = (int)Sk;
  m.groups = (int)(Hq / Hkv);
  m.n_qt = (int)q3_cdiv(Sq, kT32);
  m.hs = (int)head_splits(B, Hkv, Hq / Hkv, Sk);
  if (ws_bytes < stats_bytes(B, Hq, Sq) + part_bytes(B, Hkv, m.hs, Sk, D)) m.hs = 1;
  m.scale = scale;
  m.scale_log2 = scale * kLog2e;
  m.causal = is_causal ? 1 : 0;
  Str* const to[8] = {&m.sq, &m.sk, &m.sv, &m.so, &m.sg, &m.sdq, &m.sdk, &m.sdv};
  for (int t = 0; t < 8; ++t) *to[t] = {strides[3 * t], strides[3 * t + 1], strides[3 * t + 2]};
  return launch(m, (int)D, st);
}

}  // namespace bmf

}  // namespace

extern "C" {

int64_t q3_flash_attention_backward_workspace_bytes(int64_t B, int64_t Hq, int64_t Sq) {
  if (B <= 0 || Hq <= 0 || Sq <= 0) return 0;
  return B * Hq * Sq * 4;
}

int64_t q3_flash_attention_backward_mfma_workspace_bytes(int64_t B, int64_t Hq, int64_t Hkv, int64_t Sq, int64_t Sk,
                                                         int64_t D, int dtype) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv || Sq <= 0 || Sk <= 0) return 0;
  const int64_t base = q3_flash_attention_backward_workspace_bytes(B, Hq, Sq);
  if (dtype != Q3_BF16 || !bmf::head_dim_ok(D)) return base;
  return std::max(base, bmf::stats_bytes(B, Hq, Sq) +
                            bmf::part_bytes(B, Hkv, bmf::head_splits(B, Hkv, Hq / Hkv, Sk), Sk, D));
}

int q3_flash_attention_backward(const void* q, const void* k, const void* v, const void* o, const float* lse,
                                const void* grad_out, void* grad_q, void* grad_k, void* grad_v, int64_t B, int64_t Hq,
                                int64_t Hkv, int64_t Sq, int64_t Sk, int64_t D, float scale, int is_causal,
                                int dtype, void* workspace, int64_t workspace_bytes, void* stream) {
  Q3_REQUIRE(q && k && v && o && lse && grad_out && grad_q && grad_k && grad_v, Q3_ERR_NULL);
  Q3_REQUIRE(B >= 0 && Hq >= 1 && Hkv >= 1 && Sq >= 0 && Sk >= 0 && D >= 1, Q3_ERR_SHAPE);
  Q3_REQUIRE(Hq % Hkv == 0 && B * Hq < 65536 && Sq < (1ll << 30) && Sk < (1ll << 30), Q3_ERR_SHAPE);
  Q3_REQUIRE(D <= kMaxD, Q3_ERR_UNSUPPORTED);
  Q3_REQUIRE(dtype == Q3_BF16 || dtype == Q3_F32, Q3_ERR_DTYPE);
  if (B == 0 || Sq == 0) return Q3_OK;
  Q3_REQUIRE(workspace && workspace_bytes >= q3_flash_attention_backward_workspace_bytes(B, Hq, Sq),
             Q3_ERR_WORKSPACE);
  Q3_REQUIRE(q3_aligned(workspace, 4), Q3_ERR_ALIGN);
  BwdParams p{};
  p.q = q;
  p.k = k;
  p.v = v;
  p.o = o;
  p.dout = grad_out;
  p.lse = lse;
  p.dvec = static_cast<float*>(workspace);
  p.dq = grad_q;
  p.dk = grad_k;
  p.dv = grad_v;
  p.B = (int)B;
  p.Hq = (int)Hq;
  p.Hkv = (int)Hkv;
  p.Sq = (int)Sq;
  p.Sk = (int)Sk;
  p.D = (int)D;
  p.groups = (int)(Hq / Hkv);
  p.scale = scale;
  p.causal = is_causal ? 1 : 0;
  hipStream_t st = static_cast<hipStream_t>(stream);
  // The MFMA kernels where they take the call (a caller that sized the workspace by the fp32-per-row query alone gets
  // the SIMT kernels).
  const int64_t sq[3] = {Hq * Sq * D, Sq * D, D}, sk[3] = {Hkv * Sk * D, Sk * D, D};
  int64_t strides[24];
  for (int t = 0; t < 8; ++t)
    for (int i = 0; i < 3; ++i) strides[3 * t + i] = (t == 1 || t == 2 || t == 6 || t == 7) ? sk[i] : sq[i];
  if (bmf::takes(q, k, v, o, grad_out, grad_q, grad_k, grad_v, B, Hq, Hkv, Sq, Sk, D, strides, dtype, workspace,
                 workspace_bytes))
    return bmf::run(q, k, v, o, lse, grad_out, grad_q, grad_k, grad_v, B, Hq, Hkv, Sq, Sk, D, strides, scale,
                    is_causal, workspace, workspace_bytes, st);
  if (dtype == Q3_BF16) return attn_bwd_d<bf16>(p, st);
  return attn_bwd_d<float>(p, st);
}

int q3_flash_attention_backward_strided(const void* q, const void* k, const void* v, const void* o, const float* lse,
                                        const void* grad_out, void* grad_q, void* grad_k, void* grad_v, int64_t B,
                                        int64_t Hq, int64_t Hkv, int64_t Sq, int64_t Sk, int64_t D,
                                        const int64_t* strides, float scale, int is_causal, int dtype,
                                        void* workspace, int64_t workspace_bytes, void* stream) {
  Q3_REQUIRE(q && k && v && o && lse && grad_out && grad_q && grad_k && grad_v && strides, Q3_ERR_NULL);
  Q3_REQUIRE(B >= 0 && Hq >= 1 && Hkv >= 1 && Sq >= 0 && Sk >= 0 && D >= 1, Q3_ERR_SHAPE);
  Q3_REQUIRE(Hq % Hkv == 0 && B * Hq < 65536 && Sq < (1ll << 30) && Sk < (1ll << 30), Q3_ERR_SHAPE);
  if (B == 0 || Sq == 0) return Q3_OK;
  Q3_REQUIRE(workspace && workspace_bytes >= bmf::stats_bytes(B, Hq, Sq), Q3_ERR_WORKSPACE);
  Q3_REQUIRE(bmf::takes(q, k, v, o, grad_out, grad_q, grad_k, grad_v, B, Hq, Hkv, Sq, Sk, D, strides, dtype,
                        workspace, workspace_bytes),
             Q3_ERR_UNSUPPORTED);
  return bmf::run(q, k, v, o, lse, grad_out, grad_q, grad_k, grad_v, B, Hq, Hkv, Sq, Sk, D, strides, scale, is_causal,
                  workspace, workspace_bytes, static_cast<hipStream_t>(stream));
}

}  // extern "C"
