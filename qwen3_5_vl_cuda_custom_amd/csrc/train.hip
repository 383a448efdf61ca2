// The rest of the reference's op namespace and the backward of every op that
// has an autograd wrapper there:
//
//  * forward: sigmoid_mul (x * sigmoid(gate)) and cross_entropy (per-row
//    log-sum-exp in one pass with an online max, the mean over targets that
//    are not ignore_index computed on the device);
//  * backward: sigmoid_mul, swiglu, gelu_tanh (elementwise); softmax (row);
//    rmsnorm and layernorm (row pass for the input gradient, fixed-order
//    reductions for the weight / bias gradients); cross_entropy; top-k (a
//    scatter of the value gradients); matmul (the MFMA GEMMs of gemm.hip on
//    the operands as they are, or, like the batched GEMM, on operands
//    transposed into a workspace; the bias gradient as a fixed-order column sum).
//
// Everything computes in fp32 and rounds once to the tensor dtype. No
// reduction uses atomics: every sum runs in a fixed order, so results are
// bitwise reproducible run to run.
#include <type_traits>

#include "gemm_bwd.h"
#include "q3_common.h"

namespace {

constexpr int kT = 256;  // threads per block of every kernel here

__device__ __forceinline__ float sigmoid_f(float g) { return 1.0f / (1.0f + expf(-g)); }

// d/dx of 0.5 x (1 + tanh(k0 (x + c x^3))).
__device__ __forceinline__ float gelu_tanh_grad(float x) {
  const float k0 = 0.7978845608028654f, c = 0.044715f;
  const float t = tanhf(k0 * (x + c * x * x * x));
  return 0.5f * (1.0f + t) + 0.5f * x * (1.0f - t * t) * k0 * (1.0f + 3.0f * c * x * x);
}

// ===================================================================== elementwise
// Up to three inputs (a, b, c) and two outputs (y0, y1) of one shape.
enum EwOp : int { kSigMulFwd = 0, kSigMulBwd = 1, kSwiGLUBwd = 2, kGeluBwd = 3 };

template <int OP>
__device__ __forceinline__ void ew_eval(float a, float b, float c, float& y0, float& y1) {
  if constexpr (OP == kSigMulFwd) {  // a = x, b = gate
    y0 = a * sigmoid_f(b);
  } else if constexpr (OP == kSigMulBwd) {  // a = x, b = gate, c = dy
    const float s = sigmoid_f(b);
    y0 = c * s;
    y1 = c * a * s * (1.0f - s);
  } else if constexpr (OP == kSwiGLUBwd) {  // a = gate, b = up, c = dy
    const float s = sigmoid_f(a);
    y0 = c * b * s * (1.0f + a * (1.0f - s));
    y1 = c * a * s;
  } else {  // kGeluBwd: a = x, c = dy
    y0 = c * gelu_tanh_grad(a);
  }
}

template <int OP>
constexpr bool ew_uses_b() { return OP != kGeluBwd; }
template <int OP>
constexpr bool ew_uses_c() { return OP != kSigMulFwd; }
template <int OP>
constexpr bool ew_two_out() { return OP == kSigMulBwd || OP == kSwiGLUBwd; }

template <typename T, int OP, bool VEC>
__global__ __launch_bounds__(kT) void ew3_kernel(const T* __restrict__ a, const T* __restrict__ b,
                                                 const T* __restrict__ c, T* __restrict__ y0, T* __restrict__ y1,
                                                 int64_t n) {
  constexpr int V = VEC ? Vec16<T>::N : 1;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t nv = n / V;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nv; i += stride) {
    T va[V], vb[V], vc[V], o0[V], o1[V];
    if constexpr (VEC) {
      typedef typename Vec16<T>::type VT;
      *reinterpret_cast<VT*>(va) = reinterpret_cast<const VT*>(a)[i];
      if constexpr (ew_uses_b<OP>()) *reinterpret_cast<VT*>(vb) = reinterpret_cast<const VT*>(b)[i];
      if constexpr (ew_uses_c<OP>()) *reinterpret_cast<VT*>(vc) = reinterpret_cast<const VT*>(c)[i];
    } else {
      va[0] = a[i];
      if constexpr (ew_uses_b<OP>()) vb[0] = b[i];
      if constexpr (ew_uses_c<OP>()) vc[0] = c[i];
    }
#pragma unroll
    for (int j = 0; j < V; ++j) {
      float r0 = 0.f, r1 = 0.f;
      ew_eval<OP>(to_f<T>(va[j]), ew_uses_b<OP>() ? to_f<T>(vb[j]) : 0.f, ew_uses_c<OP>() ? to_f<T>(vc[j]) : 0.f,
                  r0, r1);
      o0[j] = from_f<T>(r0);
      o1[j] = from_f<T>(r1);
    }
    if constexpr (VEC) {
      typedef typename Vec16<T>::type VT;
      reinterpret_cast<VT*>(y0)[i] = *reinterpret_cast<VT*>(o0);
      if constexpr (ew_two_out<OP>()) reinterpret_cast<VT*>(y1)[i] = *reinterpret_cast<VT*>(o1);
    } else {
      y0[i] = o0[0];
      if constexpr (ew_two_out<OP>()) y1[i] = o1[0];
    }
  }
  if constexpr (VEC) {  // the tail past the last whole vector
    for (int64_t i = nv * V + blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += stride) {
      float r0 = 0.f, r1 = 0.f;
      ew_eval<OP>(to_f<T>(a[i]), ew_uses_b<OP>() ? to_f<T>(b[i]) : 0.f, ew_uses_c<OP>() ? to_f<T>(c[i]) : 0.f, r0,
                  r1);
      y0[i] = from_f<T>(r0);
      if constexpr (ew_two_out<OP>()) y1[i] = from_f<T>(r1);
    }
  }
}

template <typename T, int OP>
int launch_ew3(const void* a, const void* b, const void* c, void* y0, void* y1, int64_t n, hipStream_t st) {
  constexpr int V = Vec16<T>::N;
  bool vec = q3_aligned(a, 16) && q3_aligned(y0, 16);
  if (ew_uses_b<OP>()) vec = vec && q3_aligned(b, 16);
  if (ew_uses_c<OP>()) vec = vec && q3_aligned(c, 16);
  if (ew_two_out<OP>()) vec = vec && q3_aligned(y1, 16);
  const int64_t work = vec ? q3_cdiv(n, V) : n;
  const unsigned blocks = (unsigned)std::max<int64_t>(1, std::min<int64_t>(q3_cdiv(work, kT), 256 * 16));
  const T* pa = static_cast<const T*>(a);
  const T* pb = static_cast<const T*>(b);
  const T* pc = static_cast<const T*>(c);
  if (vec)
    hipLaunchKernelGGL((ew3_kernel<T, OP, true>), dim3(blocks), dim3(kT), 0, st, pa, pb, pc, static_cast<T*>(y0),
                       static_cast<T*>(y1), n);
  else
    hipLaunchKernelGGL((ew3_kernel<T, OP, false>), dim3(blocks), dim3(kT), 0, st, pa, pb, pc, static_cast<T*>(y0),
                       static_cast<T*>(y1), n);
  Q3_LAUNCH_CHECK();
  return Q3_OK;
}

template <int OP>
int ew3_entry(const void* a, const void* b, const void* c, void* y0, void* y1, int64_t n, int dtype, void* stream) {
  Q3_REQUIRE(a && y0, Q3_ERR_NULL);
  Q3_REQUIRE(!ew_uses_b<OP>() || b, Q3_ERR_NULL);
  Q3_REQUIRE(!ew_uses_c<OP>() || c, Q3_ERR_NULL);
  Q3_REQUIRE(!ew_two_out<OP>() || y1, Q3_ERR_NULL);
  Q3_REQUIRE(n >= 0, Q3_ERR_SHAPE);
  if (n == 0) return Q3_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == Q3_BF16) return launch_ew3<bf16, OP>(a, b, c, y0, y1, n, st);
  if (dtype == Q3_F32) return launch_ew3<float, OP>(a, b, c, y0, y1, n, st);
  return Q3_ERR_DTYPE;
}

// ===================================================================== softmax backward
// One wave per row: dot = sum(out * dy), gx = out * (dy - dot).
template <typename T>
__global__ __launch_bounds__(kT) void softmax_bwd_kernel(const T* __restrict__ out, const T* __restrict__ dy,
                                                         T* __restrict__ gx, int64_t rows, int cols) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6;
  if (row >= rows) return;
  const T* o = out + row * (int64_t)cols;
  const T* g = dy + row * (int64_t)cols;
  float dot = 0.f;
  for (int c = lane; c < cols; c += 64) dot += to_f<T>(o[c]) * to_f<T>(g[c]);
  dot = wave_sum(dot);
  T* r = gx + row * (int64_t)cols;
  for (int c = lane; c < cols; c += 64) r[c] = from_f<T>(to_f<T>(o[c]) * (to_f<T>(g[c]) - dot));
}

// ===================================================================== norm backward
// A block takes kNormRows consecutive rows. Phase 1: one wave per row computes
// the row's statistics into LDS. Phase 2: each thread takes columns c, c + 256,
// ... and, for each of them, walks the block's rows in order: it writes the
// input gradient and sums the weight (and bias) gradient terms, which it
// stores as the block's partial row. colsum_reduce_kernel then sums the
// partial rows in block order.
//   rmsnorm:   r = rsqrt(mean(x^2) + eps), gx = dy w r - x (r^3 / n) sum(dy w x),
//              gw = sum_rows dy x r
//   layernorm: m = mean(x), r = rsqrt(mean((x - m)^2) + eps), xh = (x - m) r, g = dy w,
//              gx = r (g - mean(g) - xh mean(g xh)), gw = sum_rows dy xh, gb = sum_rows dy
constexpr int kNormRows = 32;

template <typename T, bool LAYER>
__global__ __launch_bounds__(kT) void norm_bwd_kernel(const T* __restrict__ x, const T* __restrict__ w,
                                                      const T* __restrict__ dy, T* __restrict__ gx,
                                                      float* __restrict__ pw, float* __restrict__ pb, int64_t rows,
                                                      int cols, float eps) {
  __shared__ float s_mean[kNormRows], s_rstd[kNormRows], s_k1[kNormRows], s_k2[kNormRows];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t r0 = (int64_t)blockIdx.x * kNormRows;
  const int nr = (int)std::min<int64_t>(kNormRows, rows - r0);
  const float inv_n = 1.0f / (float)cols;
  for (int rr = wave; rr < nr; rr += kT / 64) {
    const T* xr = x + (r0 + rr) * (int64_t)cols;
    const T* gr = dy + (r0 + rr) * (int64_t)cols;
    if constexpr (LAYER) {
      float s = 0.f;
      for (int c = lane; c < cols; c += 64) s += to_f<T>(xr[c]);
      const float mean = wave_sum(s) * inv_n;
      float v = 0.f, sg = 0.f, sgd = 0.f;
      for (int c = lane; c < cols; c += 64) {
        const float d = to_f<T>(xr[c]) - mean;
        const float g = to_f<T>(gr[c]) * to_f<T>(w[c]);
        v += d * d;
        sg += g;
        sgd += g * d;
      }
      const float rstd = rsqrtf(wave_sum(v) * inv_n + eps);
      sg = wave_sum(sg);
      sgd = wave_sum(sgd);
      if (lane == 0) {
        s_mean[rr] = mean;
        s_rstd[rr] = rstd;
        s_k1[rr] = sg * inv_n;          // mean(g)
        s_k2[rr] = sgd * rstd * inv_n;  // mean(g * xh)
      }
    } else {
      float ss = 0.f, dot = 0.f;
      for (int c = lane; c < cols; c += 64) {
        const float xv = to_f<T>(xr[c]);
        ss += xv * xv;
        dot += to_f<T>(gr[c]) * to_f<T>(w[c]) * xv;
      }
      const float rstd = rsqrtf(wave_sum(ss) * inv_n + eps);
      dot = wave_sum(dot);
      if (lane == 0) {
        s_rstd[rr] = rstd;
        s_k1[rr] = dot * rstd * rstd * rstd * inv_n;
      }
    }
  }
  __syncthreads();
  for (int c = threadIdx.x; c < cols; c += kT) {
    const float wc = to_f<T>(w[c]);
    float aw = 0.f, ab = 0.f;
    for (int rr = 0; rr < nr; ++rr) {
      const int64_t o = (r0 + rr) * (int64_t)cols + c;
      const float xv = to_f<T>(x[o]), g = to_f<T>(dy[o]);
      const float rstd = s_rstd[rr];
      float gxv;
      if constexpr (LAYER) {
        const float xh = (xv - s_mean[rr]) * rstd;
        gxv = rstd * (g * wc - s_k1[rr] - xh * s_k2[rr]);
        aw += g * xh;
        ab += g;
      } else {
        gxv = g * wc * rstd - xv * s_k1[rr];
        aw += g * xv * rstd;
      }
      gx[o] = from_f<T>(gxv);
    }
    if (pw) pw[(int64_t)blockIdx.x * cols + c] = aw;
    if (LAYER && pb) pb[(int64_t)blockIdx.x * cols + c] = ab;
  }
}

// Vector form, for rows of whole 16-byte pieces: G lanes (or the block, G =
// kT) hold a row (NCH pieces each) of x and dy in registers, so both are read once, the row sums
// are lane exchanges, and a lane sums the weight (and bias) gradient of its
// own columns over all rows its block takes. At the end the lane groups of a
// wave and the block's waves are added in order and the block leaves one
// partial row. Bound by memory: reads x and dy, writes gx once. No barrier in
// the row loop. Against the kernel above, which read both operands twice by
// 2-byte loads, idled half of a block at 128 columns and left a partial row
// per 32 rows: (a dense layer at S=2048) 65,536 x 128, 16,384 x 128 and two of
// 2048 x 4096 together 644 -> 60 us, and the sums over the partial rows
// 653 -> 19 us.
template <typename T, bool LAYER, int G, int NCH>
__global__ __launch_bounds__(kT) void norm_bwd_vec_kernel(const T* __restrict__ x, const T* __restrict__ w,
                                                          const T* __restrict__ dy, T* __restrict__ gx,
                                                          float* __restrict__ pw, float* __restrict__ pb,
                                                          int64_t rows, int cols, float eps, int iters) {
  constexpr bool BLK = G == kT;  // the whole block holds one row
  constexpr int V = Vec16<T>::N, RPB = kT / G, CPB = G * NCH * V;
  typedef typename Vec16<T>::type VT;
  __shared__ float s_red[BLK ? 1 : (kT / 64) * CPB];
  __shared__ float s_x[2][kT / 64][4];  // BLK: the waves' sums, two sets used in turn (one barrier per exchange)
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, gl = threadIdx.x % G;
  int turn = 0;
  // the first n of (a, b, c), each summed over the G lanes of the row
  auto sum_rows = [&](auto n, float a, float b, float c) -> float4 {
    constexpr int kN = decltype(n)::value, kG = BLK ? 64 : G;
    a = group_sum<kG>(a);
    if constexpr (kN > 1) b = group_sum<kG>(b);
    if constexpr (kN > 2) c = group_sum<kG>(c);
    if constexpr (!BLK) return {a, b, c, 0.f};
    if (lane == 0) {
      s_x[turn][wave][0] = a;
      s_x[turn][wave][1] = b;
      s_x[turn][wave][2] = c;
    }
    __syncthreads();
    float4 r = {s_x[turn][0][0], s_x[turn][0][1], s_x[turn][0][2], 0.f};
#pragma unroll
    for (int u = 1; u < kT / 64; ++u) {
      r.x += s_x[turn][u][0];
      r.y += s_x[turn][u][1];
      r.z += s_x[turn][u][2];
    }
    turn ^= 1;
    return r;
  };
  const float inv_n = 1.0f / (float)cols;
  float aw[NCH][V] = {}, ab[LAYER ? NCH : 1][V] = {};
  VT wv[NCH];
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int c = (gl + i * G) * V;
    wv[i] = c < cols ? *reinterpret_cast<const VT*>(w + c) : VT{};
  }
  for (int it = 0; it < iters; ++it) {
    const int64_t row = ((int64_t)blockIdx.x * iters + it) * RPB + threadIdx.x / G;
    const bool live = row < rows;
    VT xv[NCH], gv[NCH];
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = (gl + i * G) * V;
      const bool ok = live && c < cols;
      xv[i] = ok ? *reinterpret_cast<const VT*>(x + row * cols + c) : VT{};
      gv[i] = ok ? *reinterpret_cast<const VT*>(dy + row * cols + c) : VT{};
    }
    float mean = 0.f, rstd, k1, k2 = 0.f;
    if constexpr (LAYER) {
      float sx = 0.f;
#pragma unroll
      for (int i = 0; i < NCH; ++i)
#pragma unroll
        for (int j = 0; j < V; ++j) sx += to_f<T>(xv[i][j]);
      mean = sum_rows(std::integral_constant<int, 1>{}, sx, 0.f, 0.f).x * inv_n;
      float v = 0.f, sg = 0.f, sgd = 0.f;
#pragma unroll
      for (int i = 0; i < NCH; ++i) {
        const bool in = (gl + i * G) * V < cols;  // a piece past the row holds zeros, not the mean
#pragma unroll
        for (int j = 0; j < V; ++j) {
          const float d = in ? to_f<T>(xv[i][j]) - mean : 0.f;
          const float g = to_f<T>(gv[i][j]) * to_f<T>(wv[i][j]);
          v += d * d;
          sg += g;
          sgd += g * d;
        }
      }
      const float4 r = sum_rows(std::integral_constant<int, 3>{}, v, sg, sgd);
      rstd = rsqrtf(r.x * inv_n + eps);
      k1 = r.y * inv_n;
      k2 = r.z * rstd * inv_n;
    } else {
      float ss = 0.f, dot = 0.f;
#pragma unroll
      for (int i = 0; i < NCH; ++i)
#pragma unroll
        for (int j = 0; j < V; ++j) {
          const float v = to_f<T>(xv[i][j]);
          ss += v * v;
          dot += to_f<T>(gv[i][j]) * to_f<T>(wv[i][j]) * v;
        }
      const float4 r = sum_rows(std::integral_constant<int, 2>{}, ss, dot, 0.f);
      rstd = rsqrtf(r.x * inv_n + eps);
      k1 = r.y * rstd * rstd * rstd * inv_n;
    }
    if (!live) continue;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = (gl + i * G) * V;
      VT o;
#pragma unroll
      for (int j = 0; j < V; ++j) {
        const float xf = to_f<T>(xv[i][j]), g = to_f<T>(gv[i][j]), wc = to_f<T>(wv[i][j]);
        float r;
        if constexpr (LAYER) {
          const float xh = (xf - mean) * rstd;
          r = rstd * (g * wc - k1 - xh * k2);
          aw[i][j] += g * xh;
          ab[i][j] += g;
        } else {
          r = g * wc * rstd - xf * k1;
          aw[i][j] += g * xf * rstd;
        }
        o[j] = from_f<T>(r);
      }
      if (c < cols) *reinterpret_cast<VT*>(gx + row * cols + c) = o;
    }
  }
  auto flush = [&](float (&acc)[NCH][V], float* part) {
    if constexpr (BLK) {  // every thread has columns of its own
#pragma unroll
      for (int i = 0; i < NCH; ++i)
#pragma unroll
        for (int j = 0; j < V; ++j) {
          const int c = (gl + i * G) * V + j;
          if (c < cols) part[(int64_t)blockIdx.x * cols + c] = acc[i][j];
        }
      return;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NCH; ++i)
#pragma unroll
      for (int j = 0; j < V; ++j) {
        float v = acc[i][j];
#pragma unroll
        for (int o = G; o < 64; o <<= 1) v += __shfl_xor(v, o, 64);
        if (lane < G) s_red[wave * CPB + (gl + i * G) * V + j] = v;
      }
    __syncthreads();
    for (int c = threadIdx.x; c < cols; c += kT) {
      float v = s_red[c];
#pragma unroll
      for (int u = 1; u < kT / 64; ++u) v += s_red[u * CPB + c];
      part[(int64_t)blockIdx.x * cols + c] = v;
    }
  };
  if (pw) flush(aw, pw);
  if constexpr (LAYER) {
    if (pb) flush(ab, pb);
  }
}

// Partial column sums of a (rows, cols) matrix over kColRows-row chunks:
// part[chunk][c] = sum of the chunk's rows, in row order.
constexpr int kColRows = 256;

template <typename T>
__global__ __launch_bounds__(kT) void colsum_partial_kernel(const T* __restrict__ a, float* __restrict__ part,
                                                            int64_t rows, int64_t cols) {
  const int64_t c = (int64_t)blockIdx.x * kT + threadIdx.x;
  if (c >= cols) return;
  const int64_t r0 = (int64_t)blockIdx.y * kColRows;
  const int64_t r1 = std::min<int64_t>(rows, r0 + kColRows);
  float acc = 0.f;
  for (int64_t r = r0; r < r1; ++r) acc += to_f<T>(a[r * cols + c]);
  part[(int64_t)blockIdx.y * cols + c] = acc;
}

// The same for rows of whole 16-byte pieces: 32 pieces x 8 row lanes per
// block, chunks of `per` rows (a multiple of 8, at least 64), the 8 lanes'
// sums added in lane order. One thread per column over 256 rows kept a single
// 2-byte load in flight: the four bias gradients of a vision block at 3136
// rows 248 -> 21 us.
template <typename T>
__global__ __launch_bounds__(kT) void colsum_partial_vec_kernel(const T* __restrict__ a, float* __restrict__ part,
                                                                int64_t rows, int64_t cols, int per) {
  constexpr int V = Vec16<T>::N;
  typedef typename Vec16<T>::type VT;
  __shared__ float s_red[8][32 * V];
  const int cl = threadIdx.x & 31, rl = threadIdx.x >> 5;
  const int64_t c = ((int64_t)blockIdx.x * 32 + cl) * V;
  const int64_t r0 = (int64_t)blockIdx.y * per, r1 = std::min<int64_t>(rows, r0 + per);
  float acc[V] = {};
  if (c < cols) {
#pragma unroll 8
    for (int64_t r = r0 + rl; r < r1; r += 8) {
      const VT v = *reinterpret_cast<const VT*>(a + r * cols + c);
#pragma unroll
      for (int j = 0; j < V; ++j) acc[j] += to_f<T>(v[j]);
    }
  }
#pragma unroll
  for (int j = 0; j < V; ++j) s_red[rl][cl * V + j] = acc[j];
  __syncthreads();
  for (int i = threadIdx.x; i < 32 * V; i += kT) {
    float v = s_red[0][i];
#pragma unroll
    for (int u = 1; u < 8; ++u) v += s_red[u][i];
    const int64_t cc = (int64_t)blockIdx.x * 32 * V + i;
    if (cc < cols) part[(int64_t)blockIdx.y * cols + cc] = v;
  }
}

// out[c] = sum over the nparts partial rows, rounded once. PL lanes per column:
// lane l takes rows l, l + PL, ... in order, the lanes' sums are added in lane
// order. (One thread per column walked the rows one dependent load at a time:
// 2048 partial rows of 128 columns, ~0.6 ms.)
template <typename T, int PL>
__global__ __launch_bounds__(kT) void colsum_reduce_kernel(const float* __restrict__ part, T* __restrict__ out,
                                                           int64_t nparts, int64_t cols) {
  constexpr int COLS = kT / PL;
  __shared__ float s_red[PL][COLS + 1];
  const int cl = threadIdx.x % COLS, pl = threadIdx.x / COLS;
  const int64_t c = (int64_t)blockIdx.x * COLS + cl;
  float acc = 0.f;
  if (c < cols) {
#pragma unroll 8
    for (int64_t p = pl; p < nparts; p += PL) acc += part[p * cols + c];
  }
  if constexpr (PL > 1) {
    s_red[pl][cl] = acc;
    __syncthreads();
    if (pl != 0) return;
    acc = s_red[0][cl];
#pragma unroll
    for (int u = 1; u < PL; ++u) acc += s_red[u][cl];
  }
  if (c < cols) out[c] = from_f<T>(acc);
}

// One lane per column where the rows are few, or where the columns fill the
// chip: with 16 lanes most of a block has nothing to load. One lane / 16, the
// whole column sum in us: 1 row of 128 columns 3.8 / 4.0, of 151,936 4.1 / 7.2; 4
// rows of 1152 4.5 / 4.4, 6 rows 5.1 / 4.4; of 12,288, 8 rows 4.5 / 5.0, 16 rows
// 5.1 / 5.6, 32 rows 12.4 / 12.0.
template <typename T>
int colsum_reduce(const float* part, void* out, int64_t nparts, int64_t cols, hipStream_t st) {
  if (nparts <= 4 || (cols >= 4096 && nparts <= 16))
    hipLaunchKernelGGL((colsum_reduce_kernel<T, 1>), dim3((unsigned)q3_cdiv(cols, kT)), dim3(kT), 0, st, part,
                       static_cast<T*>(out), nparts, cols);
  else
    hipLaunchKernelGGL((colsum_reduce_kernel<T, 16>), dim3((unsigned)q3_cdiv(cols, kT / 16)), dim3(kT), 0, st, part,
                       static_cast<T*>(out), nparts, cols);
  Q3_LAUNCH_CHECK();
  return Q3_OK;
}

// Rows per chunk of the vector column sum: at least 64 (8 loads in flight per
// lane), at most 256 chunks.
int64_t colsum_rows(int64_t rows) { return std::max<int64_t>(64, q3_cdiv(q3_cdiv(rows, 256), 8) * 8); }
int64_t colsum_parts(int64_t rows) { return std::max(q3_cdiv(rows, kColRows), q3_cdiv(rows, colsum_rows(rows))); }

template <typename T>
int colsum_t(const void* a, void* out, int64_t rows, int64_t cols, float* part, hipStream_t st) {
  const T* src = static_cast<const T*>(a);
  int64_t nparts = q3_cdiv(rows, kColRows);
  if (cols % Vec16<T>::N == 0 && q3_aligned(a, 16) && rows < (1ll << 31)) {
    const int per = (int)colsum_rows(rows);
    nparts = q3_cdiv(rows, per);
    hipLaunchKernelGGL(colsum_partial_vec_kernel<T>,
                       dim3((unsigned)q3_cdiv(cols, 32 * Vec16<T>::N), (unsigned)nparts), dim3(kT), 0, st, src, part,
                       rows, cols, per);
  } else {
    hipLaunchKernelGGL(colsum_partial_kernel<T>, dim3((unsigned)q3_cdiv(cols, kT), (unsigned)nparts), dim3(kT), 0, st,
                       src, part, rows, cols);
  }
  Q3_LAUNCH_CHECK();
  return colsum_reduce<T>(part, out, nparts, cols, st);
}

// Blocks of the vector norm backward (each leaves a partial row of `cols`
// floats): up to 512, fewer for wide rows, where 256 fill the chip and the
// partial rows would cost as much as the operands.
int64_t norm_vec_blocks_max(int64_t cols) { return std::max<int64_t>(256, std::min<int64_t>(512, (1 << 20) / cols)); }

template <typename T, bool LAYER, int G, int NCH>
int norm_bwd_vec_t(const void* x, const void* w, const void* dy, void* gx, float* pw, float* pb, int64_t rows,
                   int cols, float eps, int64_t* nblk, hipStream_t st) {
  constexpr int RPB = kT / G;
  const int64_t steps = q3_cdiv(rows, RPB);
  const int64_t iters = q3_cdiv(steps, norm_vec_blocks_max(cols));
  *nblk = q3_cdiv(steps, iters);
  hipLaunchKernelGGL((norm_bwd_vec_kernel<T, LAYER, G, NCH>), dim3((unsigned)*nblk), dim3(kT), 0, st,
                     static_cast<const T*>(x), static_cast<const T*>(w), static_cast<const T*>(dy),
                     static_cast<T*>(gx), pw, pb, rows, cols, eps, (int)iters);
  Q3_LAUNCH_CHECK();
  return Q3_OK;
}

// The narrowest instance that holds a row: 16 lanes, a wave (up to 4 pieces a
// lane: 8 would leave one wave per SIMD, 10 spill), else the whole block. Rows
// of more pieces than the widest instance holds take the scalar kernel.
template <typename T>
constexpr int norm_vec_max_pieces() { return 4 * kT; }

template <typename T, bool LAYER>
int norm_bwd_vec(const void* x, const void* w, const void* dy, void* gx, float* pw, float* pb, int64_t rows, int cols,
                 float eps, int64_t* nblk, hipStream_t st) {
  const int n = cols / Vec16<T>::N;
  if (n <= 16) return norm_bwd_vec_t<T, LAYER, 16, 1>(x, w, dy, gx, pw, pb, rows, cols, eps, nblk, st);
  if (n <= 64) return norm_bwd_vec_t<T, LAYER, 64, 1>(x, w, dy, gx, pw, pb, rows, cols, eps, nblk, st);
  if (n <= 128) return norm_bwd_vec_t<T, LAYER, 64, 2>(x, w, dy, gx, pw, pb, rows, cols, eps, nblk, st);
  if (n <= 192) return norm_bwd_vec_t<T, LAYER, 64, 3>(x, w, dy, gx, pw, pb, rows, cols, eps, nblk, st);
  if (n <= 256) return norm_bwd_vec_t<T, LAYER, 64, 4>(x, w, dy, gx, pw, pb, rows, cols, eps, nblk, st);
  if (n <= 512) return norm_bwd_vec_t<T, LAYER, kT, 2>(x, w, dy, gx, pw, pb, rows, cols, eps, nblk, st);
  return norm_bwd_vec_t<T, LAYER, kT, 4>(x, w, dy, gx, pw, pb, rows, cols, eps, nblk, st);
}

// Floats of one partial buffer the workspace query reports: enough for either form.
int64_t norm_bwd_parts(int64_t rows, int64_t cols) {
  return std::max(q3_cdiv(rows, kNormRows), std::min<int64_t>(rows, norm_vec_blocks_max(cols)));
}
int64_t norm_bwd_ws(int64_t rows, int64_t cols) { return 2 * norm_bwd_parts(rows, cols) * cols * 4; }

template <typename T, bool LAYER>
int norm_bwd_t(const void* x, const void* w, const void* dy, void* gx, void* gw, void* gb, int64_t rows, int cols,
               float eps, float* ws, int64_t ws_bytes, hipStream_t st) {
  int64_t nblk = q3_cdiv(rows, kNormRows);
  const bool parts = gw || (LAYER && gb);
  // 16-byte pieces on every side, a row that the registers hold, and a
  // workspace of the queried size (the scalar form needs less).
  const bool vec = cols % Vec16<T>::N == 0 && cols / Vec16<T>::N <= norm_vec_max_pieces<T>() && q3_aligned(x, 16) &&
                   q3_aligned(w, 16) && q3_aligned(dy, 16) && q3_aligned(gx, 16) &&
                   (!parts || ws_bytes >= norm_bwd_ws(rows, cols));
  const int64_t plane = (vec ? norm_bwd_parts(rows, cols) : nblk) * cols;
  float* pw = gw ? ws : nullptr;
  float* pb = (LAYER && gb) ? ws + plane : nullptr;
  if (vec) {
    const int rc = norm_bwd_vec<T, LAYER>(x, w, dy, gx, pw, pb, rows, cols, eps, &nblk, st);
    if (rc != Q3_OK) return rc;
  } else {
    hipLaunchKernelGGL((norm_bwd_kernel<T, LAYER>), dim3((unsigned)nblk), dim3(kT), 0, st, static_cast<const T*>(x),
                       static_cast<const T*>(w), static_cast<const T*>(dy), static_cast<T*>(gx), pw, pb, rows, cols,
                       eps);
    Q3_LAUNCH_CHECK();
  }
  if (gw) {
    const int rc = colsum_reduce<T>(pw, gw, nblk, cols, st);
    if (rc != Q3_OK) return rc;
  }
  if (pb) return colsum_reduce<T>(pb, gb, nblk, cols, st);
  return Q3_OK;
}

template <bool LAYER>
int norm_bwd_entry(const void* x, const void* w, const void* dy, void* gx, void* gw, void* gb, int64_t rows,
                   int64_t cols, float eps, int dtype, void* ws, int64_t ws_bytes, void* stream) {
  Q3_REQUIRE(x && w && dy && gx, Q3_ERR_NULL);
  Q3_REQUIRE(rows >= 0 && cols >= 1 && cols < (1 << 24), Q3_ERR_SHAPE);
  Q3_REQUIRE(!(gw || gb) || (ws && ws_bytes >= 2 * q3_cdiv(rows, kNormRows) * cols * 4), Q3_ERR_WORKSPACE);
  Q3_REQUIRE(!ws || q3_aligned(ws, 16), Q3_ERR_ALIGN);
  if (rows == 0) return Q3_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  float* f = static_cast<float*>(ws);
  if (dtype == Q3_BF16) return norm_bwd_t<bf16, LAYER>(x, w, dy, gx, gw, gb, rows, (int)cols, eps, f, ws_bytes, st);
  if (dtype == Q3_F32) return norm_bwd_t<float, LAYER>(x, w, dy, gx, gw, gb, rows, (int)cols, eps, f, ws_bytes, st);
  return Q3_ERR_DTYPE;
}

// ===================================================================== cross entropy
// Forward: one block per row. Each thread keeps an online (max, sum of
// exp(x - max)) over its strided share of the row (16-byte vectors when the
// row allows), the block merges the 256 pairs in a fixed tree, and thread 0
// writes lse = max + log(sum) and loss = lse - x[target] (both 0 for a target
// equal to ignore_index, as the reference's kernel does; a target outside
// [0, V) is treated the same and sets bit 0 of *status).
__device__ __forceinline__ void lse_merge(float& m, float& s, float m2, float s2) {
  const float mm = fmaxf(m, m2);
  // the sum of a side without a maximum is 0, or NaN where it met one
  s = (m == -INFINITY ? s : s * expf(m - mm)) + (m2 == -INFINITY ? s2 : s2 * expf(m2 - mm));
  m = mm;
}

// e^x of the loss kernels, x <= 0 up to rounding: for bf16 logits the hardware
// exponential of x log2(e), whose relative error (|x| 2^-24 from the product)
// is at most 0.4 x 2^-24 of the row's sum per term; fp32 logits keep expf.
template <typename T>
__device__ __forceinline__ float exp_of(float x) {
  if constexpr (sizeof(T) == 2) return __builtin_amdgcn_exp2f(x * 1.4426950408889634f);
  return expf(x);
}

template <typename T, bool VEC>
__global__ __launch_bounds__(kT) void ce_fwd_kernel(const T* __restrict__ logits, const int64_t* __restrict__ tgt,
                                                    float* __restrict__ loss, float* __restrict__ lse, int64_t V,
                                                    int64_t ignore_index, int* __restrict__ status) {
  __shared__ float s_m[kT / 64], s_s[kT / 64];
  const int64_t row = blockIdx.x;
  const int64_t t = tgt[row];
  const bool valid = t != ignore_index && t >= 0 && t < V;
  if (!valid) {
    if (threadIdx.x == 0) {
      loss[row] = 0.f;
      lse[row] = 0.f;
      if (t != ignore_index && status) atomicOr(status, 1);
    }
    return;
  }
  const T* xr = logits + row * V;
  float m = -INFINITY, s = 0.f;
  // A piece at a time: one rescale per piece whose maximum is new, so the exponentials of a piece are independent
  // of each other. A piece of -inf only (masked logits) adds nothing.
  auto add = [&](const auto& u, auto n) {
    constexpr int kN = decltype(n)::value;
    float v[kN], mx = m;
#pragma unroll
    for (int j = 0; j < kN; ++j) {
      v[j] = to_f<T>(u[j]);
      mx = fmaxf(mx, v[j]);
    }
    if (mx == -INFINITY) {  // nothing but -inf so far (fmaxf drops NaN, which the sum has to keep)
#pragma unroll
      for (int j = 0; j < kN; ++j) s += v[j] == -INFINITY ? 0.f : v[j];
      return;
    }
    float acc = m == mx ? s : s * exp_of<T>(m - mx);
#pragma unroll
    for (int j = 0; j < kN; ++j) acc += exp_of<T>(v[j] - mx);
    s = acc;
    m = mx;
  };
  if constexpr (VEC) {
    constexpr int NV = Vec16<T>::N;
    typedef typename Vec16<T>::type VT;
    const int64_t nv = V / NV;
    constexpr int kU = 4;  // pieces in flight per thread
    const VT* xv = reinterpret_cast<const VT*>(xr);
    int64_t i = threadIdx.x;
    for (; i + (kU - 1) * kT < nv; i += kU * kT) {
      VT u[kU];
#pragma unroll
      for (int k = 0; k < kU; ++k) u[k] = xv[i + k * kT];
#pragma unroll
      for (int k = 0; k < kU; ++k) add(u[k], std::integral_constant<int, NV>{});
    }
    for (; i < nv; i += kT) add(xv[i], std::integral_constant<int, NV>{});
    for (i = nv * NV + threadIdx.x; i < V; i += kT) add(xr + i, std::integral_constant<int, 1>{});
  } else {
    // 4 values in flight per thread, -inf past the row's end: 33 x 151,937 fp32 logits 150 -> 65 us, bf16 118 -> 47
    constexpr int kU = 4;
    for (int64_t i = threadIdx.x; i < V; i += kU * kT) {
      T u[kU];
#pragma unroll
      for (int k = 0; k < kU; ++k) u[k] = i + k * kT < V ? xr[i + k * kT] : from_f<T>(-INFINITY);
      add(u, std::integral_constant<int, kU>{});
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const float m2 = __shfl_xor(m, o, 64), s2 = __shfl_xor(s, o, 64);
    lse_merge(m, s, m2, s2);
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    s_m[wave] = m;
    s_s[wave] = s;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    float mm = s_m[0], ss = s_s[0];
    for (int w = 1; w < kT / 64; ++w) lse_merge(mm, ss, s_m[w], s_s[w]);
    const float l = mm + logf(ss);
    lse[row] = l;
    loss[row] = l - to_f<T>(xr[t]);
  }
}

// The mean over valid targets: one block sums the per-row losses and counts the
// valid targets in a fixed order; out = sum / max(count, 1) (fp32), and the
// count goes to *n_valid for the backward.
__global__ __launch_bounds__(kT) void ce_mean_kernel(const float* __restrict__ loss, const int64_t* __restrict__ tgt,
                                                     int64_t N, int64_t V, int64_t ignore_index,
                                                     float* __restrict__ out, int* __restrict__ n_valid) {
  __shared__ float s_sum[kT];
  __shared__ int s_cnt[kT];
  float acc = 0.f;
  int cnt = 0;
  for (int64_t i = threadIdx.x; i < N; i += kT) {
    acc += loss[i];
    const int64_t t = tgt[i];
    cnt += (t != ignore_index && t >= 0 && t < V) ? 1 : 0;
  }
  s_sum[threadIdx.x] = acc;
  s_cnt[threadIdx.x] = cnt;
  __syncthreads();
  for (int o = kT / 2; o >= 1; o >>= 1) {
    if ((int)threadIdx.x < o) {
      s_sum[threadIdx.x] += s_sum[threadIdx.x + o];
      s_cnt[threadIdx.x] += s_cnt[threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[0] = s_sum[0] / (float)max(s_cnt[0], 1);
    if (n_valid) n_valid[0] = s_cnt[0];
  }
}

// Backward: grad[i, j] = (exp(x_ij - lse_i) - [j == t_i]) * dloss / max(n_valid, 1);
// rows whose target is ignored (or out of range) get zeros. dloss and n_valid
// are read on the device (no host synchronisation).
// VEC: 16-byte pieces of rows of whole pieces. Bound by memory: 1023 x 151,936
// bf16 logits 219 us by 2-byte accesses, 91 us by pieces (6.8 TB/s).
template <typename T, bool VEC>
__global__ __launch_bounds__(kT) void ce_bwd_kernel(const T* __restrict__ logits, const int64_t* __restrict__ tgt,
                                                    const float* __restrict__ lse, const float* __restrict__ dloss,
                                                    const int* __restrict__ n_valid, T* __restrict__ grad, int64_t V,
                                                    int64_t ignore_index) {
  const int64_t row = blockIdx.y;
  const int64_t t = tgt[row];
  const bool valid = t != ignore_index && t >= 0 && t < V;
  const float scale = dloss[0] / (float)max(n_valid[0], 1);
  const float l = lse[row];
  const T* xr = logits + row * V;
  T* gr = grad + row * V;
  const int64_t step = (int64_t)gridDim.x * kT;
  if constexpr (VEC) {
    constexpr int NV = Vec16<T>::N;
    typedef typename Vec16<T>::type VT;
    for (int64_t i = (int64_t)blockIdx.x * kT + threadIdx.x; i < V / NV; i += step) {
      VT o = VT{};
      if (valid) {
        const VT u = reinterpret_cast<const VT*>(xr)[i];
        const int64_t at = t - i * NV;
#pragma unroll
        for (int j = 0; j < NV; ++j)
          o[j] = from_f<T>((exp_of<T>(to_f<T>(u[j]) - l) - (j == at ? 1.0f : 0.0f)) * scale);
      }
      reinterpret_cast<VT*>(gr)[i] = o;
    }
  } else {
    for (int64_t j = (int64_t)blockIdx.x * kT + threadIdx.x; j < V; j += step) {
      float g = 0.f;
      if (valid) g = (exp_of<T>(to_f<T>(xr[j]) - l) - (j == t ? 1.0f : 0.0f)) * scale;
      gr[j] = from_f<T>(g);
    }
  }
}

// ===================================================================== top-k backward
// grad_x[r, c] = grad_vals[r, j] where idx[r, j] == c, else 0 (the indices of a
// row are distinct). One wave per row.
template <typename T>
__global__ __launch_bounds__(kT) void topk_bwd_kernel(const T* __restrict__ gv, const int64_t* __restrict__ idx,
                                                      T* __restrict__ gx, int64_t rows, int cols, int k) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6;
  if (row >= rows) return;
  for (int c = lane; c < cols; c += 64) {
    float v = 0.f;
    for (int j = 0; j < k; ++j)
      if (idx[row * k + j] == c) v = to_f<T>(gv[row * k + j]);
    gx[row * (int64_t)cols + c] = from_f<T>(v);
  }
}

// ===================================================================== transpose
// (E, R, C) -> (E, C, ldb), columns R .. ldb - 1 of the result zero. Bound by
// memory: one read and one write of each element.
//
// bf16 with 16-byte rows on both sides: a 64 x 64 tile through LDS (rows 72
// elements apart, so the 4 rows of a transposed read fall into distinct
// banks); 16-byte loads, and ds_read_b64_tr_b16 hands each lane 4 rows of its
// column, two of them one 16-byte piece of an output row (64-byte runs per
// wave and row). Against 2-byte accesses through a 64 x 65 tile: the 21
// transposes of a dense layer's backward at S=2048 583 -> 311 us, the three of
// a 151936 x 4096 head's at 1023 rows 1306 -> 623 us (4.6 TB/s).
typedef short tr_short4 __attribute__((ext_vector_type(4)));
typedef short tr_short8 __attribute__((ext_vector_type(8)));
constexpr int kTrLd = 72;

__global__ __launch_bounds__(kT) void transpose_vec_kernel(const bf16* __restrict__ a, bf16* __restrict__ b,
                                                           int64_t R, int64_t C, int64_t ldb) {
  __shared__ __attribute__((aligned(16))) bf16 tile[64 * kTrLd];
  const int64_t e = blockIdx.z;
  const bf16* ae = a + e * R * C;
  bf16* be = b + e * C * ldb;
  const int64_t c0 = (int64_t)blockIdx.x * 64, r0 = (int64_t)blockIdx.y * 64;
  const int tid = threadIdx.x;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = (tid >> 3) + 32 * i, c = (tid & 7) * 8;
    bf16x8 v = bf16x8{};
    if (r0 + r < R && c0 + c < C) v = *reinterpret_cast<const bf16x8*>(ae + (r0 + r) * C + c0 + c);
    *reinterpret_cast<bf16x8*>(tile + r * kTrLd + c) = v;
  }
  __syncthreads();
  // wave w takes columns 16 w .. 16 w + 15; lane group g (16 lanes) rows 32 i + 8 g .. + 7
  const int lane = tid & 63, w = tid >> 6, g = lane >> 4, rr = (lane & 15) >> 2, qq = lane & 3;
  const int64_t c = c0 + 16 * w + (lane & 15);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = 32 * i + 8 * g;
    auto rd = [&](int row) {
      return __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_short4 __attribute__((address_space(3)))*)(
          reinterpret_cast<uintptr_t>(tile + (row + rr) * kTrLd + 16 * w + 4 * qq)));
    };
    const tr_short4 lo = rd(r), hi = rd(r + 4);
    const tr_short8 v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    if (c < C && r0 + r < ldb) *reinterpret_cast<tr_short8*>(be + c * ldb + r0 + r) = v;
  }
}

// Any type and row length, through a 64 x 65 LDS tile.
template <typename T>
__global__ __launch_bounds__(kT) void transpose_kernel(const T* __restrict__ a, T* __restrict__ b, int64_t R,
                                                       int64_t C, int64_t ldb) {
  __shared__ T tile[64][65];
  const int64_t e = blockIdx.z;
  const T* ae = a + e * R * C;
  T* be = b + e * C * ldb;
  const int64_t c0 = (int64_t)blockIdx.x * 64, r0 = (int64_t)blockIdx.y * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int i = ty; i < 64; i += kT / 64) {
    const int64_t r = r0 + i, c = c0 + tx;
    tile[i][tx] = r < R && c < C ? ae[r * C + c] : from_f<T>(0.f);
  }
  __syncthreads();
  for (int i = ty; i < 64; i += kT / 64) {
    const int64_t c = c0 + i, r = r0 + tx;
    if (r < ldb && c < C) be[c * ldb + r] = tile[tx][i];
  }
}

int transpose(const void* a, void* b, int64_t E, int64_t R, int64_t C, int64_t ldb, int dtype, hipStream_t st) {
  if (E == 0 || R == 0 || C == 0) return Q3_OK;
  const dim3 grid((unsigned)q3_cdiv(C, 64), (unsigned)q3_cdiv(ldb, 64), (unsigned)E);
  if (dtype == Q3_BF16) {
    const bf16* s = static_cast<const bf16*>(a);
    bf16* d = static_cast<bf16*>(b);
    if (C % 8 == 0 && ldb % 8 == 0 && q3_aligned(a, 16) && q3_aligned(b, 16))
      hipLaunchKernelGGL(transpose_vec_kernel, grid, dim3(kT), 0, st, s, d, R, C, ldb);
    else
      hipLaunchKernelGGL(transpose_kernel<bf16>, grid, dim3(kT), 0, st, s, d, R, C, ldb);
  } else {
    hipLaunchKernelGGL(transpose_kernel<float>, grid, dim3(kT), 0, st, static_cast<const float*>(a),
                       static_cast<float*>(b), R, C, ldb);
  }
  Q3_LAUNCH_CHECK();
  return Q3_OK;
}

// Row length of the transposed activations (dY^T and X^T of M rows), the
// reduction length of the weight gradient's GEMM: the MFMA kernels take rows
// of a multiple of 8 elements (any other M would leave the GEMM to the SIMT
// kernel: M = 1023, N = 151936, K = 4096 70.2 ms), and whole 64-element stages
// start on cache lines; the padding columns are zeros on both sides.
int64_t padded_rows(int64_t M, int dtype) { return dtype == Q3_BF16 ? q3_cdiv(M, 64) * 64 : M; }

int64_t align256(int64_t n) { return (n + 255) / 256 * 256; }

// Workspace of the matmul backward: W^T (K, N), dY^T (N, Mp), X^T (K, Mp) with
// Mp = padded_rows(M), and the bias gradient's partial sums.
struct MmBwdLayout {
  int64_t wt, dyt, xt, part, total;
};
MmBwdLayout mm_bwd_layout(int64_t M, int64_t N, int64_t K, int dtype) {
  const int64_t es = dtype == Q3_BF16 ? 2 : 4, Mp = padded_rows(M, dtype);
  MmBwdLayout l{};
  l.wt = 0;
  l.dyt = l.wt + align256(K * N * es);
  l.xt = l.dyt + align256(N * Mp * es);
  l.part = l.xt + align256(K * Mp * es);
  l.total = l.part + align256(colsum_parts(M) * N * 4);
  return l;
}

// The products on the operands as they are (no transposes): bf16 rows of whole
// 16-byte pieces and byte offsets below 2 GiB, or fp32 (gemm_bwd.h). The 21 transposes
// of a dense layer's backward at S=2048 took 311 us of its 3143, the three of
// a 151936 x 4096 head's 641 of 4289.
bool mm_bwd_direct_x(const void* w, const void* dy, int64_t M, int64_t N, int64_t K, int dtype) {
  return dtype == Q3_BF16 ? q3::gemm_t_ok(dy, w, M, K, N, false) : q3::gemm_f32_t_ok(dy, M, N, false);
}
bool mm_bwd_direct_w(const void* x, const void* dy, int64_t M, int64_t N, int64_t K, int dtype) {
  return dtype == Q3_BF16 ? q3::gemm_t_ok(dy, x, N, K, M, true) : q3::gemm_f32_t_ok(dy, N, M, true);
}
bool mm_bwd_direct(const void* x, const void* w, const void* dy, int64_t M, int64_t N, int64_t K, int dtype) {
  return mm_bwd_direct_x(w, dy, M, N, K, dtype) && mm_bwd_direct_w(x, dy, M, N, K, dtype);
}
// The fp32 planes of whichever of the two untransposed products splits over K into more.
int64_t mm_bwd_planes(int64_t M, int64_t N, int64_t K, int dtype) {
  return dtype == Q3_BF16 ? std::max(q3::gemm_t_workspace_bytes(M, K, N), q3::gemm_t_workspace_bytes(N, K, M)) : 0;
}

}  // namespace

namespace q3 {
int colsum_reduce_rows(const float* part, void* out, int64_t nparts, int64_t cols, int dtype, hipStream_t st) {
  return dtype == Q3_BF16 ? colsum_reduce<bf16>(part, out, nparts, cols, st)
                          : colsum_reduce<float>(part, out, nparts, cols, st);
}
}  // namespace q3

extern "C" {

int q3_sigmoid_mul(const void* x, const void* gate, void* y, int64_t n, int dtype, void* stream) {
  return ew3_entry<kSigMulFwd>(x, gate, nullptr, y, nullptr, n, dtype, stream);
}

int q3_sigmoid_mul_backward(const void* x, const void* gate, const void* grad_out, void* grad_x, void* grad_gate,
                            int64_t n, int dtype, void* stream) {
  return ew3_entry<kSigMulBwd>(x, gate, grad_out, grad_x, grad_gate, n, dtype, stream);
}

int q3_swiglu_backward(const void* gate, const void* up, const void* grad_out, void* grad_gate, void* grad_up,
                       int64_t n, int dtype, void* stream) {
  return ew3_entry<kSwiGLUBwd>(gate, up, grad_out, grad_gate, grad_up, n, dtype, stream);
}

int q3_gelu_tanh_backward(const void* x, const void* grad_out, void* grad_x, int64_t n, int dtype, void* stream) {
  return ew3_entry<kGeluBwd>(x, nullptr, grad_out, grad_x, nullptr, n, dtype, stream);
}

int q3_softmax_backward(const void* out, const void* grad_out, void* grad_x, int64_t rows, int64_t cols, int dtype,
                        void* stream) {
  Q3_REQUIRE(out && grad_out && grad_x, Q3_ERR_NULL);
  Q3_REQUIRE(rows >= 0 && cols >= 1 && cols < (1 << 30), Q3_ERR_SHAPE);
  if (rows == 0) return Q3_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const unsigned blocks = (unsigned)q3_cdiv(rows, kT / 64);
  if (dtype == Q3_BF16)
    hipLaunchKernelGGL(softmax_bwd_kernel<bf16>, dim3(blocks), dim3(kT), 0, st, static_cast<const bf16*>(out),
                       static_cast<const bf16*>(grad_out), static_cast<bf16*>(grad_x), rows, (int)cols);
  else if (dtype == Q3_F32)
    hipLaunchKernelGGL(softmax_bwd_kernel<float>, dim3(blocks), dim3(kT), 0, st, static_cast<const float*>(out),
                       static_cast<const float*>(grad_out), static_cast<float*>(grad_x), rows, (int)cols);
  else
    return Q3_ERR_DTYPE;
  Q3_LAUNCH_CHECK();
  return Q3_OK;
}

int64_t q3_norm_backward_workspace_bytes(int64_t rows, int64_t cols) {
  if (rows <= 0 || cols <= 0) return 0;
  return norm_bwd_ws(rows, cols);
}

int q3_rmsnorm_backward(const void* x, const void* weight, const void* grad_out, void* grad_x, void* grad_weight,
                        int64_t rows, int64_t cols, float eps, int dtype, void* workspace, int64_t workspace_bytes,
                        void* stream) {
  return norm_bwd_entry<false>(x, weight, grad_out, grad_x, grad_weight, nullptr, rows, cols, eps, dtype, workspace,
                               workspace_bytes, stream);
}

int q3_layernorm_backward(const void* x, const void* weight, const void* grad_out, void* grad_x, void* grad_weight,
                          void* grad_bias, int64_t rows, int64_t cols, float eps, int dtype, void* workspace,
                          int64_t workspace_bytes, void* stream) {
  return norm_bwd_entry<true>(x, weight, grad_out, grad_x, grad_weight, grad_bias, rows, cols, eps, dtype, workspace,
                              workspace_bytes, stream);
}

int q3_cross_entropy(const void* logits, const int64_t* targets, float* loss_per_token, float* lse, float* loss,
                     int* n_valid, int64_t N, int64_t V, int64_t ignore_index, int dtype, int* status, void* stream) {
  Q3_REQUIRE(logits && targets && loss_per_token && lse && loss, Q3_ERR_NULL);
  Q3_REQUIRE(N >= 0 && V >= 1 && N < (1ll << 31), Q3_ERR_SHAPE);
  Q3_REQUIRE(dtype == Q3_BF16 || dtype == Q3_F32, Q3_ERR_DTYPE);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (N > 0) {
    const bool vec = q3_aligned(logits, 16) && V % (dtype == Q3_BF16 ? 8 : 4) == 0;
    const dim3 grid((unsigned)N);
    if (dtype == Q3_BF16) {
      const bf16* l = static_cast<const bf16*>(logits);
      if (vec)
        hipLaunchKernelGGL((ce_fwd_kernel<bf16, true>), grid, dim3(kT), 0, st, l, targets, loss_per_token, lse, V,
                           ignore_index, status);
      else
        hipLaunchKernelGGL((ce_fwd_kernel<bf16, false>), grid, dim3(kT), 0, st, l, targets, loss_per_token, lse, V,
                           ignore_index, status);
    } else {
      const float* l = static_cast<const float*>(logits);
      if (vec)
        hipLaunchKernelGGL((ce_fwd_kernel<float, true>), grid, dim3(kT), 0, st, l, targets, loss_per_token, lse, V,
                           ignore_index, status);
      else
        hipLaunchKernelGGL((ce_fwd_kernel<float, false>), grid, dim3(kT), 0, st, l, targets, loss_per_token, lse,
                           V, ignore_index, status);
    }
    Q3_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(ce_mean_kernel, dim3(1), dim3(kT), 0, st, loss_per_token, targets, N, V, ignore_index, loss,
                     n_valid);
  Q3_LAUNCH_CHECK();
  return Q3_OK;
}

int q3_cross_entropy_backward(const void* logits, const int64_t* targets, const float* lse, const float* grad_loss,
                              const int* n_valid, void* grad_logits, int64_t N, int64_t V, int64_t ignore_index,
                              int dtype, void* stream) {
  Q3_REQUIRE(logits && targets && lse && grad_loss && n_valid && grad_logits, Q3_ERR_NULL);
  Q3_REQUIRE(N >= 0 && V >= 1 && N < 65536ll * 1024, Q3_ERR_SHAPE);
  if (N == 0) return Q3_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  Q3_REQUIRE(dtype == Q3_BF16 || dtype == Q3_F32, Q3_ERR_DTYPE);
  const int64_t piece = dtype == Q3_BF16 ? 8 : 4;
  const bool vec = V % piece == 0 && q3_aligned(logits, 16) && q3_aligned(grad_logits, 16);
  // Blocks per row: 16 of whole pieces, more where the rows are too few to fill the chip with those (16 x 151,936
  // fp32 6.8 -> 5.1 us); 64 of single values.
  const int64_t per_row = vec ? std::max<int64_t>(16, std::min<int64_t>(64, q3_cdiv(1024, N))) : 64;
  const unsigned gx = (unsigned)std::min<int64_t>(q3_cdiv(vec ? V / piece : V, kT), per_row);
  auto run = [&](auto tag, auto v, int64_t r0, unsigned nr) {
    using T = decltype(tag);
    hipLaunchKernelGGL((ce_bwd_kernel<T, decltype(v)::value>), dim3(gx, nr), dim3(kT), 0, st,
                       static_cast<const T*>(logits) + r0 * V, targets + r0, lse + r0, grad_loss, n_valid,
                       static_cast<T*>(grad_logits) + r0 * V, V, ignore_index);
  };
  // grid.y = rows (at most 65535 per launch): launch in row chunks (a chunk's rows keep the 16-byte alignment)
  for (int64_t r0 = 0; r0 < N; r0 += 65535) {
    const unsigned nr = (unsigned)std::min<int64_t>(65535, N - r0);
    if (dtype == Q3_BF16)
      vec ? run(bf16{}, std::true_type{}, r0, nr) : run(bf16{}, std::false_type{}, r0, nr);
    else
      vec ? run(float{}, std::true_type{}, r0, nr) : run(float{}, std::false_type{}, r0, nr);
    Q3_LAUNCH_CHECK();
  }
  return Q3_OK;
}

int q3_topk_backward(const void* grad_vals, const int64_t* idx, void* grad_x, int64_t rows, int64_t cols, int64_t k,
                     int dtype, void* stream) {
  Q3_REQUIRE(grad_vals && idx && grad_x, Q3_ERR_NULL);
  Q3_REQUIRE(rows >= 0 && cols >= 1 && k >= 1 && k <= cols && cols < (1 << 30), Q3_ERR_SHAPE);
  if (rows == 0) return Q3_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const unsigned blocks = (unsigned)q3_cdiv(rows, kT / 64);
  if (dtype == Q3_BF16)
    hipLaunchKernelGGL(topk_bwd_kernel<bf16>, dim3(blocks), dim3(kT), 0, st, static_cast<const bf16*>(grad_vals),
                       idx, static_cast<bf16*>(grad_x), rows, (int)cols, (int)k);
  else if (dtype == Q3_F32)
    hipLaunchKernelGGL(topk_bwd_kernel<float>, dim3(blocks), dim3(kT), 0, st, static_cast<const float*>(grad_vals),
                       idx, static_cast<float*>(grad_x), rows, (int)cols, (int)k);
  else
    return Q3_ERR_DTYPE;
  Q3_LAUNCH_CHECK();
  return Q3_OK;
}

int q3_transpose(const void* a, void* b, int64_t E, int64_t R, int64_t C, int dtype, void* stream) {
  Q3_REQUIRE(a && b, Q3_ERR_NULL);
  Q3_REQUIRE(E >= 0 && R >= 0 && C >= 0 && E < 65536, Q3_ERR_SHAPE);
  Q3_REQUIRE(dtype == Q3_BF16 || dtype == Q3_F32, Q3_ERR_DTYPE);
  return transpose(a, b, E, R, C, R, dtype, static_cast<hipStream_t>(stream));
}

int64_t q3_matmul_backward_workspace_bytes(int64_t M, int64_t N, int64_t K, int dtype) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  return mm_bwd_layout(M, N, K, dtype).total;
}

int64_t q3_matmul_backward_gemm_workspace_bytes(int64_t M, int64_t N, int64_t K, int dtype) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  int64_t need = std::max(q3_matmul_workspace_bytes(M, K, N, dtype, 0),
                          q3_matmul_workspace_bytes(N, K, padded_rows(M, dtype), dtype, 0));
  return std::max(need, mm_bwd_planes(M, N, K, dtype));
}

int64_t q3_matmul_backward_workspace_bytes_for(const void* x, const void* w, const void* dy, int64_t M, int64_t N,
                                               int64_t K, int dtype) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  if (!mm_bwd_direct(x, w, dy, M, N, K, dtype)) return mm_bwd_layout(M, N, K, dtype).total;
  return align256(colsum_parts(M) * N * 4) + mm_bwd_planes(M, N, K, dtype);
}

int64_t q3_matmul_backward_gemm_workspace_bytes_for(const void* x, const void* w, const void* dy, int64_t M, int64_t N,
                                                    int64_t K, int dtype) {
  if (M <= 0 || N <= 0 || K <= 0 || mm_bwd_direct(x, w, dy, M, N, K, dtype)) return 0;
  return q3_matmul_backward_gemm_workspace_bytes(M, N, K, dtype);
}

int q3_matmul_backward(const void* x, const void* w, const void* dy, void* gx, void* gw, void* gb, int64_t M,
                       int64_t N, int64_t K, int dtype, void* workspace, int64_t workspace_bytes, void* gemm_ws,
                       int64_t gemm_ws_bytes, void* stream) {
  Q3_REQUIRE(x && w && dy, Q3_ERR_NULL);
  Q3_REQUIRE(M >= 0 && N >= 0 && K >= 0 && M < (1ll << 31) && N < (1ll << 31) && K < (1ll << 31), Q3_ERR_SHAPE);
  Q3_REQUIRE(dtype == Q3_BF16 || dtype == Q3_F32, Q3_ERR_DTYPE);
  if (M == 0 || N == 0 || K == 0) return Q3_OK;
  const bool dir_x = mm_bwd_direct_x(w, dy, M, N, K, dtype), dir_w = mm_bwd_direct_w(x, dy, M, N, K, dtype);
  MmBwdLayout l = mm_bwd_layout(M, N, K, dtype);
  if (dir_x && dir_w) {  // no operand is transposed: the bias gradient's partial sums, then the products' planes
    l.part = 0;
    l.total = align256(colsum_parts(M) * N * 4);
    const int64_t planes = mm_bwd_planes(M, N, K, dtype);
    if (planes > 0 && workspace_bytes >= l.total + planes) {  // (else the planes go to gemm_ws)
      gemm_ws = static_cast<char*>(workspace) + l.total;
      gemm_ws_bytes = planes;
    }
  }
  Q3_REQUIRE(workspace && workspace_bytes >= l.total, Q3_ERR_WORKSPACE);
  Q3_REQUIRE(q3_aligned(workspace, 256), Q3_ERR_ALIGN);
  char* ws = static_cast<char*>(workspace);
  hipStream_t st = static_cast<hipStream_t>(stream);
  int rc;
  if (gx) {  // gx (M, K) = dY (M, N) . W (N, K)
    if (dir_x) {
      rc = dtype == Q3_BF16 ? q3::gemm_nn(dy, w, gx, M, K, N, gemm_ws, gemm_ws_bytes, st)
                            : q3::gemm_f32_t(dy, w, gx, M, K, N, false, st);
      if (rc != Q3_OK) return rc;
    } else {  // dY . (W^T)^T with W^T (K, N) as the GEMM's weight
      const int64_t need = q3_matmul_workspace_bytes(M, K, N, dtype, 0);
      Q3_REQUIRE(need <= 0 || (gemm_ws && gemm_ws_bytes >= need), Q3_ERR_WORKSPACE);
      if ((rc = transpose(w, ws + l.wt, 1, N, K, N, dtype, st)) != Q3_OK) return rc;
      if ((rc = q3_matmul(dy, ws + l.wt, nullptr, nullptr, gx, M, K, N, N, N, 0, K, dtype, gemm_ws, gemm_ws_bytes,
                          stream)) != Q3_OK)
        return rc;
    }
  }
  if (gw) {  // gw (N, K) = dY^T (N, M) . X (M, K)
    if (dir_w) {
      rc = dtype == Q3_BF16 ? q3::gemm_tn(dy, x, gw, N, K, M, gemm_ws, gemm_ws_bytes, st)
                            : q3::gemm_f32_t(dy, x, gw, N, K, M, true, st);
      if (rc != Q3_OK) return rc;
    } else {  // dY^T . (X^T)^T with X^T (K, M) as the weight
      const int64_t need = q3_matmul_workspace_bytes(N, K, M, dtype, 0);
      Q3_REQUIRE(need <= 0 || (gemm_ws && gemm_ws_bytes >= need), Q3_ERR_WORKSPACE);
      // A tiled GEMM whose workspace covers only the unpadded length runs unsplit; the GEMV (N <= 32) needs all of it.
      int64_t Mp = padded_rows(M, dtype);
      if (N <= 32 && gemm_ws_bytes < q3_matmul_workspace_bytes(N, K, Mp, dtype, 0)) Mp = M;
      if ((rc = transpose(dy, ws + l.dyt, 1, M, N, Mp, dtype, st)) != Q3_OK) return rc;
      if ((rc = transpose(x, ws + l.xt, 1, M, K, Mp, dtype, st)) != Q3_OK) return rc;
      if ((rc = q3_matmul(ws + l.dyt, ws + l.xt, nullptr, nullptr, gw, N, K, Mp, Mp, Mp, 0, K, dtype, gemm_ws,
                          gemm_ws_bytes, stream)) != Q3_OK)
        return rc;
    }
  }
  if (gb) {  // gb (N) = sum over the M rows of dY, in row order
    float* part = reinterpret_cast<float*>(ws + l.part);
    if (dtype == Q3_BF16) return colsum_t<bf16>(dy, gb, M, N, part, st);
    return colsum_t<float>(dy, gb, M, N, part, st);
  }
  return Q3_OK;
}

int64_t q3_batched_gemm_backward_workspace_bytes(int64_t E, int64_t M, int64_t N, int64_t K, int dtype) {
  if (E <= 0 || M <= 0 || N <= 0 || K <= 0) return 0;
  const int64_t es = dtype == Q3_BF16 ? 2 : 4, Mp = padded_rows(M, dtype);
  return align256(E * K * N * es) + align256(E * N * Mp * es) + align256(E * K * Mp * es);
}

int q3_batched_gemm_backward(const void* x, const void* w, const void* dy, void* gx, void* gw, int64_t E, int64_t M,
                             int64_t N, int64_t K, int dtype, void* workspace, int64_t workspace_bytes,
                             void* stream) {
  Q3_REQUIRE(x && w && dy, Q3_ERR_NULL);
  Q3_REQUIRE(E >= 0 && M >= 0 && N >= 0 && K >= 0 && E < 65536, Q3_ERR_SHAPE);
  Q3_REQUIRE(dtype == Q3_BF16 || dtype == Q3_F32, Q3_ERR_DTYPE);
  if (E == 0 || M == 0 || N == 0 || K == 0) return Q3_OK;
  const int64_t es = dtype == Q3_BF16 ? 2 : 4, Mp = padded_rows(M, dtype);
  Q3_REQUIRE(workspace && workspace_bytes >= q3_batched_gemm_backward_workspace_bytes(E, M, N, K, dtype),
             Q3_ERR_WORKSPACE);
  Q3_REQUIRE(q3_aligned(workspace, 256), Q3_ERR_ALIGN);
  char* wt = static_cast<char*>(workspace);
  char* dyt = wt + align256(E * K * N * es);
  char* xt = dyt + align256(E * N * Mp * es);
  hipStream_t st = static_cast<hipStream_t>(stream);
  int rc;
  if (gx) {  // gx[e] (M, K) = dY[e] (M, N) . W[e] (N, K)
    if ((rc = transpose(w, wt, E, N, K, N, dtype, st)) != Q3_OK) return rc;
    if ((rc = q3_batched_gemm(dy, wt, gx, E, M, K, N, dtype, stream)) != Q3_OK) return rc;
  }
  if (gw) {  // gw[e] (N, K) = dY[e]^T (N, M) . X[e] (M, K)
    if ((rc = transpose(dy, dyt, E, M, N, Mp, dtype, st)) != Q3_OK) return rc;
    if ((rc = transpose(x, xt, E, M, K, Mp, dtype, st)) != Q3_OK) return rc;
    if ((rc = q3_batched_gemm(dyt, xt, gw, E, N, K, Mp, dtype, stream)) != Q3_OK) return rc;
  }
  return Q3_OK;
}

}  // extern "C"
