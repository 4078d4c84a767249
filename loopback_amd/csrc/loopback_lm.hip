// loopback_lm.hip -- MI355X (gfx950, CDNA4) kernels of the language model around the Loopback read, in three kinds:
//   * RMSNorm, SwiGLU and the next-token cross entropy, forward and backward, bound by the HBM stream of their rows.
//     torch's composed forms move those rows several times (an fp32 copy of the logits, the softmax, its gradient and its
//     cast; silu and the product; the norm's gradient, its weight's gradient and the residual's add): each is one pass
//     here, with fp32 statistics and one rounding per result;
//   * causal rotary attention in bf16, forward and backward, on the matrix cores, bound by the vector units (the softmax);
//   * weight gradients of the linear layers on the matrix cores, the tokens split over the CUs, bound by LDS reads.
// Every sum has a fixed order: results are deterministic.

#include <hip/hip_runtime.h>
#include <math.h>
#include <stddef.h>
#include <stdint.h>

#include "loopback_lm.h"
#include "loopback_read.h"
#include "device_io.h"

namespace {

constexpr int WG = 256, WAVES = WG / 64;

// ---------------------------------------------------------------------------------------------------------------
// RMSNorm: one wave per row of up to 2048 elements (VPT eight-element vectors per lane). Bound by its rows: the forward
// with the add 2 in and 2 out, the backward 3 in and 1 out. 16384 x 768 bf16: forward 14.8 us (6.8 TB/s of its rows with
// the add; torch's norm 21 and its add 17), backward 18.4 us + the weight's sum (torch: 45 for dx, 21 for the
// weight's partials and 12 for the residual's add)
// ---------------------------------------------------------------------------------------------------------------
template <typename T, int VPT>
__global__ __launch_bounds__(WG) void k_rms_norm_fwd(const T* __restrict__ x, const T* __restrict__ add,
                                                     const T* __restrict__ w, T* __restrict__ h_out,
                                                     T* __restrict__ y, float* __restrict__ rstd, int64_t rows, int d,
                                                     float eps) {
  const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6, d8 = d >> 3;
  typename IO<T>::Raw wv[VPT];
#pragma unroll
  for (int v = 0; v < VPT; ++v) wv[v] = IO<T>::raw(w + 8 * min(lane + 64 * v, d8 - 1));
  for (int64_t row = (int64_t)blockIdx.x * WAVES + wave; row < rows; row += (int64_t)gridDim.x * WAVES) {
    const int64_t ro = row * d;
    typename IO<T>::Raw xr[VPT], ar[VPT];
#pragma unroll
    for (int v = 0; v < VPT; ++v) {
      const int64_t o = ro + 8 * min(lane + 64 * v, d8 - 1);
      xr[v] = IO<T>::raw(x + o);
      if (add) ar[v] = IO<T>::raw(add + o);
    }
    float e[VPT][8], ss = 0.f;
#pragma unroll
    for (int v = 0; v < VPT; ++v) {
      IO<T>::unpack(xr[v], e[v]);
      const bool act = lane + 64 * v < d8;
      if (add) {
        float a[8];
        IO<T>::unpack(ar[v], a);
#pragma unroll
        for (int k = 0; k < 8; ++k) e[v][k] = IO<T>::round(e[v][k] + a[k]);
        if (act) IO<T>::store(h_out + ro + 8 * (lane + 64 * v), e[v]);
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) ss = __builtin_fmaf(act ? e[v][k] : 0.f, e[v][k], ss);
    }
    ss = lanes_reduce(ss, 64, AddOp());
    const float r = rsqrtf(ss / (float)d + eps);
    if (lane == 0) rstd[row] = r;
#pragma unroll
    for (int v = 0; v < VPT; ++v) {
      if (lane + 64 * v < d8) {
        float o[8];
        IO<T>::unpack(wv[v], o);
#pragma unroll
        for (int k = 0; k < 8; ++k) o[k] = e[v][k] * r * o[k];
        IO<T>::store(y + ro + 8 * (lane + 64 * v), o);
      }
    }
  }
}

// A workgroup's waves take rows in turn and keep the weight gradient's columns in registers; the four waves' sums meet
// in LDS, one partial row per workgroup. dx or dw_part NULL: not asked for, not written.
constexpr int NORM_GRID = 512;

template <typename T, int VPT>
__global__ __launch_bounds__(WG) void k_rms_norm_bwd(const T* __restrict__ dy, const T* __restrict__ h,
                                                     const T* __restrict__ w, const float* __restrict__ rstd,
                                                     const T* __restrict__ dres, T* __restrict__ dx,
                                                     float* __restrict__ dw_part, int64_t rows, int d) {
  __shared__ float s_dw[VPT * 512];
  const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6, d8 = d >> 3;
  float wv[VPT][8], dw[VPT][8];
#pragma unroll
  for (int v = 0; v < VPT; ++v) {
    IO<T>::load(w + 8 * min(lane + 64 * v, d8 - 1), wv[v]);
#pragma unroll
    for (int k = 0; k < 8; ++k) dw[v][k] = 0.f;
  }
  for (int64_t row = (int64_t)blockIdx.x * WAVES + wave; row < rows; row += (int64_t)gridDim.x * WAVES) {
    const int64_t ro = row * d;
    typename IO<T>::Raw yr[VPT], hr[VPT], rr[VPT];
    const float r = rstd[row];
#pragma unroll
    for (int v = 0; v < VPT; ++v) {
      const int64_t o = ro + 8 * min(lane + 64 * v, d8 - 1);
      yr[v] = IO<T>::raw(dy + o);
      hr[v] = IO<T>::raw(h + o);
      if (dres) rr[v] = IO<T>::raw(dres + o);
    }
    float c = 0.f;   // sum dy w h
#pragma unroll
    for (int v = 0; v < VPT; ++v) {
      float a[8], b[8];
      IO<T>::unpack(yr[v], a);
      IO<T>::unpack(hr[v], b);
      const bool act = lane + 64 * v < d8;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        c = __builtin_fmaf(act ? a[k] * wv[v][k] : 0.f, b[k], c);
        dw[v][k] = __builtin_fmaf(a[k], b[k] * r, dw[v][k]);
      }
    }
    if (!dx) continue;
    c = lanes_reduce(c, 64, AddOp()) * r * r / (float)d;
#pragma unroll
    for (int v = 0; v < VPT; ++v) {
      if (lane + 64 * v < d8) {
        float a[8], b[8], o[8];
        IO<T>::unpack(yr[v], a);
        IO<T>::unpack(hr[v], b);
#pragma unroll
        for (int k = 0; k < 8; ++k) o[k] = r * (a[k] * wv[v][k] - c * b[k]);
        if (dres) {
          float g[8];
          IO<T>::unpack(rr[v], g);
#pragma unroll
          for (int k = 0; k < 8; ++k) o[k] += g[k];
        }
        IO<T>::store(dx + ro + 8 * (lane + 64 * v), o);
      }
    }
  }
  if (!dw_part) return;
  for (int k = 0; k < WAVES; ++k) {
    if (wave == k) {
#pragma unroll
      for (int v = 0; v < VPT; ++v)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          float* o = s_dw + 8 * (lane + 64 * v) + e;
          *o = k == 0 ? dw[v][e] : *o + dw[v][e];
        }
    }
    __syncthreads();
  }
  for (int c = (int)threadIdx.x; c < d; c += WG) dw_part[(int64_t)blockIdx.x * d + c] = s_dw[c];
}

// out[c] = round(sum_p part[p][c]): 16 columns per workgroup, rows p = group mod 16 added in order, then the groups
template <typename T>
__global__ __launch_bounds__(WG) void k_sum_rows(const float* __restrict__ part, int64_t rows, int d,
                                                 T* __restrict__ out) {
  __shared__ float s[WG];
  const int tid = (int)threadIdx.x, cl = tid & 15, grp = tid >> 4, c = blockIdx.x * 16 + cl;
  float acc = 0.f;
  if (c < d) {
    int64_t p = grp;
    for (; p + 7 * 16 < rows; p += 8 * 16) {   // eight rows' loads in flight
      float a[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) a[u] = part[(p + 16 * u) * d + c];
#pragma unroll
      for (int u = 0; u < 8; ++u) acc += a[u];
    }
    for (; p < rows; p += 16) acc += part[p * d + c];
  }
  s[tid] = acc;
  __syncthreads();
  if (grp == 0 && c < d) {
    float t = s[cl];
    for (int k = 1; k < 16; ++k) t += s[k * 16 + cl];
    st1(out + c, t);
  }
}

// ---------------------------------------------------------------------------------------------------------------
// SwiGLU, bound by its rows (3 of n in and out forward, 5 backward). 16384 x 2048 bf16: forward 34-38 us (5.6 TB/s),
// backward 52 us (6.5 TB/s); torch's silu, product, their gradients and the concatenation of the halves took ~290 us
// ---------------------------------------------------------------------------------------------------------------
// (the fast exponential: its error, some 2^-24 |x|, is far below the results' own rounding -- from 64 bits at N(0, 1) to
// N(0, 256): forward 1.66e-3 to 1.65e-3 in bf16 and 2.1e-4 in fp16, to the sixth digit what the accurate one gives;
// torch's two operations 1.67e-3 to 2.4e-3 and 2.1e-4 to 2.9e-4)
__device__ __forceinline__ float sigmoid(float x) { return 1.f / (1.f + __expf(-x)); }

template <typename T>
__global__ __launch_bounds__(WG) void k_swiglu_fwd(const T* __restrict__ gu, T* __restrict__ act, int64_t nvec,
                                                   int n8) {
  for (int64_t i = (int64_t)blockIdx.x * WG + threadIdx.x; i < nvec; i += (int64_t)gridDim.x * WG) {
    const int64_t row = i / n8, c = 8 * (i - row * n8), base = row * 16 * n8;
    float g[8], u[8];
    IO<T>::load(gu + base + c, g);
    IO<T>::load(gu + base + 8 * n8 + c, u);
#pragma unroll
    for (int k = 0; k < 8; ++k) g[k] = g[k] * sigmoid(g[k]) * u[k];
    IO<T>::store(act + 8 * i, g);
  }
}

template <typename T>
__global__ __launch_bounds__(WG) void k_swiglu_bwd(const T* __restrict__ gu, const T* __restrict__ dact,
                                                   T* __restrict__ dgu, int64_t nvec, int n8) {
  for (int64_t i = (int64_t)blockIdx.x * WG + threadIdx.x; i < nvec; i += (int64_t)gridDim.x * WG) {
    const int64_t row = i / n8, c = 8 * (i - row * n8), base = row * 16 * n8;
    float g[8], u[8], a[8];
    IO<T>::load(gu + base + c, g);
    IO<T>::load(gu + base + 8 * n8 + c, u);
    IO<T>::load(dact + 8 * i, a);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float s = sigmoid(g[k]), sg = g[k] * s;
      const float dg = a[k] * u[k] * (s + sg * (1.f - s));
      u[k] = a[k] * sg;
      g[k] = dg;
    }
    IO<T>::store(dgu + base + c, g);
    IO<T>::store(dgu + base + 8 * n8 + c, u);
  }
}

// ---------------------------------------------------------------------------------------------------------------
// next-token cross entropy: one workgroup per row of logits, eight logits per lane and load (element alignment: any
// vocabulary size), the last vocab mod 8 one per lane. A vocabulary of 32000 is 16 vectors per lane: the row's online
// maximum and sum stay in registers, so a pass reads each logit once: 16384 x 32000 bf16 188 us forward (5.6 TB/s) and
// 387 us backward (5.4 TB/s), against ~5.5 ms for an fp32 copy, torch's log-softmax and its gradient, and the casts.
// Exponentials of differences from the maximum by the fast form: where its error (some 2^-24 of the difference) is large
// the term is small. The loss lies as far from 64 bits as torch's fp32 form (1.8e-8 to 9e-8 of it over logits of
// N(0, 0.25) to N(0, 400), vocabularies 4096 to 32000), its gradient to six digits where the accurate exponential puts
// it; that one took 298 us forward.
// ---------------------------------------------------------------------------------------------------------------
// sum of exp(x - m) over a workgroup's lanes, each holding (m, s); every lane ends with the totals
__device__ __forceinline__ void join_lse(float& m, float& s, float (&red)[2 * WAVES]) {
  const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
  const float mw = lanes_reduce(m, 64, MaxOp());
  s = lanes_reduce(m == -INFINITY ? 0.f : s * expf(m - mw), 64, AddOp());
  if (lane == 0) {
    red[wave] = mw;
    red[WAVES + wave] = s;
  }
  __syncthreads();
  m = red[0];
#pragma unroll
  for (int k = 1; k < WAVES; ++k) m = fmaxf(m, red[k]);
  s = 0.f;
#pragma unroll
  for (int k = 0; k < WAVES; ++k) s += red[k] == -INFINITY ? 0.f : red[WAVES + k] * expf(red[k] - m);
}

template <typename T>
__global__ __launch_bounds__(WG) void k_next_token_fwd(const T* __restrict__ logits, const int64_t* __restrict__ ids,
                                                       float* __restrict__ lse, float* __restrict__ nll, int64_t t,
                                                       int64_t vocab) {
  __shared__ float red[2 * WAVES];
  const int64_t row = blockIdx.x;
  const T* x = logits + row * vocab;
  const bool counted = row % t != t - 1;   // workgroup-uniform
  if (!counted) {
    if (threadIdx.x == 0) lse[2 * row] = lse[2 * row + 1] = nll[row] = 0.f;
    return;
  }
  float m = -INFINITY, s = 0.f;
  const int64_t nv = vocab >> 3;
  for (int64_t c = threadIdx.x; c < nv; c += WG) {
    float e[8];
    IO<T>::unpack(UIO<T>::raw(x + 8 * c), e);
    float mx = e[0];
    bool nan = false;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      mx = fmaxf(mx, e[k]);
      nan |= e[k] != e[k];
    }
    if (mx > m) {
      s *= __expf(m - mx);
      m = mx;
    }
    float a = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) a += m == -INFINITY ? 0.f : __expf(e[k] - m);
    s = nan ? NAN : s + a;
  }
  if ((int64_t)threadIdx.x < (vocab & 7)) {
    const float e = ld1(x + 8 * nv + threadIdx.x);
    if (e > m) {
      s *= __expf(m - e);
      m = e;
    }
    s += e != e ? e : (m == -INFINITY ? 0.f : __expf(e - m));
  }
  if (s != s && m == -INFINITY) m = 0.f;   // a row of NaN only: keep the NaN in the sum
  join_lse(m, s, red);
  if (threadIdx.x == 0) {
    const int64_t label = ids[row + 1];
    const float l = logf(s);   // kept apart from the maximum: their sum would lose it beside large logits
    lse[2 * row] = m;
    lse[2 * row + 1] = l;
    nll[row] = label >= 0 && label < vocab ? l + (m - ld1(x + label)) : NAN;
  }
}

// loss = sum nll / count by one workgroup of 1024 lanes: lane sums in order, then a fixed tree
__global__ __launch_bounds__(1024) void k_mean(const float* __restrict__ nll, int64_t n, float count,
                                               float* __restrict__ loss) {
  __shared__ float s[1024];
  const int tid = (int)threadIdx.x;
  float a = 0.f;
  for (int64_t i = tid; i < n; i += 1024) a += nll[i];
  s[tid] = a;
  __syncthreads();
  for (int w = 512; w > 0; w >>= 1) {
    if (tid < w) s[tid] += s[tid + w];
    __syncthreads();
  }
  if (tid == 0) *loss = s[0] / count;
}

template <typename T>
__global__ __launch_bounds__(WG) void k_next_token_bwd(const T* __restrict__ logits, const int64_t* __restrict__ ids,
                                                       const float* __restrict__ lse, const float* __restrict__ dloss,
                                                       T* __restrict__ dlogits, int64_t t, int64_t vocab,
                                                       float inv_count) {
  const int64_t row = blockIdx.x;
  const T* x = logits + row * vocab;
  T* o = dlogits + row * vocab;
  const bool counted = row % t != t - 1;
  const float m = lse[2 * row], l = lse[2 * row + 1], g = counted ? *dloss * inv_count : 0.f;
  const int64_t label = counted ? ids[row + 1] : -1, nv = vocab >> 3;
  for (int64_t c = threadIdx.x; c < nv; c += WG) {
    float e[8];
    if (counted) {
      IO<T>::unpack(UIO<T>::raw(x + 8 * c), e);
#pragma unroll
      for (int k = 0; k < 8; ++k) e[k] = (__expf((e[k] - m) - l) - (8 * c + k == label ? 1.f : 0.f)) * g;
    } else {
#pragma unroll
      for (int k = 0; k < 8; ++k) e[k] = 0.f;
    }
    UIO<T>::store(o + 8 * c, e);
  }
  if ((int64_t)threadIdx.x < (vocab & 7)) {
    const int64_t k = 8 * nv + threadIdx.x;
    st1(o + k, counted ? (__expf((ld1(x + k) - m) - l) - (k == label ? 1.f : 0.f)) * g : 0.f);
  }
}

// ---------------------------------------------------------------------------------------------------------------
// causal rotary attention, head width 64, bf16 (fp32 scores, softmax and accumulators; the probabilities and score
// gradients enter the matrix cores in bf16, as in every flash attention)
//
// Operands go through v_mfma_f32_32x32x16_bf16: lane l holds row (A) or column (B) l mod 32 at k = 8 (l / 32) .. + 8; of
// the 32 x 32 result it holds column l mod 32 and, in register r, row 4 (l / 32) + r mod 4 + 8 (r / 4). The scores are
// formed transposed where the next product sums over their rows, so a product's result is the next one's B operand as
// it lies in the registers (its k order permuted: slot j of lane half h of a 16-row step is row 4 h + j, + 4 past j = 3),
// and a row's softmax is in-lane but for one exchange of lane halves. The matching A operands, columns of a tile kept by
// rows, come from LDS with ds_read_b64_tr_b16: of the 16 lanes that read 4 rows x 16 columns together, lane i gets
// column i of the 4 rows. Tiles of 64 rows sit in LDS in rows of 144 bytes (16 of padding: the 16-byte operand reads of
// 16 rows then cover the 64 banks once), two buffers each, the next tile's rows in registers while one is worked on.
//
// Per 64 x 32 tile a wave issues 512 matrix-core cycles forward (512 per product pair backward) and ~1000 vector cycles
// (per score an exponential, 16 cycles, and 4-7 operations of 4): the vector units bound it, so two or three waves
// share a SIMD and the maximum is moved, and the sums rescaled, only when it grows by more than 2^8.
// 8 x 2048 tokens, 12 heads: the rotation 16 us, forward 75-80 us (640-690 TFLOP/s of the causal half), both backward
// kernels 273-280; the flash attention of torch took 172 and 780 us, and the rotation, its gradient and the copies
// between layouts another ~700 in some twenty elementwise launches. What took these kernels there from 113 and 362 us:
// the masks under a wave-uniform branch and before the exponential (they had been a branch per score in the dk, dv
// kernel), two waves per SIMD asked for (the accumulators then stay in vector registers, 128 moves less per tile),
// addresses moved on instead of formed per tile, and the order of the work (attn_work). Three waves per SIMD in the
// dk, dv kernel spill 116 bytes and cost a third; one row half at a time in the backward kernels is level.
// ---------------------------------------------------------------------------------------------------------------
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int AT_M = 128, AT_N = 64, AT_LD = 72;   // rows per workgroup (32 per wave), rows per LDS tile, its row length
constexpr float AT_LAZY = 8.f;                      // the maximum moves when it grows by 2^8 or more
constexpr float AT_SCALE = 0.125f, LOG2E = 1.4426950408889634f;   // 1 / sqrt(64)

__device__ __forceinline__ f32x16 mfma(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 zero16() {
  f32x16 z;
#pragma unroll
  for (int i = 0; i < 16; ++i) z[i] = 0.f;
  return z;
}
__device__ __forceinline__ bf16x8 frag(uint4 u) { return __builtin_bit_cast(bf16x8, u); }
// registers 8 s .. 8 s + 7 of a result as the B operand of the next product's 16-row step s
__device__ __forceinline__ bf16x8 operand(const f32x16& x, int s) {
  return frag(make_uint4(pack2(x[8 * s], x[8 * s + 1]), pack2(x[8 * s + 2], x[8 * s + 3]),
                         pack2(x[8 * s + 4], x[8 * s + 5]), pack2(x[8 * s + 6], x[8 * s + 7])));
}
// A operand, rows as they lie: rows r0 + l mod 32, columns 16 ks + 8 (l / 32) .. + 8
__device__ __forceinline__ bf16x8 rows_frag(const bf16_t* tile, int r0, int ks, int lane) {
  return frag(*reinterpret_cast<const uint4*>(tile + (r0 + (lane & 31)) * AT_LD + 16 * ks + 8 * (lane >> 5)));
}
// A operand, columns of the tile: columns c0 + l mod 32, rows r0 + {4 h + 0..3, 8 + 4 h + 0..3}, the order of operand()
template <int LD = AT_LD> __device__ __forceinline__ bf16x8 cols_frag(const bf16_t* tile, int r0, int c0, int lane) {
  typedef __attribute__((address_space(3))) s16x4* lds4;
  const int j = lane & 15;
  const bf16_t* p = tile + (r0 + 4 * (lane >> 5) + (j >> 2)) * LD + c0 + (lane & 16) + 4 * (j & 3);
  const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(const_cast<bf16_t*>(p)));
  const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(const_cast<bf16_t*>(p + 8 * LD)));
  const uint2 ua = __builtin_bit_cast(uint2, a), ub = __builtin_bit_cast(uint2, b);
  return frag(make_uint4(ua.x, ua.y, ub.x, ub.y));
}
__device__ __forceinline__ float other_half(float x, bool sum) {   // x joined with the other lane half's
  const unsigned u = __float_as_uint(x);
  const auto sw = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  const float a = __uint_as_float((unsigned)sw[0]), b = __uint_as_float((unsigned)sw[1]);
  return sum ? a + b : fmaxf(a, b);
}

// 64 rows of 64 elements, row stride `stride` elements: 512 16-byte pieces, two per lane. The cursor's addresses move on
// by a tile per load; rows past the last repeat it.
struct TileRegs { uint4 u[2]; };
struct Cursor {
  const bf16_t* p[2];
  int64_t stride;
  int row0, t;
  __device__ __forceinline__ Cursor(const bf16_t* base, int64_t stride_, int row0_, int t_)
      : stride(stride_), row0(row0_), t(t_) {
#pragma unroll
    for (int i = 0; i < 2; ++i) p[i] = base + (int64_t)(row0 + row(i)) * stride + 8 * ((int)threadIdx.x & 7);
  }
  static __device__ __forceinline__ int row(int i) { return ((int)threadIdx.x >> 3) + 32 * i; }
  __device__ __forceinline__ TileRegs next() {
    TileRegs r;
    if (row0 + AT_N <= t) {
#pragma unroll
      for (int i = 0; i < 2; ++i) r.u[i] = *reinterpret_cast<const uint4*>(p[i]);
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i)
        r.u[i] = *reinterpret_cast<const uint4*>(p[i] - (int64_t)max(row0 + row(i) - (t - 1), 0) * stride);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) p[i] += AT_N * stride;
    row0 += AT_N;
    return r;
  }
};
__device__ __forceinline__ void tile_store(bf16_t* tile, const TileRegs& r) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int c = (int)threadIdx.x + 256 * i;
    *reinterpret_cast<uint4*>(tile + (c >> 3) * AT_LD + 8 * (c & 7)) = r.u[i];
  }
}

// Which (batch, head) and block of rows a workgroup takes: the blocks of one head on one XCD (workgroups go to XCDs in
// turn), so its rows are read from that XCD's L2, and in each XCD the most work of every head first: a head's blocks in
// one run instead put three long ones on one CU and three short ones on another (2 x 4096 tokens, 12 heads: forward 118
// -> 82 us, backward 304 -> 244; 8 x 2048: 103 -> 76 and 307 -> 273). False past the last head.
struct AttnWork { int bh, block; };
__device__ __forceinline__ bool attn_work(int bhs, int blocks, AttnWork& w) {
  const int i = (int)blockIdx.x >> 3, heads = (bhs + 7) >> 3;   // heads of an XCD
  w.bh = ((int)blockIdx.x & 7) + 8 * (i % heads);
  w.block = i / heads;
  return w.bh < bhs;
}

// q and k of [b, t, 3, heads, 64] rotated (pairs j, j + 32; cos, sin [t, 64] fp32 with both halves alike) into
// [b, t, 2, heads, 64]: products, then the sum, each rounded in fp32, and one rounding to bf16, as the torch form
__global__ __launch_bounds__(WG) void k_rotary(const bf16_t* __restrict__ qkv, const float* __restrict__ cosT,
                                               const float* __restrict__ sinT, bf16_t* __restrict__ qk, int64_t n,
                                               int t, int heads) {
#pragma clang fp contract(off)
  const int per = 2 * heads * 4;   // work items of a token: (q or k, head, 8 of the 32 pairs)
  for (int64_t i = (int64_t)blockIdx.x * WG + threadIdx.x; i < n; i += (int64_t)gridDim.x * WG) {
    const int64_t tok = i / per;
    const int r = (int)(i - tok * per), j = 8 * (r & 3), head = r >> 2;   // head counts q's, then k's
    const bf16_t* x = qkv + (tok * 3 * heads + head) * 64 + j;
    const int64_t pos = (tok % t) * 64 + j;
    float a[8], b[8], c[8], s[8], o[8];
    IO<bf16_t>::load(x, a);
    IO<bf16_t>::load(x + 32, b);
    load_f32x8(cosT + pos, c);
    load_f32x8(sinT + pos, s);
    bf16_t* y = qk + (tok * 2 * heads + head) * 64 + j;
#pragma unroll
    for (int k = 0; k < 8; ++k) o[k] = a[k] * c[k] + -b[k] * s[k];
    IO<bf16_t>::store(y, o);
#pragma unroll
    for (int k = 0; k < 8; ++k) o[k] = b[k] * c[k] + a[k] * s[k];
    IO<bf16_t>::store(y + 32, o);
  }
}

// out [b, t, heads, 64] and lse2 [b heads, t] (the base-2 logarithm of each query's sum of exponentials of c times its
// scores, c = log2(e) / 8). A workgroup takes 128 queries, the last blocks (the most keys) first.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_attn_fwd(const bf16_t* __restrict__ qk, const bf16_t* __restrict__ qkv,
                                                  bf16_t* __restrict__ out, float* __restrict__ lse2, int bhs, int t,
                                                  int heads, float c) {
  __shared__ __align__(16) bf16_t s_k[2][AT_N * AT_LD], s_v[2][AT_N * AT_LD];
  const int lane = (int)threadIdx.x & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int blocks = (t + AT_M - 1) / AT_M;
  AttnWork wk;
  if (!attn_work(bhs, blocks, wk)) return;
  const int q0 = (blocks - 1 - wk.block) * AT_M, b = wk.bh / heads, head = wk.bh - b * heads;
  const int64_t sqk = 2 * (int64_t)heads * 64, sv = 3 * (int64_t)heads * 64, so = (int64_t)heads * 64;
  const bf16_t* qp = qk + (int64_t)b * t * sqk + head * 64;
  const bf16_t* kp = qp + heads * 64;
  const bf16_t* vp = qkv + (int64_t)b * t * sv + (2 * heads + head) * 64;
  const int w0 = q0 + 32 * wave, query = w0 + (lane & 31), qrow = min(query, t - 1);
  bf16x8 qf[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
    qf[ks] = frag(*reinterpret_cast<const uint4*>(qp + qrow * sqk + 16 * ks + 8 * half));
  f32x16 o[2] = {zero16(), zero16()};
  float m = -INFINITY, l = 0.f;
  const int ntiles = (min(q0 + AT_M, t) + AT_N - 1) / AT_N;
  Cursor kc(kp, sqk, 0, t), vc(vp, sv, 0, t);
  TileRegs kr = kc.next(), vr = vc.next();
  tile_store(s_k[0], kr);
  tile_store(s_v[0], vr);
  __syncthreads();
  for (int j = 0; j < ntiles; ++j) {
    const int k0 = j * AT_N, cur = j & 1;
    if (j + 1 < ntiles) {
      kr = kc.next();
      vr = vc.next();
    }
    if (k0 <= w0 + 31 && w0 < t) {   // this wave has queries past the tile's first key
      f32x16 s[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        s[i] = zero16();
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) s[i] = mfma(rows_frag(s_k[cur], 32 * i, ks, lane), qf[ks], s[i]);
      }
      if (k0 + AT_N - 1 > w0) {        // keys past the query
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (k0 + 32 * i + 4 * half + (r & 3) + 8 * (r >> 2) > query) s[i][r] = -INFINITY;
      }
      float mx = s[0][0];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[i][r]);
      mx = other_half(mx, false) * c;
      if (__any(mx > m + AT_LAZY)) {
        const float mn = fmaxf(m, mx), a = m == mn ? 1.f : __builtin_amdgcn_exp2f(m - mn);
        m = mn;
        l *= a;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[i][r] *= a;
      }
      float ls[4] = {0.f, 0.f, 0.f, 0.f};   // four sums: no chain of 32 dependent adds
#pragma unroll
      for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          s[i][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i][r], c, -m));
          ls[r & 3] += s[i][r];
        }
#pragma unroll
        for (int st = 0; st < 2; ++st) {
          const bf16x8 p = operand(s[i], st);
#pragma unroll
          for (int d = 0; d < 2; ++d) o[d] = mfma(cols_frag(s_v[cur], 32 * i + 16 * st, 32 * d, lane), p, o[d]);
        }
      }
      l += (ls[0] + ls[1]) + (ls[2] + ls[3]);
    }
    if (j + 1 < ntiles) {
      tile_store(s_k[cur ^ 1], kr);
      tile_store(s_v[cur ^ 1], vr);
      __syncthreads();
    }
  }
  l = other_half(l, true);
  if (query < t) {
    const float inv = 1.f / l;
    bf16_t* op = out + ((int64_t)b * t + query) * so + head * 64 + 4 * half;
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<uint2*>(op + 32 * d + 8 * g) =
            make_uint2(pack2(o[d][4 * g] * inv, o[d][4 * g + 1] * inv), pack2(o[d][4 * g + 2] * inv, o[d][4 * g + 3] * inv));
    if (half == 0) lse2[(int64_t)wk.bh * t + query] = m + __builtin_amdgcn_logf(l);
  }
}

// The gradient of a rotated row, dims j (x) and j + 32 (y) in the registers of a transposed result, turned back and
// stored in bf16 (scaled by `scale`); row: the 64 elements to write, pos: the token's position.
__device__ __forceinline__ void store_unrotated(bf16_t* row, const f32x16& x, const f32x16& y, const float* cosT,
                                                const float* sinT, int pos, int half, float scale) {
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int j = 8 * g + 4 * half;
    const float4 c = *reinterpret_cast<const float4*>(cosT + (int64_t)pos * 64 + j);
    const float4 s = *reinterpret_cast<const float4*>(sinT + (int64_t)pos * 64 + j);
    const float cc[4] = {c.x, c.y, c.z, c.w}, ss[4] = {s.x, s.y, s.z, s.w};
    float a[4], b[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float u = x[4 * g + k] * scale, v = y[4 * g + k] * scale;
      a[k] = u * cc[k] + v * ss[k];
      b[k] = v * cc[k] - u * ss[k];
    }
    *reinterpret_cast<uint2*>(row + j) = make_uint2(pack2(a[0], a[1]), pack2(a[2], a[3]));
    *reinterpret_cast<uint2*>(row + 32 + j) = make_uint2(pack2(b[0], b[1]), pack2(b[2], b[3]));
  }
}

// dq into dqkv's first third, and delta [b heads, t] = sum of dout out for the kernel below. As the forward: 128
// queries per workgroup, the scores and their gradients transposed (columns = queries).
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_attn_bwd_q(
    const bf16_t* __restrict__ qk, const bf16_t* __restrict__ qkv, const bf16_t* __restrict__ out,
    const bf16_t* __restrict__ dout, const float* __restrict__ lse2, const float* __restrict__ cosT,
    const float* __restrict__ sinT, float* __restrict__ delta, bf16_t* __restrict__ dqkv, int bhs, int t, int heads,
    float c, float scale) {
  __shared__ __align__(16) bf16_t s_k[2][AT_N * AT_LD], s_v[2][AT_N * AT_LD];
  const int lane = (int)threadIdx.x & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int blocks = (t + AT_M - 1) / AT_M;
  AttnWork wk;
  if (!attn_work(bhs, blocks, wk)) return;
  const int q0 = (blocks - 1 - wk.block) * AT_M, b = wk.bh / heads, head = wk.bh - b * heads;
  const int64_t sqk = 2 * (int64_t)heads * 64, sv = 3 * (int64_t)heads * 64, so = (int64_t)heads * 64;
  const bf16_t* qp = qk + (int64_t)b * t * sqk + head * 64;
  const bf16_t* kp = qp + heads * 64;
  const bf16_t* vp = qkv + (int64_t)b * t * sv + (2 * heads + head) * 64;
  const int w0 = q0 + 32 * wave, query = w0 + (lane & 31), qrow = min(query, t - 1);
  const int64_t orow = ((int64_t)b * t + qrow) * so + head * 64 + 8 * half;
  bf16x8 qf[4], gf[4];
  float dl = 0.f;
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    qf[ks] = frag(*reinterpret_cast<const uint4*>(qp + qrow * sqk + 16 * ks + 8 * half));
    float g[8], y[8];
    const uint4 gu = *reinterpret_cast<const uint4*>(dout + orow + 16 * ks);
    gf[ks] = frag(gu);
    IO<bf16_t>::unpack(IO<bf16_t>::Raw{gu}, g);
    IO<bf16_t>::load(out + orow + 16 * ks, y);
#pragma unroll
    for (int k = 0; k < 8; ++k) dl = __builtin_fmaf(g[k], y[k], dl);
  }
  dl = other_half(dl, true);
  const float ls = lse2[(int64_t)wk.bh * t + qrow];
  if (query < t && half == 0) delta[(int64_t)wk.bh * t + query] = dl;
  f32x16 dq[2] = {zero16(), zero16()};
  const int ntiles = (min(q0 + AT_M, t) + AT_N - 1) / AT_N;
  Cursor kc(kp, sqk, 0, t), vc(vp, sv, 0, t);
  TileRegs kr = kc.next(), vr = vc.next();
  tile_store(s_k[0], kr);
  tile_store(s_v[0], vr);
  __syncthreads();
  for (int j = 0; j < ntiles; ++j) {
    const int k0 = j * AT_N, cur = j & 1;
    if (j + 1 < ntiles) {
      kr = kc.next();
      vr = vc.next();
    }
    if (k0 <= w0 + 31 && w0 < t) {
      const bool edge = k0 + AT_N - 1 > w0;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        f32x16 s = zero16(), dp = zero16();
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          s = mfma(rows_frag(s_k[cur], 32 * i, ks, lane), qf[ks], s);
          dp = mfma(rows_frag(s_v[cur], 32 * i, ks, lane), gf[ks], dp);
        }
        if (edge) {
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (k0 + 32 * i + 4 * half + (r & 3) + 8 * (r >> 2) > query) s[r] = -INFINITY;
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], c, -ls)) * (dp[r] - dl);
#pragma unroll
        for (int st = 0; st < 2; ++st) {
          const bf16x8 ds = operand(s, st);
#pragma unroll
          for (int d = 0; d < 2; ++d) dq[d] = mfma(cols_frag(s_k[cur], 32 * i + 16 * st, 32 * d, lane), ds, dq[d]);
        }
      }
    }
    if (j + 1 < ntiles) {
      tile_store(s_k[cur ^ 1], kr);
      tile_store(s_v[cur ^ 1], vr);
      __syncthreads();
    }
  }
  if (query < t)
    store_unrotated(dqkv + ((int64_t)b * t + query) * sv + head * 64, dq[0], dq[1], cosT, sinT, query, half, scale);
}

// dk and dv into dqkv's other thirds: 128 keys per workgroup, the first blocks (the most queries) first; the scores as
// they are (columns = keys, rows = queries), each query's lse2 and delta from LDS.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_attn_bwd_kv(
    const bf16_t* __restrict__ qk, const bf16_t* __restrict__ qkv, const bf16_t* __restrict__ dout,
    const float* __restrict__ lse2, const float* __restrict__ delta, const float* __restrict__ cosT,
    const float* __restrict__ sinT, bf16_t* __restrict__ dqkv, int bhs, int t, int heads, float c, float scale) {
  __shared__ __align__(16) bf16_t s_q[2][AT_N * AT_LD], s_g[2][AT_N * AT_LD];
  __shared__ __align__(16) float s_ls[2][AT_N], s_dl[2][AT_N];
  const int lane = (int)threadIdx.x & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int blocks = (t + AT_M - 1) / AT_M;
  AttnWork wk;
  if (!attn_work(bhs, blocks, wk)) return;
  const int k0 = wk.block * AT_M, b = wk.bh / heads, head = wk.bh - b * heads;
  const int64_t sqk = 2 * (int64_t)heads * 64, sv = 3 * (int64_t)heads * 64, so = (int64_t)heads * 64;
  const bf16_t* qp = qk + (int64_t)b * t * sqk + head * 64;
  const bf16_t* gp = dout + (int64_t)b * t * so + head * 64;
  const int w0 = k0 + 32 * wave, key = w0 + (lane & 31), krow = min(key, t - 1);
  const bf16_t* kp = qp + heads * 64 + krow * sqk + 8 * half;
  const bf16_t* vp = qkv + ((int64_t)b * t + krow) * sv + (2 * heads + head) * 64 + 8 * half;
  const float* lp = lse2 + (int64_t)wk.bh * t;
  const float* dp_ = delta + (int64_t)wk.bh * t;
  bf16x8 kf[4], vf[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    kf[ks] = frag(*reinterpret_cast<const uint4*>(kp + 16 * ks));
    vf[ks] = frag(*reinterpret_cast<const uint4*>(vp + 16 * ks));
  }
  f32x16 dk[2] = {zero16(), zero16()}, dv[2] = {zero16(), zero16()};
  const int first = k0 / AT_N, ntiles = (t + AT_N - 1) / AT_N;
  const int tid = (int)threadIdx.x, sr = min(tid, 2 * AT_N - 1);   // lanes 0..63 carry lse2, 64..127 delta
  auto load_scalar = [&](int row0) { return (sr < AT_N ? lp : dp_)[min(row0 + (sr & (AT_N - 1)), t - 1)]; };
  auto put = [&](int buf, const TileRegs& qr, const TileRegs& gr, float sc) {
    tile_store(s_q[buf], qr);
    tile_store(s_g[buf], gr);
    if (tid < AT_N) s_ls[buf][tid] = sc;
    else if (tid < 2 * AT_N) s_dl[buf][tid - AT_N] = sc;
  };
  Cursor qc(qp, sqk, first * AT_N, t), gc(gp, so, first * AT_N, t);
  TileRegs qr = qc.next(), gr = gc.next();
  float sc = load_scalar(first * AT_N);
  put(first & 1, qr, gr, sc);
  __syncthreads();
  for (int j = first; j < ntiles; ++j) {
    const int q0 = j * AT_N, cur = j & 1;
    if (j + 1 < ntiles) {
      qr = qc.next();
      gr = gc.next();
      sc = load_scalar(q0 + AT_N);
    }
    if (q0 + AT_N - 1 >= w0 && w0 < t) {   // the tile has queries at or past this wave's first key
      const bool edge = q0 < w0 + 31 || q0 + AT_N > t;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        f32x16 s = zero16(), dp = zero16();
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          s = mfma(rows_frag(s_q[cur], 32 * i, ks, lane), kf[ks], s);
          dp = mfma(rows_frag(s_g[cur], 32 * i, ks, lane), vf[ks], dp);
        }
        if (edge) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int query = q0 + 32 * i + 4 * half + (r & 3) + 8 * (r >> 2);
            if (key > query || query >= t) s[r] = -INFINITY;
          }
        }
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int r0 = 32 * i + 8 * g + 4 * half;
          const float4 l4 = *reinterpret_cast<const float4*>(&s_ls[cur][r0]);
          const float4 d4 = *reinterpret_cast<const float4*>(&s_dl[cur][r0]);
          const float ll[4] = {l4.x, l4.y, l4.z, l4.w}, dd[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const int r = 4 * g + k;
            s[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], c, -ll[k]));
            dp[r] = s[r] * (dp[r] - dd[k]);
          }
        }
#pragma unroll
        for (int st = 0; st < 2; ++st) {
          const bf16x8 pf = operand(s, st), df = operand(dp, st);
#pragma unroll
          for (int d = 0; d < 2; ++d) {
            dv[d] = mfma(cols_frag(s_g[cur], 32 * i + 16 * st, 32 * d, lane), pf, dv[d]);
            dk[d] = mfma(cols_frag(s_q[cur], 32 * i + 16 * st, 32 * d, lane), df, dk[d]);
          }
        }
      }
    }
    if (j + 1 < ntiles) {
      put(cur ^ 1, qr, gr, sc);
      __syncthreads();
    }
  }
  if (key < t) {
    bf16_t* row = dqkv + ((int64_t)b * t + key) * sv + head * 64;
    store_unrotated(row + heads * 64, dk[0], dk[1], cosT, sinT, key, half, scale);
    bf16_t* vo = row + 2 * heads * 64 + 4 * half;
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<uint2*>(vo + 32 * d + 8 * g) =
            make_uint2(pack2(dv[d][4 * g], dv[d][4 * g + 1]), pack2(dv[d][4 * g + 2], dv[d][4 * g + 3]));
  }
}

// ---------------------------------------------------------------------------------------------------------------
// weight gradient of a bias-free linear layer: dw [n, k] = sum over tokens of dy [tok, n] x [tok, k], bf16 with fp32 sums
//
// A product whose reduction is long (16384 tokens) and whose result is small (a few dozen 256 x 256 tiles): the library
// gives each tile's whole reduction to one workgroup, which leaves most of the 256 CUs idle, and reads both operands
// down their columns. Here the tokens are split so that about one workgroup per CU works (WGRAD_WGS), each on a
// 256 x 256 tile of one run of tokens; the runs' fp32 tiles are summed in order by a second kernel and rounded once.
// 64 tokens of both operands sit in LDS as they lie in memory (two buffers; the next 64 tokens' rows in registers), and
// the matrix cores' operands, columns of those rows, are read with ds_read_b64_tr_b16. An LDS row is 576 bytes: eight
// rows of 64 bytes, what a wave reads at once, then cover the 64 banks twice. Eight waves, 128 x 64 each: 6 KiB of LDS
// reads per eight v_mfma_f32_32x32x16_bf16 (256 cycles), 96 of the LDS's 128 bytes per cycle with two waves per SIMD.
// 16384 tokens, both kernels against the library's product: 2304 x 768 85 us (680 TFLOP/s) and 137, 4096 x 768 128 and
// 156, 768 x 2048 74 and 122, 768 x 768 44 and 95 (a layer's four in its backward: 585 us before, 360 now).
// ---------------------------------------------------------------------------------------------------------------
constexpr int WGRAD_WGS = 256;   // workgroups to split the tokens for
constexpr int WT = 256, WK = 64, W_LD = 288, W_LANES = 512;   // tile edge, tokens per step, LDS row, lanes

__global__ __launch_bounds__(W_LANES) __attribute__((amdgpu_waves_per_eu(2))) void k_wgrad(
    const bf16_t* __restrict__ dy, const bf16_t* __restrict__ x, float* __restrict__ part, int64_t m, int n, int k,
    int tiles_k, int tiles, int splits, int64_t run, int per) {
  __shared__ __align__(16) bf16_t w_lds[4 * WK * W_LD];   // [2 buffers][dy, x][WK][W_LD]
  // XCD x (workgroups go to XCDs in turn) takes `per` consecutive (run, tile) pairs, mostly of one run of tokens: its
  // rows are then read from memory once per XCD
  const int id = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
  if (id >= tiles * splits || (int)blockIdx.x >> 3 >= per) return;
  const int split = id / tiles, tile = id - split * tiles, n0 = (tile / tiles_k) * WT, k0 = (tile % tiles_k) * WT;
  const int64_t t0 = split * run, t1 = min(m, t0 + run);
  const int tid = (int)threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wn = 128 * (wave >> 2), wk = 64 * (wave & 3);
  const int row = tid >> 5, col = 8 * (tid & 31);   // this lane's pieces: rows row + 16 i, columns col .. col + 8
  const bf16_t* pa = dy + (t0 + row) * n + min(n0 + col, n - 8);
  const bf16_t* pb = x + (t0 + row) * k + min(k0 + col, k - 8);
  uint4 ra[4], rb[4];
  auto load = [&](int64_t tok) {   // rows past the run's end: zeros, from its last row's address
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t over = tok + row + 16 * i - (t1 - 1);
      const bool ok = over <= 0;
      const int64_t back = ok ? 0 : over;
      ra[i] = *reinterpret_cast<const uint4*>(pa + (16 * i - back) * n);
      rb[i] = *reinterpret_cast<const uint4*>(pb + (16 * i - back) * k);
      if (!ok) ra[i] = rb[i] = make_uint4(0u, 0u, 0u, 0u);
    }
    pa += (int64_t)WK * n;
    pb += (int64_t)WK * k;
  };
  auto store = [&](int buf) {
    bf16_t* a = w_lds + buf * 2 * WK * W_LD;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      *reinterpret_cast<uint4*>(a + (row + 16 * i) * W_LD + col) = ra[i];
      *reinterpret_cast<uint4*>(a + (WK + row + 16 * i) * W_LD + col) = rb[i];
    }
  };
  f32x16 acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = zero16();
  load(t0);
  store(0);
  __syncthreads();
  int buf = 0;
  for (int64_t tok = t0; tok < t1; tok += WK, buf ^= 1) {
    const bool more = tok + WK < t1;   // workgroup-uniform
    if (more) load(tok + WK);
    const bf16_t* a = w_lds + buf * 2 * WK * W_LD;
    const bf16_t* b = a + WK * W_LD;
#pragma unroll
    for (int s = 0; s < WK; s += 16) {
      bf16x8 fa[4], fb[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) fb[j] = cols_frag<W_LD>(b, s, wk + 32 * j, lane);
#pragma unroll
      for (int i = 0; i < 4; ++i) fa[i] = cols_frag<W_LD>(a, s, wn + 32 * i, lane);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma(fa[i], fb[j], acc[i][j]);
    }
    if (more) {
      store(buf ^ 1);
      __syncthreads();
    }
  }
  float* out = part + (int64_t)split * n * k;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int c = k0 + wk + 32 * j + (lane & 31);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int rr = n0 + wn + 32 * i + 4 * (lane >> 5) + (r & 3) + 8 * (r >> 2);
        if (rr < n && c < k) out[(int64_t)rr * k + c] = acc[i][j][r];
      }
    }
}

// dw = round(sum of the runs' tiles, in order), eight elements per lane
__global__ __launch_bounds__(WG) void k_wgrad_sum(const float* __restrict__ part, int splits, int64_t nk,
                                                  bf16_t* __restrict__ dw) {
  for (int64_t i = 8 * ((int64_t)blockIdx.x * WG + threadIdx.x); i < nk; i += 8 * (int64_t)gridDim.x * WG) {
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    int s = 0;
    for (; s + 4 <= splits; s += 4) {   // four runs' loads in flight
      float e[4][8];
#pragma unroll
      for (int u = 0; u < 4; ++u) load_f32x8(part + (s + u) * nk + i, e[u]);
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int x = 0; x < 8; ++x) acc[x] += e[u][x];
    }
    for (; s < splits; ++s) {
      float e[8];
      load_f32x8(part + s * nk + i, e);
#pragma unroll
      for (int x = 0; x < 8; ++x) acc[x] += e[x];
    }
    IO<bf16_t>::store(dw + i, acc);
  }
}

inline bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
inline bool al2(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 1u) == 0; }
inline bool dtype_ok(int dt) { return dt == LDR_BF16 || dt == LDR_F16; }
inline unsigned grid_of(int64_t blocks, int64_t cap) { return (unsigned)(blocks < cap ? blocks : cap); }
inline int launched() { return (int)hipGetLastError(); }

#define LLM_DTYPE_SWITCH(DT, ...)                                \
  if ((DT) == LDR_BF16) { typedef bf16_t T; __VA_ARGS__; }       \
  else { typedef _Float16 T; __VA_ARGS__; }
#define LLM_VPT_SWITCH(V, ...)                                   \
  switch (V) {                                                   \
    case 1: { constexpr int VPT = 1; __VA_ARGS__; } break;       \
    case 2: { constexpr int VPT = 2; __VA_ARGS__; } break;       \
    case 3: { constexpr int VPT = 3; __VA_ARGS__; } break;       \
    default: { constexpr int VPT = 4; __VA_ARGS__; } break;      \
  }

}  // namespace

extern "C" {

int llm_abi_version(void) { return LLM_ABI_VERSION; }

int llm_rms_norm_fwd(const void* x, const void* add, const void* w, void* h_out, void* y, float* rstd, int64_t rows,
                     int64_t d, float eps, int dtype, void* stream) {
  if (!dtype_ok(dtype)) return LDR_E_DTYPE;
  if (d < 8 || (d & 7) || d > LLM_NORM_MAX_WIDTH) return LDR_E_SHAPE;
  if (rows < 0 || !w) return LDR_E_ARG;
  if (rows == 0) return LDR_OK;
  if (!x || !y || !rstd || (add && !h_out)) return LDR_E_ARG;
  if (!al16(x) || !al16(w) || !al16(y) || (add && (!al16(add) || !al16(h_out)))) return LDR_E_ALIGN;
  const int vpt = (int)((d / 8 + 63) / 64);
  LLM_DTYPE_SWITCH(dtype, LLM_VPT_SWITCH(vpt, hipLaunchKernelGGL((k_rms_norm_fwd<T, VPT>),
      dim3(grid_of((rows + WAVES - 1) / WAVES, 4096)), dim3(WG), 0, static_cast<hipStream_t>(stream),
      static_cast<const T*>(x), static_cast<const T*>(add), static_cast<const T*>(w), static_cast<T*>(h_out),
      static_cast<T*>(y), rstd, rows, (int)d, eps)))
  return launched();
}

int64_t llm_rms_norm_parts(int64_t rows) { return rows < 1 ? 0 : grid_of((rows + WAVES - 1) / WAVES, NORM_GRID); }

int llm_rms_norm_bwd(const void* dy, const void* h, const void* w, const float* rstd, const void* dres, void* dx,
                     float* dw_part, int64_t rows, int64_t d, int dtype, void* stream) {
  if (!dtype_ok(dtype)) return LDR_E_DTYPE;
  if (d < 8 || (d & 7) || d > LLM_NORM_MAX_WIDTH) return LDR_E_SHAPE;
  if (rows < 0 || !w) return LDR_E_ARG;
  if (rows == 0) return LDR_OK;
  if (!dy || !h || !rstd || (!dx && !dw_part)) return LDR_E_ARG;
  if (!al16(dy) || !al16(h) || !al16(w) || !al16(dx) || !al16(dres)) return LDR_E_ALIGN;
  const int vpt = (int)((d / 8 + 63) / 64);
  LLM_DTYPE_SWITCH(dtype, LLM_VPT_SWITCH(vpt, hipLaunchKernelGGL((k_rms_norm_bwd<T, VPT>),
      dim3((unsigned)llm_rms_norm_parts(rows)), dim3(WG), 0, static_cast<hipStream_t>(stream),
      static_cast<const T*>(dy), static_cast<const T*>(h), static_cast<const T*>(w), rstd, static_cast<const T*>(dres),
      static_cast<T*>(dx), dw_part, rows, (int)d)))
  return launched();
}

int llm_sum_rows(const float* part, int64_t rows, int64_t d, void* out, int dtype, void* stream) {
  if (!dtype_ok(dtype)) return LDR_E_DTYPE;
  if (!out || rows < 0 || d < 1 || (rows > 0 && !part)) return LDR_E_ARG;
  LLM_DTYPE_SWITCH(dtype, hipLaunchKernelGGL(k_sum_rows<T>, dim3((unsigned)((d + 15) / 16)), dim3(WG), 0,
                                             static_cast<hipStream_t>(stream), part, rows, (int)d,
                                             static_cast<T*>(out)))
  return launched();
}

int llm_swiglu_fwd(const void* gate_up, void* act, int64_t rows, int64_t n, int dtype, void* stream) {
  if (!dtype_ok(dtype)) return LDR_E_DTYPE;
  if (n < 8 || (n & 7)) return LDR_E_SHAPE;
  if (rows < 0) return LDR_E_ARG;
  if (rows == 0) return LDR_OK;
  if (!gate_up || !act) return LDR_E_ARG;
  if (!al16(gate_up) || !al16(act)) return LDR_E_ALIGN;
  const int64_t nvec = rows * (n / 8);
  LLM_DTYPE_SWITCH(dtype, hipLaunchKernelGGL(k_swiglu_fwd<T>, dim3(grid_of((nvec + WG - 1) / WG, 8192)), dim3(WG), 0,
                                             static_cast<hipStream_t>(stream), static_cast<const T*>(gate_up),
                                             static_cast<T*>(act), nvec, (int)(n / 8)))
  return launched();
}

int llm_swiglu_bwd(const void* gate_up, const void* dact, void* dgate_up, int64_t rows, int64_t n, int dtype,
                   void* stream) {
  if (!dtype_ok(dtype)) return LDR_E_DTYPE;
  if (n < 8 || (n & 7)) return LDR_E_SHAPE;
  if (rows < 0) return LDR_E_ARG;
  if (rows == 0) return LDR_OK;
  if (!gate_up || !dact || !dgate_up) return LDR_E_ARG;
  if (!al16(gate_up) || !al16(dact) || !al16(dgate_up)) return LDR_E_ALIGN;
  const int64_t nvec = rows * (n / 8);
  LLM_DTYPE_SWITCH(dtype, hipLaunchKernelGGL(k_swiglu_bwd<T>, dim3(grid_of((nvec + WG - 1) / WG, 8192)), dim3(WG), 0,
                                             static_cast<hipStream_t>(stream), static_cast<const T*>(gate_up),
                                             static_cast<const T*>(dact), static_cast<T*>(dgate_up), nvec,
                                             (int)(n / 8)))
  return launched();
}

int llm_next_token_loss_fwd(const void* logits, const int64_t* ids, float* lse, float* scratch, float* loss, int64_t b,
                            int64_t t, int64_t vocab, int dtype, void* stream) {
  if (!dtype_ok(dtype)) return LDR_E_DTYPE;
  if (b < 0 || t < 0 || vocab < 1 || !loss || b * t > 0x7fffffff) return LDR_E_ARG;
  const int64_t rows = b * t;
  if (rows > 0 && (!logits || !ids || !lse || !scratch)) return LDR_E_ARG;
  if (!al2(logits)) return LDR_E_ALIGN;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (rows > 0) {
    LLM_DTYPE_SWITCH(dtype, hipLaunchKernelGGL(k_next_token_fwd<T>, dim3((unsigned)rows), dim3(WG), 0, st,
                                               static_cast<const T*>(logits), ids, lse, scratch, t, vocab))
    const int e = launched();
    if (e) return e;
  }
  hipLaunchKernelGGL(k_mean, dim3(1), dim3(1024), 0, st, scratch, rows, rows > 0 ? (float)(b * (t - 1)) : 0.f, loss);
  return launched();
}

int llm_next_token_loss_bwd(const void* logits, const int64_t* ids, const float* lse, const float* dloss, void* dlogits,
                            int64_t b, int64_t t, int64_t vocab, int dtype, void* stream) {
  if (!dtype_ok(dtype)) return LDR_E_DTYPE;
  if (b < 0 || t < 0 || vocab < 1 || b * t > 0x7fffffff) return LDR_E_ARG;
  if (b * t == 0) return LDR_OK;
  if (!logits || !ids || !lse || !dloss || !dlogits) return LDR_E_ARG;
  if (!al2(logits) || !al2(dlogits)) return LDR_E_ALIGN;
  const double count = (double)b * (double)(t - 1);
  LLM_DTYPE_SWITCH(dtype, hipLaunchKernelGGL(k_next_token_bwd<T>, dim3((unsigned)(b * t)), dim3(WG), 0,
                                             static_cast<hipStream_t>(stream), static_cast<const T*>(logits), ids, lse,
                                             dloss, static_cast<T*>(dlogits), t, vocab,
                                             count > 0 ? (float)(1.0 / count) : 0.f))
  return launched();
}

int llm_rotary(const void* qkv, const float* cosT, const float* sinT, void* qk, int64_t b, int64_t t, int64_t heads,
               void* stream) {
  if (b < 0 || t < 0 || heads < 1 || b * t * heads > 0x7fffffff) return LDR_E_ARG;
  if (b * t == 0) return LDR_OK;
  if (!qkv || !cosT || !sinT || !qk) return LDR_E_ARG;
  if (!al16(qkv) || !al16(cosT) || !al16(sinT) || !al16(qk)) return LDR_E_ALIGN;
  const int64_t n = b * t * heads * 8;
  hipLaunchKernelGGL(k_rotary, dim3(grid_of((n + WG - 1) / WG, 8192)), dim3(WG), 0, static_cast<hipStream_t>(stream),
                     static_cast<const bf16_t*>(qkv), cosT, sinT, static_cast<bf16_t*>(qk), n, (int)t, (int)heads);
  return launched();
}

static int attn_grid(int64_t b, int64_t t, int64_t heads, unsigned* grid) {
  if (b < 0 || t < 0 || heads < 1 || b * heads > 0x7fffff || t > 0x7fffff) return LDR_E_ARG;
  const int64_t g = 8 * ((b * heads + 7) / 8) * ((t + AT_M - 1) / AT_M);
  if (g > 0x7fffffff) return LDR_E_SHAPE;
  *grid = (unsigned)g;
  return LDR_OK;
}

int llm_attn_fwd(const void* qk, const void* qkv, void* out, float* lse2, int64_t b, int64_t t, int64_t heads,
                 void* stream) {
  unsigned grid = 0;
  const int e = attn_grid(b, t, heads, &grid);
  if (e) return e;
  if (grid == 0) return LDR_OK;
  if (!qk || !qkv || !out || !lse2) return LDR_E_ARG;
  if (!al16(qk) || !al16(qkv) || !al16(out)) return LDR_E_ALIGN;
  hipLaunchKernelGGL(k_attn_fwd, dim3(grid), dim3(256), 0, static_cast<hipStream_t>(stream),
                     static_cast<const bf16_t*>(qk), static_cast<const bf16_t*>(qkv), static_cast<bf16_t*>(out), lse2,
                     (int)(b * heads), (int)t, (int)heads, AT_SCALE * LOG2E);
  return launched();
}

int llm_attn_bwd(const void* qk, const void* qkv, const void* out, const void* dout, const float* lse2,
                 const float* cosT, const float* sinT, float* delta, void* dqkv, int64_t b, int64_t t, int64_t heads,
                 void* stream) {
  unsigned grid = 0;
  int e = attn_grid(b, t, heads, &grid);
  if (e) return e;
  if (grid == 0) return LDR_OK;
  if (!qk || !qkv || !out || !dout || !lse2 || !cosT || !sinT || !delta || !dqkv) return LDR_E_ARG;
  if (!al16(qk) || !al16(qkv) || !al16(out) || !al16(dout) || !al16(cosT) || !al16(sinT) || !al16(dqkv))
    return LDR_E_ALIGN;
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(k_attn_bwd_q, dim3(grid), dim3(256), 0, st, static_cast<const bf16_t*>(qk),
                     static_cast<const bf16_t*>(qkv), static_cast<const bf16_t*>(out),
                     static_cast<const bf16_t*>(dout), lse2, cosT, sinT, delta, static_cast<bf16_t*>(dqkv),
                     (int)(b * heads), (int)t, (int)heads, AT_SCALE * LOG2E, AT_SCALE);
  if ((e = launched())) return e;
  hipLaunchKernelGGL(k_attn_bwd_kv, dim3(grid), dim3(256), 0, st, static_cast<const bf16_t*>(qk),
                     static_cast<const bf16_t*>(qkv), static_cast<const bf16_t*>(dout), lse2, delta, cosT, sinT,
                     static_cast<bf16_t*>(dqkv), (int)(b * heads), (int)t, (int)heads, AT_SCALE * LOG2E, AT_SCALE);
  return launched();
}

// the runs of tokens llm_wgrad splits m into: about one workgroup per CU, runs of at least 512 tokens (a run's fp32 tile
// is written and read again: 512 KiB for the 512 KiB of operands that 512 tokens are)
int64_t llm_wgrad_splits(int64_t m, int64_t n, int64_t k) {
  if (m < 1 || n < 8 || k < 8) return 0;
  const int64_t tiles = ((n + WT - 1) / WT) * ((k + WT - 1) / WT), fill = WGRAD_WGS / tiles, most = m / 512;
  const int64_t s = fill < most ? fill : most;
  return s < 1 ? 1 : s;
}

int llm_wgrad(const void* dy, const void* x, float* part, void* dw, int64_t m, int64_t n, int64_t k, void* stream) {
  if (m < 0 || n < 8 || k < 8 || (n & 7) || (k & 7) || n > 0x7fffff || k > 0x7fffff) return LDR_E_SHAPE;
  if (!dw || m < 1 || !dy || !x || !part) return LDR_E_ARG;
  if (!al16(dy) || !al16(x) || !al16(part) || !al16(dw)) return LDR_E_ALIGN;
  const int64_t tn = (n + WT - 1) / WT, tk = (k + WT - 1) / WT, tiles = tn * tk, splits = llm_wgrad_splits(m, n, k);
  if (tiles * splits > 0xffffff) return LDR_E_SHAPE;
  const int64_t run = ((m + splits - 1) / splits + WK - 1) / WK * WK, runs = (m + run - 1) / run;
  const int64_t per = (tiles * runs + 7) / 8;
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(k_wgrad, dim3((unsigned)(8 * per)), dim3(W_LANES), 0, st, static_cast<const bf16_t*>(dy),
                     static_cast<const bf16_t*>(x), part, m, (int)n, (int)k, (int)tk, (int)tiles, (int)runs, run,
                     (int)per);
  const int e = launched();
  if (e) return e;
  hipLaunchKernelGGL(k_wgrad_sum, dim3(grid_of((n * k / 8 + WG - 1) / WG, 4096)), dim3(WG), 0, st, part, (int)runs,
                     n * k, static_cast<bf16_t*>(dw));
  return launched();
}

}  // extern "C"
