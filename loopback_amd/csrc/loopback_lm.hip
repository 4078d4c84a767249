// loopback_lm.hip -- MI355X (gfx950, CDNA4) kernels of the language model around the Loopback read: RMSNorm, SwiGLU
// and the next-token cross entropy, forward and backward. All are bound by the HBM stream of their rows, and torch's
// composed forms move those rows several times (an fp32 copy of the logits, the softmax, its gradient and its cast;
// silu and the product; the norm's gradient, its weight's gradient and the residual's add): each is one pass here,
// with fp32 statistics and one rounding per result. Every sum has a fixed order: results are deterministic.

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
// in LDS, one partial row per workgroup.
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
  if (!dy || !h || !rstd || !dx || !dw_part) return LDR_E_ARG;
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

}  // extern "C"
