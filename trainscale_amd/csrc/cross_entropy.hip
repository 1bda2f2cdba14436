// Vocabulary cross-entropy forward/backward for gfx950.
//
// Rows start anywhere: a row of a [N, V] tensor whose V is no multiple of the 16-byte
// vector (GPT-2's 50257 in bf16) lies on no 16-byte boundary. Lanes own the same elements
// of a row whatever its address, so a result does not depend on strides or alignment:
// whole vectors from the row's first element on, read and written with 16-byte accesses
// at element alignment, and the V % VE elements after the last vector one each by the
// row's first lanes (ts_plan::tail_col). Measured on MI355X at [7959, 50257]
// bf16, against kernels that went element by element: loss and gradient 1033 -> 359 us,
// forward alone 437 -> 161 us, backward alone 603 -> 259 us.
//
// Forward: one 256-thread workgroup per row. Each lane streams the row with
// 16-byte non-temporal loads (kUnroll vectors in flight per lane) and keeps an
// online (max, sum of exp) pair: a new chunk's max rescales the running sum
// once per chunk, not once per element. exp is evaluated as
// exp2(z*log2(e) - m*log2(e)) with one FMA and one v_exp_f32. The per-lane
// pairs are folded with a wave64 DPP max, a rescale, and DPP sums, then across
// the four waves through LDS. Rows whose label is ignore_index are not read:
// their loss is 0 and their lse is stored as 0 (the backward never reads it).
//
// Backward: one read and one write per element, grad = dloss * (softmax -
// onehot) (with the label-smoothing, softcap and logit-scale chain rules),
// written with 16-byte stores; it may overwrite the logits in place. The grid
// is one-shot over (row, chunk of 256 vectors) with one vector per thread:
// on MI355X a streaming kernel with few accesses per thread keeps more of HBM
// busy than one that loops along a row, or than two vectors per thread. Ignored rows are written as zeros
// without being read.
#include "cross_entropy.hpp"

namespace {

using namespace ts;
using namespace ts_ce;

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;
constexpr int kUnroll = 4;   // vectors in flight per lane in the forward's row loop
// Vectors per thread in the backward's one-shot grid: one measured 1.304 ms
// against 1.405 ms with two at C3 [16384, 128256] bf16 on MI355X.
constexpr int kBwdKv = 1;
constexpr int64_t kMaxGridY = 65535;  // rows per backward launch

// Block-wide (max, sum exp, sum z) fold. Every thread receives the results.
__device__ inline void block_fold(float& m, float& s, float& sz, float* lds) {
  float bm = wave_max(m);
  const int wid = threadIdx.x / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  if (lane == 0) lds[wid] = bm;
  __syncthreads();
  bm = lds[0];
#pragma unroll
  for (int i = 1; i < kWaves; ++i) bm = fmaxf(bm, lds[i]);
  __syncthreads();
  // Rescale this lane's sum to the row max. A lane that saw only -inf has
  // s == 0 and contributes nothing.
  const float scaled = s == 0.f ? 0.f : s * fast_exp2((m - bm) * kLog2e);
  float ws = wave_sum(scaled);
  float wz = wave_sum(sz);
  if (lane == 0) {
    lds[wid] = ws;
    lds[kWaves + wid] = wz;
  }
  __syncthreads();
  float ts = 0.f, tz = 0.f;
#pragma unroll
  for (int i = 0; i < kWaves; ++i) {
    ts += lds[i];
    tz += lds[kWaves + i];
  }
  m = bm;
  s = ts;
  sz = tz;
}

template <typename T, int kMode>
__global__ __launch_bounds__(kThreads) void ce_fwd_vec(const T* __restrict__ logits, int64_t ld,
                                                       const int64_t* __restrict__ labels,
                                                       int64_t V, int64_t ignore_index, Xform xf,
                                                       float smoothing, float* __restrict__ loss,
                                                       float* __restrict__ lse_out) {
  constexpr int VE = Elt<T>::kVec;
  __shared__ float lds[2 * kWaves];
  const int64_t row = blockIdx.x;
  const int64_t label = labels[row];
  if (label == ignore_index) {
    if (threadIdx.x == 0) {
      loss[row] = 0.f;
      lse_out[row] = 0.f;
    }
    return;
  }
  const T* xr = logits + row * ld;
  const int64_t nvec = V / VE;
  const int64_t ec = tail_col<VE>(V);
  float m = -INFINITY, s = 0.f, sz = 0.f;
  // whole chunks of kThreads * kUnroll vectors (ts_plan::chunk_vec), then the rest
  const int64_t full = nvec / ((int64_t)kThreads * kUnroll);
  int64_t c = 0;
  for (; c < full; ++c) {
    u32x4 buf[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u)
      buf[u] = ld16_any_stream(xr + ts_plan::chunk_vec(c, u, threadIdx.x, kThreads, kUnroll) * VE);
    float z[kUnroll][VE];
    float lm = -INFINITY;
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      Elt<T>::unpack(buf[u], z[u]);
      xform_vec<kMode, VE>(z[u], xf);
#pragma unroll
      for (int i = 0; i < VE; ++i) {
        lm = fmaxf(lm, z[u][i]);
        if constexpr (kMode != kPlain) sz += z[u][i];
      }
    }
    if (lm > m) {
      s = s == 0.f ? 0.f : s * fast_exp2((m - lm) * kLog2e);
      m = lm;
    }
    if (fabsf(m) < kRefMax) {
      const float mb = m * kLog2e;
      float cs = 0.f;
#pragma unroll
      for (int u = 0; u < kUnroll; ++u)
#pragma unroll
        for (int i = 0; i < VE; ++i) cs += fast_exp2(__builtin_fmaf(z[u][i], kLog2e, -mb));
      s += __builtin_fmaf(cs, -bias_lack(m, mb), cs);
    } else {
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) s += sum_exp_far<VE>(z[u], m);
    }
  }
  // Tail: fewer than kThreads*kUnroll vectors remain.
  for (int64_t v = ts_plan::chunk_vec(c, 0, threadIdx.x, kThreads, kUnroll); v < nvec;
       v += kThreads) {  // chunk_vec(c, u, ...) for u = 0, 1, ...
    float z[VE];
    Elt<T>::unpack(ld16_any_stream(xr + v * VE), z);
    xform_vec<kMode, VE>(z, xf);
    float lm = -INFINITY;
#pragma unroll
    for (int i = 0; i < VE; ++i) {
      lm = fmaxf(lm, z[i]);
      if constexpr (kMode != kPlain) sz += z[i];
    }
    if (lm > m) {
      s = s == 0.f ? 0.f : s * fast_exp2((m - lm) * kLog2e);
      m = lm;
    }
    if (fabsf(m) < kRefMax) {
      const float mb = m * kLog2e;
      float cs = 0.f;
#pragma unroll
      for (int i = 0; i < VE; ++i) cs += fast_exp2(__builtin_fmaf(z[i], kLog2e, -mb));
      s += __builtin_fmaf(cs, -bias_lack(m, mb), cs);
    } else {
      s += sum_exp_far<VE>(z, m);
    }
  }
  if (ec >= 0) {
    const float ze = xform1<kMode>(Elt<T>::load1(xr + ec), xf);
    fold1(ze, m, s);
    if constexpr (kMode != kPlain) sz += ze;
  }
  block_fold(m, s, sz, lds);
  if (threadIdx.x == 0) {
    const float l = log_sum(m, s);
    loss[row] = row_loss<kMode>(xr, label, V, ignore_index, l, sz, smoothing, xf);
    lse_out[row] = l;
  }
}

// Stores one vector of VE gradients (as one or two 16-byte stores).
template <typename G, int VE>
__device__ inline void store_grad(G* p, const float* g) {
  if constexpr (sizeof(G) == 4 && VE == 8) {
    st16_any_stream(p, Elt<float>::pack(g));
    st16_any_stream(p + 4, Elt<float>::pack(g + 4));
  } else {
    st16_any_stream(p, Elt<G>::pack(g));
  }
}

// One-shot grid: blockIdx.y is the row (offset by row0), blockIdx.x a chunk
// of kThreads * kBwdKv vectors of it; each thread handles kBwdKv vectors, and the
// first lanes of chunk 0 the elements after the row's last vector.
template <typename T, typename G, int kMode>
__global__ __launch_bounds__(kThreads) void ce_bwd_vec(
    const T* logits, int64_t ld, const int64_t* __restrict__ labels,
    const float* __restrict__ lse, const float* __restrict__ dloss, int64_t dloss_stride,
    float dloss_scale, G* grad, int64_t ld_grad, int64_t V, int64_t nvec, int64_t ignore_index,
    Xform xf, float smoothing, int64_t row0) {
  constexpr int VE = Elt<T>::kVec;
  static_assert(Elt<G>::kVec == VE || sizeof(G) == 4, "grad vector width");
  const int64_t row = row0 + blockIdx.y;
  const int64_t label = labels[row];
  const T* xr = logits + row * ld;
  G* gr = grad + row * ld_grad;
  // uniform: only the first chunk of rows that are not whole vectors runs the tail's code
  const bool has_tail = blockIdx.x == 0 && V % VE != 0;
  int64_t vk[kBwdKv];  // this thread's vectors of the row (ts_plan::chunk_vec)
#pragma unroll
  for (int k = 0; k < kBwdKv; ++k)
    vk[k] = ts_plan::chunk_vec(blockIdx.x, k, threadIdx.x, kThreads, kBwdKv);
  if (label == ignore_index) {
    const float zero[VE] = {};
#pragma unroll
    for (int k = 0; k < kBwdKv; ++k) {
      if (vk[k] < nvec) store_grad<G, VE>(gr + vk[k] * VE, zero);
    }
    if (has_tail) {
      const int64_t ec = tail_col<VE>(V);
      if (ec >= 0) Elt<G>::store1(gr + ec, 0.f);
    }
    return;
  }
  GradRow r;
  r.dl = dloss[row * dloss_stride] * dloss_scale;
  r.lse2 = lse[row] * kLog2e;
  set_smoothing(r, smoothing, V);
  u32x4 buf[kBwdKv];
#pragma unroll
  for (int k = 0; k < kBwdKv; ++k) {
    const int64_t v = vk[k];
    buf[k] = v < nvec ? ld16_any_stream(xr + v * VE) : u32x4{0, 0, 0, 0};
  }
  if (has_tail) {
    const int64_t ec = tail_col<VE>(V);
    if (ec >= 0)
      Elt<G>::store1(gr + ec, grad1<kMode>(Elt<T>::load1(xr + ec), ec == label, r, xf));
  }
#pragma unroll
  for (int k = 0; k < kBwdKv; ++k) {
    const int64_t v = vk[k];
    if (v < nvec) {
      float x[VE], g[VE];
      Elt<T>::unpack(buf[k], x);
      // modulo 2^64, so that no label overflows the difference
      const int64_t lab = (int64_t)((uint64_t)label - (uint64_t)(v * VE));
      grad_vec<kMode, VE>(x, g, lab, r, xf);
      store_grad<G, VE>(gr + v * VE, g);
    }
  }
}

// ---------------------------------------------------------------------------
// The reductions around the row losses. One workgroup each, fixed order; a wave keeps
// kRedUnroll loads of every lane in flight, so 16384 rows take two round trips to memory.
// Each replaces half a dozen elementwise and reduction launches of a few microseconds:
// on MI355X the mean loss and gradient of [2048, 32000] fp32 logits went from 202 to 133 us,
// of [16384, 128256] bf16 logits from 1380 to 1349.
// ---------------------------------------------------------------------------
constexpr int kRedThreads = 1024;
constexpr int kRedWaves = kRedThreads / kWave;
constexpr int kRedUnroll = 8;

// Rows whose label is not ignore_index; thread 0 receives the count. lds: kRedWaves values.
__device__ inline int64_t count_valid(const int64_t* __restrict__ labels, int64_t N,
                                      int64_t ignore_index, int64_t* lds) {
  int64_t c = 0;  // of this lane
  for (int64_t i0 = threadIdx.x; i0 < N; i0 += (int64_t)kRedThreads * kRedUnroll) {
    int64_t l[kRedUnroll];
#pragma unroll
    for (int u = 0; u < kRedUnroll; ++u) {
      const int64_t i = i0 + u * kRedThreads;
      l[u] = i < N ? labels[i] : ignore_index;
    }
#pragma unroll
    for (int u = 0; u < kRedUnroll; ++u) c += l[u] != ignore_index;
  }
  for (int h = 32; h >= 1; h >>= 1) c += __shfl_down((long long)c, h);
  if ((threadIdx.x & (kWave - 1)) == 0) lds[threadIdx.x / kWave] = c;
  __syncthreads();
  int64_t t = 0;
  if (threadIdx.x == 0)
    for (int i = 0; i < kRedWaves; ++i) t += lds[i];
  return t;
}

__global__ __launch_bounds__(kRedThreads) void ce_loss_weight(
    const int64_t* __restrict__ labels, int64_t N, int64_t ignore_index, int mean, float fixed,
    const float* __restrict__ hint, float* __restrict__ weight, float* __restrict__ used) {
  __shared__ int64_t lds[kRedWaves];
  float w = fixed;
  if (mean) {
    const int64_t c = count_valid(labels, N, ignore_index, lds);
    w = 1.f / (float)(c > 0 ? c : 1);
  }
  if (threadIdx.x != 0) return;
  const float h = hint != nullptr ? *hint : 1.f;
  *weight = w * h;
  if (used != nullptr) *used = h;
}

// The sum in double, rounded once after the division: its order then costs nothing in fp32.
__global__ __launch_bounds__(kRedThreads) void ce_reduce_loss(
    const float* __restrict__ rows, const int64_t* __restrict__ labels, int64_t N,
    int64_t ignore_index, int mean, float div, float* __restrict__ out) {
  __shared__ int64_t cnt[kRedWaves];
  __shared__ double sums[kRedWaves];
  double s = 0.0;
  for (int64_t i0 = threadIdx.x; i0 < N; i0 += (int64_t)kRedThreads * kRedUnroll) {
    float v[kRedUnroll];
#pragma unroll
    for (int u = 0; u < kRedUnroll; ++u) {
      const int64_t i = i0 + u * kRedThreads;
      v[u] = i < N ? rows[i] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < kRedUnroll; ++u) s += (double)v[u];
  }
  for (int h = 32; h >= 1; h >>= 1) s += __shfl_down(s, h);
  if ((threadIdx.x & (kWave - 1)) == 0) sums[threadIdx.x / kWave] = s;
  const int64_t c = mean ? count_valid(labels, N, ignore_index, cnt) : 0;
  __syncthreads();
  if (threadIdx.x != 0) return;
  double t = 0.0;
  for (int i = 0; i < kRedWaves; ++i) t += sums[i];
  *out = (float)(t / (mean ? (double)(c > 0 ? c : 1) : (double)div));
}

template <typename T>
ts_status fwd_typed(const void* logits, int64_t ld, const int64_t* labels, int64_t N, int64_t V,
                    int64_t ignore_index, Xform xf, Mode mode, float smoothing, float* loss,
                    float* lse, hipStream_t st) {
  const T* lp = static_cast<const T*>(logits);
  const dim3 grid((unsigned)N), block(kThreads);
#define TS_CE_FWD(M)                                                                          \
  if (mode == M) {                                                                            \
    hipLaunchKernelGGL((ce_fwd_vec<T, M>), grid, block, 0, st, lp, ld, labels, V,             \
                       ignore_index, xf, smoothing, loss, lse);                               \
    return ts_host::check_launch("ce_fwd_vec");                                               \
  }
  TS_CE_FWD(kPlain)
  TS_CE_FWD(kSmooth)
  TS_CE_FWD(kGeneral)
#undef TS_CE_FWD
  return ts_host::fail(TS_ERR_INVALID_ARGUMENT, "ce_fwd: unreachable");
}

template <typename T, typename G>
ts_status bwd_typed(const void* logits, int64_t ld, const int64_t* labels, const float* lse,
                    const float* dloss, int64_t dloss_stride, float dloss_scale, void* grad,
                    int64_t ld_grad, int64_t N, int64_t V, int64_t ignore_index, Xform xf,
                    Mode mode, float smoothing, hipStream_t st) {
  constexpr int VE = sizeof(T) == 4 ? 4 : 8;
  const T* lp = static_cast<const T*>(logits);
  G* gp = static_cast<G*>(grad);
  const dim3 block(kThreads);
  // chunk 0 also holds the elements after a row's last vector
  const int64_t chunks = ts_plan::chunks_for(V / VE, kThreads, kBwdKv);
  const unsigned gx = chunks > 0 ? (unsigned)chunks : 1u;
#define TS_CE_BWD(M)                                                                           \
  if (mode == M) {                                                                             \
    for (int64_t r0 = 0; r0 < N; r0 += kMaxGridY) {                                            \
      const unsigned gy = (unsigned)(N - r0 < kMaxGridY ? N - r0 : kMaxGridY);                 \
      hipLaunchKernelGGL((ce_bwd_vec<T, G, M>), dim3(gx, gy), block, 0, st, lp, ld, labels,    \
                         lse, dloss, dloss_stride, dloss_scale, gp, ld_grad, V, V / VE,        \
                         ignore_index, xf, smoothing, r0);                                     \
      ts_status s_ = ts_host::check_launch("ce_bwd_vec");                                      \
      if (s_ != TS_OK) return s_;                                                              \
    }                                                                                          \
    return TS_OK;                                                                              \
  }
  TS_CE_BWD(kPlain)
  TS_CE_BWD(kSmooth)
  TS_CE_BWD(kGeneral)
#undef TS_CE_BWD
  return ts_host::fail(TS_ERR_INVALID_ARGUMENT, "ce_bwd: unreachable");
}

ts_status check_ce(const void* logits, int64_t ld, ts_dtype dtype, const int64_t* labels,
                   int64_t N, int64_t V, float logit_scale, float softcap,
                   float label_smoothing) {
  using ts_host::fail;
  if (!ts_host::valid_dtype(dtype)) return fail(TS_ERR_UNSUPPORTED_DTYPE, "ce: bad dtype");
  if (N < 0 || V <= 0) return fail(TS_ERR_SHAPE, "ce: bad shape N=%lld V=%lld", (long long)N,
                                   (long long)V);
  if (N > 0x7fffffffLL) return fail(TS_ERR_SHAPE, "ce: too many rows (%lld)", (long long)N);
  if (ld < V) return fail(TS_ERR_SHAPE, "ce: row stride %lld < V %lld", (long long)ld,
                          (long long)V);
  if (N > 0 && (logits == nullptr || labels == nullptr))
    return fail(TS_ERR_INVALID_ARGUMENT, "ce: logits or labels is NULL");
  if (!(label_smoothing >= 0.f && label_smoothing < 1.f))
    return fail(TS_ERR_INVALID_ARGUMENT, "ce: label_smoothing must be in [0, 1)");
  if (!isfinite(logit_scale) || !isfinite(softcap) || softcap < 0.f)
    return fail(TS_ERR_INVALID_ARGUMENT, "ce: bad logit_scale/softcap");
  return TS_OK;
}

}  // namespace

extern "C" ts_status ts_ce_fwd(const void* logits, int64_t ld, ts_dtype dtype,
                               const int64_t* labels, int64_t N, int64_t V,
                               int64_t ignore_index, float logit_scale, float softcap,
                               float label_smoothing, float* loss, float* lse,
                               ts_stream_t stream) {
  ts_status s = check_ce(logits, ld, dtype, labels, N, V, logit_scale, softcap, label_smoothing);
  if (s != TS_OK) return s;
  if (N > 0 && (loss == nullptr || lse == nullptr))
    return ts_host::fail(TS_ERR_INVALID_ARGUMENT, "ce_fwd: loss or lse is NULL");
  if (N == 0) return TS_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const Xform xf = make_xform(logit_scale, softcap);
  const Mode mode = mode_of(logit_scale, softcap, label_smoothing);
  switch (dtype) {
    case TS_BF16:
      return fwd_typed<__bf16>(logits, ld, labels, N, V, ignore_index, xf, mode, label_smoothing,
                               loss, lse, st);
    case TS_F16:
      return fwd_typed<_Float16>(logits, ld, labels, N, V, ignore_index, xf, mode, label_smoothing,
                                 loss, lse, st);
    case TS_F32:
      return fwd_typed<float>(logits, ld, labels, N, V, ignore_index, xf, mode, label_smoothing, loss,
                              lse, st);
  }
  return ts_host::fail(TS_ERR_UNSUPPORTED_DTYPE, "ce_fwd: bad dtype");
}

extern "C" ts_status ts_ce_bwd(const void* logits, int64_t ld, ts_dtype dtype,
                               const int64_t* labels, const float* lse, const float* dloss,
                               int64_t dloss_stride, float dloss_scale, void* grad,
                               int64_t ld_grad, ts_dtype grad_dtype, int64_t N, int64_t V,
                               int64_t ignore_index, float logit_scale, float softcap,
                               float label_smoothing, ts_stream_t stream) {
  using ts_host::fail;
  ts_status s = check_ce(logits, ld, dtype, labels, N, V, logit_scale, softcap, label_smoothing);
  if (s != TS_OK) return s;
  if (!ts_host::valid_dtype(grad_dtype))
    return fail(TS_ERR_UNSUPPORTED_DTYPE, "ce_bwd: bad grad dtype");
  if (grad_dtype != dtype && grad_dtype != TS_F32)
    return fail(TS_ERR_UNSUPPORTED_DTYPE, "ce_bwd: grad dtype must equal logits dtype or be f32");
  if (N > 0 && (lse == nullptr || dloss == nullptr || grad == nullptr))
    return fail(TS_ERR_INVALID_ARGUMENT, "ce_bwd: lse, dloss or grad is NULL");
  if (ld_grad < V) return fail(TS_ERR_SHAPE, "ce_bwd: grad row stride < V");
  if (dloss_stride < 0) return fail(TS_ERR_SHAPE, "ce_bwd: negative dloss stride");
  if (grad == logits && (ld_grad != ld || grad_dtype != dtype))
    return fail(TS_ERR_INVALID_ARGUMENT, "ce_bwd: in-place grad needs the logits layout");
  if (N == 0) return TS_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const Xform xf = make_xform(logit_scale, softcap);
  const Mode mode = mode_of(logit_scale, softcap, label_smoothing);
#define TS_CE_BWD_T(T)                                                                         \
  return grad_dtype == TS_F32 && dtype != TS_F32                                               \
             ? bwd_typed<T, float>(logits, ld, labels, lse, dloss, dloss_stride, dloss_scale,  \
                                   grad, ld_grad, N, V, ignore_index, xf, mode, label_smoothing, st) \
             : bwd_typed<T, T>(logits, ld, labels, lse, dloss, dloss_stride, dloss_scale,      \
                               grad, ld_grad, N, V, ignore_index, xf, mode, label_smoothing, st);
  switch (dtype) {
    case TS_BF16: TS_CE_BWD_T(__bf16)
    case TS_F16: TS_CE_BWD_T(_Float16)
    case TS_F32: TS_CE_BWD_T(float)
  }
#undef TS_CE_BWD_T
  return fail(TS_ERR_UNSUPPORTED_DTYPE, "ce_bwd: bad dtype");
}

extern "C" ts_status ts_ce_fwd_bwd(const void* logits, int64_t ld, ts_dtype dtype,
                                   const int64_t* labels, int64_t N, int64_t V,
                                   int64_t ignore_index, float logit_scale, float softcap,
                                   float label_smoothing, const float* dloss,
                                   int64_t dloss_stride, float dloss_scale, float* loss,
                                   float* lse, void* grad, int64_t ld_grad, ts_dtype grad_dtype,
                                   ts_stream_t stream) {
  using ts_host::fail;
  ts_status s = check_ce(logits, ld, dtype, labels, N, V, logit_scale, softcap, label_smoothing);
  if (s != TS_OK) return s;
  if (!ts_host::valid_dtype(grad_dtype))
    return fail(TS_ERR_UNSUPPORTED_DTYPE, "ce_fwd_bwd: bad grad dtype");
  if (grad_dtype != dtype && grad_dtype != TS_F32)
    return fail(TS_ERR_UNSUPPORTED_DTYPE,
                "ce_fwd_bwd: grad dtype must equal logits dtype or be f32");
  if (N > 0 && (loss == nullptr || lse == nullptr || dloss == nullptr || grad == nullptr))
    return fail(TS_ERR_INVALID_ARGUMENT, "ce_fwd_bwd: loss, lse, dloss or grad is NULL");
  if (ld_grad < V) return fail(TS_ERR_SHAPE, "ce_fwd_bwd: grad row stride < V");
  if (dloss_stride < 0) return fail(TS_ERR_SHAPE, "ce_fwd_bwd: negative dloss stride");
  if (grad == logits)
    return fail(TS_ERR_INVALID_ARGUMENT,
                "ce_fwd_bwd: grad must not alias the logits (use ts_ce_fwd + ts_ce_bwd)");
  if (N == 0) return TS_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const Xform xf = make_xform(logit_scale, softcap);
  const Mode mode = mode_of(logit_scale, softcap, label_smoothing);
  const FusedArgs a{logits, ld, labels, N, V, ignore_index, xf, mode, label_smoothing, dloss,
                    dloss_stride, dloss_scale, loss, lse, grad, ld_grad, st};
  const bool wide = grad_dtype == TS_F32 && dtype != TS_F32;
  bool done = false;
  switch (dtype) {
    case TS_BF16: done = fused_bf16(a, wide, &s); break;
    case TS_F16: done = fused_f16(a, wide, &s); break;
    case TS_F32: done = fused_f32(a, &s); break;
  }
  if (done) return s;
  // Rows too long for one workgroup's registers: the two-pass schedule, forward then
  // backward.
  s = ts_ce_fwd(logits, ld, dtype, labels, N, V, ignore_index, logit_scale, softcap,
                label_smoothing, loss, lse, stream);
  if (s != TS_OK) return s;
  return ts_ce_bwd(logits, ld, dtype, labels, lse, dloss, dloss_stride, dloss_scale, grad,
                   ld_grad, grad_dtype, N, V, ignore_index, logit_scale, softcap,
                   label_smoothing, stream);
}

namespace {
ts_status check_reduce(const char* who, const int64_t* labels, int64_t N, int32_t reduction) {
  using ts_host::fail;
  if (N < 0 || N > 0x7fffffffLL)
    return fail(TS_ERR_SHAPE, "%s: bad row count %lld", who, (long long)N);
  if (reduction < 0 || reduction > 2)
    return fail(TS_ERR_INVALID_ARGUMENT, "%s: reduction must be 0 (mean), 1 (sum) or 2 (batchmean)",
                who);
  if (reduction == 0 && N > 0 && labels == nullptr)
    return fail(TS_ERR_INVALID_ARGUMENT, "%s: labels is NULL", who);
  return TS_OK;
}
}  // namespace

extern "C" ts_status ts_ce_loss_weight(const int64_t* labels, int64_t N, int64_t ignore_index,
                                       int32_t reduction, const float* hint, float* weight,
                                       float* used, ts_stream_t stream) {
  const ts_status s = check_reduce("ce_loss_weight", labels, N, reduction);
  if (s != TS_OK) return s;
  if (weight == nullptr)
    return ts_host::fail(TS_ERR_INVALID_ARGUMENT, "ce_loss_weight: weight is NULL");
  const float fixed = reduction == 2 ? (float)(1.0 / (double)(N > 0 ? N : 1)) : 1.f;
  hipLaunchKernelGGL(ce_loss_weight, dim3(1), dim3(reduction == 0 ? kRedThreads : kWave), 0,
                     static_cast<hipStream_t>(stream), labels, N, ignore_index,
                     reduction == 0 ? 1 : 0, fixed, hint, weight, used);
  return ts_host::check_launch("ce_loss_weight");
}

extern "C" ts_status ts_ce_reduce_loss(const float* loss_rows, const int64_t* labels, int64_t N,
                                       int64_t ignore_index, int32_t reduction, float* loss,
                                       ts_stream_t stream) {
  const ts_status s = check_reduce("ce_reduce_loss", labels, N, reduction);
  if (s != TS_OK) return s;
  if ((N > 0 && loss_rows == nullptr) || loss == nullptr)
    return ts_host::fail(TS_ERR_INVALID_ARGUMENT, "ce_reduce_loss: loss_rows or loss is NULL");
  const float div = reduction == 2 && N > 0 ? (float)N : 1.f;
  hipLaunchKernelGGL(ce_reduce_loss, dim3(1), dim3(kRedThreads), 0,
                     static_cast<hipStream_t>(stream), loss_rows, labels, N, ignore_index,
                     reduction == 0 ? 1 : 0, div, loss);
  return ts_host::check_launch("ce_reduce_loss");
}
