// Device code shared by the cross-entropy kernels (cross_entropy.hip and the one-pass
// kernels of ce_fused_*.hip): logit transforms, gradients, the elements after a row's last
// whole vector, and the one-pass kernel with its launcher. The one-pass kernel has many
// instantiations (row shapes, modes, alignment), so each data type compiles in its own file.
#pragma once

#include <float.h>
#include <math.h>

#include "common.hpp"
#include "plan.hpp"

namespace ts_ce {

using namespace ts;

// What a kernel applies besides the softmax: nothing, label smoothing, or any of logit
// scaling, softcapping and smoothing (each tested at run time, uniformly).
enum Mode : int { kPlain = 0, kSmooth = 1, kGeneral = 2 };

// Logit scaling then softcapping, in the reference's order
// (kernels/triton_kernels.py:214-217): z = softcap * tanh(scale * x / softcap).
struct Xform {
  float scale;    // 1 when off
  float softcap;  // 0 = off
  float inv_cap, inv_cap_lo;  // 1 / softcap in two floats, both above 0 (cap_quot)
};
inline Xform make_xform(float logit_scale, float softcap) {
  Xform f{logit_scale != 0.f ? logit_scale : 1.f, softcap, 0.f, 0.f};
  if (softcap == 0.f) return f;
  const double inv = 1.0 / (double)softcap;
  if (inv > (double)FLT_MAX) {  // softcap below 2^-128
    f.inv_cap = FLT_MAX;
  } else {
    f.inv_cap = (float)inv;
    if ((double)f.inv_cap >= inv) f.inv_cap = nextafterf(f.inv_cap, 0.f);
    f.inv_cap_lo = (float)(inv - (double)f.inv_cap);
  }
  if (f.inv_cap_lo == 0.f) f.inv_cap_lo = FLT_TRUE_MIN;
  return f;
}
// z / softcap, rounded once. z times the rounded reciprocal alone carries that one's error in
// every element (at softcap 30 a relative 5.2e-8); the low part is above 0 so that infinite z
// meet no product of infinity and 0 or of two signs.
__device__ inline float cap_quot(float z, const Xform& f) {
  return __builtin_fmaf(z, f.inv_cap, z * f.inv_cap_lo);
}
inline Mode mode_of(float logit_scale, float softcap, float smoothing) {
  return logit_scale != 0.f || softcap != 0.f ? kGeneral : smoothing != 0.f ? kSmooth : kPlain;
}

// tanh in two ranges, as accurate as the device library's tanhf. Below kTanhSmall:
// x + x^3 P(x^2), P of degree 5 fitted over [0, 0.85] for least relative error, four times
// closer near 0 (2.7e-9 there, 1.3e-8 at the end, before rounding). From there on:
// 1 - 2 / (1 + exp(2|x|)) with v_exp_f32 and v_rcp_f32 (each within 1 ulp), the exponent
// shifted by kShift, which keeps its rounding small where 2 / (1 + e) still counts;
// kPower = 2^kShift (1 + 3e-8), whose excess makes up for the rounding of 2 log2 e. A vector
// whose values are all small in every lane of the wave skips the second form, which costs
// twice the first. tanhf made the softcapped kernels VALU-bound: at [4096, 32000] bf16,
// softcap 30, the forward took 98 us and now takes 62, the backward 129 and 98. Rms error of the
// softcapped logit in ulps, tanhf(x / c) against these and cap_quot, c = 30: 0.530 and 0.517 for
// |x / c| below 0.75, 0.464 and 0.460 from there to 1.5, 0.399 and 0.400 from there to 4.
constexpr float kTanhSmall = 0.85f;
__device__ inline float tanh_small(float x) {
  const float s = x * x;
  float p = 0.001508764f;
  p = __builtin_fmaf(p, s, -0.007290129f);
  p = __builtin_fmaf(p, s, 0.021238737f);
  p = __builtin_fmaf(p, s, -0.053839035f);
  p = __builtin_fmaf(p, s, 0.13332148f);
  p = __builtin_fmaf(p, s, -0.333333f);
  return __builtin_fmaf(p, s * x, x);
}
__device__ inline float tanh_large(float x) {
  constexpr float kShift = 2.974609375f, kPower = 7.8604364f;
  const float e = fast_exp2(__builtin_fmaf(fabsf(x), 2.f * kLog2e, -kShift));
  const float r = __builtin_amdgcn_rcpf(__builtin_fmaf(kPower, e, 1.f));
  return copysignf(__builtin_fmaf(-2.f, r, 1.f), x);
}
// |x| < kTanhSmall is false for NaN, and tanh_large(NaN) is NaN.
__device__ inline float tanh1(float x) {
  return fabsf(x) < kTanhSmall ? tanh_small(x) : tanh_large(x);
}

// t[i] = tanh of the VE values u[i] a lane holds.
template <int VE>
__device__ inline void tanh_vec(const float (&u)[VE], float (&t)[VE]) {
  float um = fabsf(u[0]);
#pragma unroll
  for (int i = 1; i < VE; ++i) um = fmaxf(um, fabsf(u[i]));
#pragma unroll
  for (int i = 0; i < VE; ++i) t[i] = tanh_small(u[i]);
  // fmaxf drops a NaN, whose tanh_small is NaN too
  if (__builtin_amdgcn_ballot_w64(um >= kTanhSmall) != 0) {
#pragma unroll
    for (int i = 0; i < VE; ++i) {
      const float l = tanh_large(u[i]);
      t[i] = fabsf(u[i]) < kTanhSmall ? t[i] : l;
    }
  }
}

// The transformed value of one logit.
template <int kMode>
__device__ inline float xform1(float x, const Xform& f) {
  if constexpr (kMode == kGeneral) {
    x *= f.scale;
    if (f.softcap != 0.f) x = f.softcap * tanh1(cap_quot(x, f));
  }
  return x;
}
// The same of a vector, in place.
template <int kMode, int VE>
__device__ inline void xform_vec(float (&z)[VE], const Xform& f) {
  if constexpr (kMode == kGeneral) {
#pragma unroll
    for (int i = 0; i < VE; ++i) z[i] *= f.scale;
    if (f.softcap != 0.f) {
      float u[VE], t[VE];
#pragma unroll
      for (int i = 0; i < VE; ++i) u[i] = cap_quot(z[i], f);
      tanh_vec<VE>(u, t);
#pragma unroll
      for (int i = 0; i < VE; ++i) z[i] = f.softcap * t[i];
    }
  }
}

// Per-row factors of the gradient: dl * (p - [label] (1 - a) - a / V) * dz/dx.
struct GradRow {
  float dl;    // upstream gradient of this row
  float lse2;  // lse * log2(e)
  float keep;  // 1 - a in fp32, what the label's element subtracts
  float av;    // a / V, what every other element subtracts
  float avl;   // a / V and what keep lacks of 1 - a, what the label's subtracts before keep
};
// The label's element is most of a smoothed row's gradient norm, so it takes the small terms
// first (one rounding near 1 - a, not two) and 1 - a in two floats.
__device__ inline void set_smoothing(GradRow& r, float a, int64_t V) {
  r.keep = 1.f - a;
  r.av = a / (float)V;
  r.avl = r.av + ((1.f - r.keep) - a);
}

// Gradient of one logit x.
template <int kMode>
__device__ inline float grad1(float x, bool is_label, const GradRow& r, const Xform& f) {
  float z = x, dz = 1.f;
  if constexpr (kMode == kGeneral) {
    z *= f.scale;
    dz = f.scale;
    if (f.softcap != 0.f) {
      const float t = tanh1(cap_quot(z, f));
      z = f.softcap * t;
      dz = (1.f - t * t) * f.scale;
    }
  }
  float g = fast_exp2(__builtin_fmaf(z, kLog2e, -r.lse2));
  if constexpr (kMode != kPlain) g -= is_label ? r.avl : r.av;
  if (is_label) g -= r.keep;
  if constexpr (kMode == kGeneral) g *= dz;
  return r.dl * g;
}

// Gradients of a vector of logits; `lab` is the label's position in it, if in [0, VE).
template <int kMode, int VE>
__device__ inline void grad_vec(const float (&x)[VE], float (&g)[VE], int64_t lab,
                                const GradRow& r, const Xform& f) {
  float z[VE], dz[VE];
#pragma unroll
  for (int i = 0; i < VE; ++i) z[i] = x[i];
  if constexpr (kMode == kGeneral) {
#pragma unroll
    for (int i = 0; i < VE; ++i) {
      z[i] *= f.scale;
      dz[i] = f.scale;
    }
    if (f.softcap != 0.f) {
      float u[VE], t[VE];
#pragma unroll
      for (int i = 0; i < VE; ++i) u[i] = cap_quot(z[i], f);
      tanh_vec<VE>(u, t);
#pragma unroll
      for (int i = 0; i < VE; ++i) {
        z[i] = f.softcap * t[i];
        dz[i] = (1.f - t[i] * t[i]) * f.scale;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < VE; ++i) {
    float p = fast_exp2(__builtin_fmaf(z[i], kLog2e, -r.lse2));
    if constexpr (kMode != kPlain) p -= i == lab ? r.avl : r.av;
    p = i == lab ? p - r.keep : p;
    if constexpr (kMode == kGeneral) p *= dz[i];
    g[i] = r.dl * p;
  }
}

// This lane's element after the row's last whole vector, or -1 (ts_plan::tail_col).
template <int VE>
__device__ inline int64_t tail_col(int64_t V) {
  return ts_plan::tail_col(V, (int)threadIdx.x, VE);
}

// Adds the value z to an online (max, sum of exp) pair; nothing for -inf.
__device__ inline void fold1(float z, float& m, float& s) {
  const float mn = __builtin_fmaxf(m, z);
  if (z != z) {
    s = z;  // NaN poisons the row
  } else if (mn != -INFINITY) {
    s = (s == 0.f ? 0.f : s * fast_exp2((m - mn) * kLog2e)) + fast_exp2((z - mn) * kLog2e);
    m = mn;
  }
}

// Loss of a row from its lse and (with smoothing) its sum of z; thread 0 only. The mix is
// formed in double: the fp32 rounding of 1 - a is the same in every row, so a mean over rows
// would keep it.
template <int kMode, typename T>
__device__ inline float row_loss(const T* xr, int64_t label, int64_t V, int64_t ignore_index,
                                 float l, float sz, float smoothing, const Xform& xf) {
  const int64_t col = ts_plan::label_col(label, V, ignore_index);  // not ignored here
  if (col < 0) return __builtin_nanf("");
  float out = l - xform1<kMode>(Elt<T>::load1(xr + col), xf);
  if (kMode != kPlain && smoothing != 0.f)
    out = (float)((1.0 - (double)smoothing) * (double)out +
                  (double)smoothing * (double)(l - sz / (float)V));
  return out;
}

// ---------------------------------------------------------------------------
// Forward + backward in one pass ("schedule B"): one row per workgroup, held in
// registers (kKv 16-byte vectors per thread; ts_plan::ce_fused_plan picks the shape).
// Each thread folds its vectors into a (max, sum of exp) pair as they arrive; one LDS
// exchange of the wave pairs gives the lse (a single barrier). The gradient is then
// written from the same registers: each valid row is read once and every row written
// once. Ignored rows are written as zeros without being read.
//
// Rows on 16-byte boundaries (kAligned) are addressed through buffer resources (base and
// range in SGPRs, one VGPR of offset per lane), which keeps the 64 data VGPRs of 16 vectors
// plus the working set inside the 128-VGPR budget of four waves per SIMD; other rows through
// element-aligned global accesses. Without label
// smoothing or logit transforms an element's gradient is
// exp2(z*log2e - (lse*log2e - log2|dl|)) with the sign of dl applied to the
// packed result, one FMA and one exp per element; the label element is
// corrected by the one lane that holds it.
// ---------------------------------------------------------------------------

// ln 2 times what the bias mb = m log2 e, rounded, lacks of m log2 e: a sum of
// exp2(z log2 e - mb) is exp(lack) times the sum of exp(z - m). It reaches half an ulp of m.
__device__ inline float bias_lack(float m, float mb) {
  return kLn2 * __builtin_fmaf(m, kLog2e, -mb);
}

constexpr float kLn2Lo = (float)(0.6931471805599453 - (double)kLn2);

// m + log(s), rounded about once: the exponent of s joins m, what that sum loses the logarithm
// of the rest. m + logf(s) adds logf's rounding, half an ulp of up to 7 in an lse of 8 or more.
__device__ inline float log_sum(float m, float s) {
  const int e = __builtin_amdgcn_frexp_expf(s) - 1;
  const float k = (float)e;
  const float y = __builtin_amdgcn_logf(__builtin_amdgcn_ldexpf(s, -e));  // v_log_f32: log2
  const float a = __builtin_fmaf(k, kLn2, m);
  const float b = __builtin_fmaf(k, kLn2, m - a);
  const float l = a + __builtin_fmaf(y, kLn2, __builtin_fmaf(k, kLn2Lo, b));
  return s == 0.f ? -INFINITY : l;  // nothing but -inf in the row
}

// Moves a lane's (m, sum of exp2(z log2 e - mb)) pair, mb = m log2 e rounded, to a reference
// next to its sum: s about in [1, 2) and m + log(s) the lane's log-sum, without the roundings
// of mb and of log2 e and, where m lay far below the lane's values, without two large terms
// that cancel. What the new m lost in its rounding goes into s. Rms error of lse at [512, 1001]
// fp32 N(0, 1), with log_sum: 0.31 ulp, 0.31 to 0.34 with the first 256 columns 10 to 40 lower;
// without either 0.64 and 1.1 to 2.6.
__device__ inline void settle(float& m, float mb, float& s) {
  // ln 2 in 15 bits, so that a whole multiple of it is exact, and so is its sum with a larger m of
  // the other sign; the rest of ln 2 goes into s, with the rounding of log2 e over the distance
  // that the terms lie above m
  constexpr float kHi = 0.693145751953125f;
  constexpr double kL = 0.6931471805599453, kE = 1.4426950408889634;
  constexpr float kRest = (float)(kL - (double)kHi + kL * kL * (kE - (double)kLog2e));
  const int e = __builtin_amdgcn_frexp_expf(s) - 1;
  const float k = (float)e;
  const float d = k * kHi;
  const float m1 = m + d;
  const float lost = __builtin_fmaf(k, kRest, ((m - m1) + d) - bias_lack(m, mb));
  const float s1 = __builtin_amdgcn_ldexpf(s, -e);
  s = __builtin_fmaf(s1, lost, s1);
  m = m1;
}

// Row lse (and, with smoothing, the row sum of z) from every thread's online
// (max, sum of exp) pair. lds holds 3 * kNW floats. One barrier: the
// caller must not write lds again without another barrier in between.
template <int kMode, int kNW>
__device__ inline float fused_lse(float m, float s, float& sz, float* lds) {
  const float wm = wave_max(m);
  const float ws = wave_sum(s == 0.f ? 0.f : s * fast_exp2((m - wm) * kLog2e));
  const int wid = threadIdx.x / kWave;
  if constexpr (kMode != kPlain) sz = wave_sum(sz);
  if ((threadIdx.x & (kWave - 1)) == 0) {
    lds[wid] = wm;
    lds[kNW + wid] = ws;
    if constexpr (kMode != kPlain) lds[2 * kNW + wid] = sz;
  }
  __syncthreads();
  float gm = lds[0];
#pragma unroll
  for (int i = 1; i < kNW; ++i) gm = fmaxf(gm, lds[i]);
  float gs = 0.f, gz = 0.f;
#pragma unroll
  for (int i = 0; i < kNW; ++i) {
    const float si = lds[kNW + i];
    gs += si == 0.f ? 0.f : si * fast_exp2((lds[i] - gm) * kLog2e);
    if constexpr (kMode != kPlain) gz += lds[2 * kNW + i];
  }
  if constexpr (kMode != kPlain) sz = gz;
  return log_sum(gm, gs);
}

template <typename G>
constexpr uint32_t sign_bits() {
  return sizeof(G) == 4 ? 0x80000000u : 0x80008000u;
}

// Waves per SIMD the register budget must allow: four at 16 vectors per thread (128 VGPRs),
// six at 8 and eight at 4.
constexpr int fused_waves(int kv) { return kv >= 16 ? 4 : kv >= 8 ? 6 : 8; }

// Largest sum of exp(z - m) that a lane's reference m serves for (see ce_fused_vec): one whose
// terms' exponents, up to 60, are still rounded finely beside lse. A lower bound costs more
// second folds (2^20: [4096, 50257] bf16 of N(0, 6), softcap 30, 297 us instead of 253) and
// gains nothing: with settle, lse errors do not depend on where the first vectors lie.
constexpr float kLaneSumMax = 0x1p60f;

template <typename T, typename G, int kMode, int kThr, int kKv, bool kAligned>
__global__ __launch_bounds__(kThr) __attribute__((amdgpu_waves_per_eu(fused_waves(kKv))))
void ce_fused_vec(
    const T* __restrict__ logits, int64_t ld, const int64_t* __restrict__ labels, int64_t V,
    int nvec, int64_t ignore_index, Xform xf, float smoothing, const float* __restrict__ dloss,
    int64_t dloss_stride, float dloss_scale, float* __restrict__ loss, float* __restrict__ lse_out,
    G* __restrict__ grad, int64_t ld_grad) {
  constexpr int VE = Elt<T>::kVec;
  constexpr int kNW = kThr / kWave;
  constexpr int kGradBytes = VE * (int)sizeof(G);  // grad bytes per logits vector
  __shared__ float lds[3 * kNW];
  const int64_t row = blockIdx.x;
  const int64_t label = labels[row];
  const T* xr = logits + row * ld;
  G* gr = grad + row * ld_grad;
  // Byte offset of this thread's k-th vector, past the last one an offset no row resource
  // covers (ts_plan::vec_boffset: the hardware drops such stores, loads read 0).
  auto voff = [&](int k, int vec_bytes) {
    return ts_plan::vec_boffset(ts_plan::chunk_vec(0, k, threadIdx.x, kThr, kKv), nvec,
                                vec_bytes);
  };
  const Rsrc go = buf_rsrc(gr, (uint32_t)nvec * kGradBytes);
  // Stores the gradients of this thread's k-th vector (p1 the second half of fp32 ones).
  auto store = [&](int k, const u32x4& p0, const u32x4& p1) {
    if constexpr (kAligned) {
      const int off = voff(k, kGradBytes);
      buf_st16_stream(p0, go, off);
      if constexpr (kGradBytes == 32) buf_st16_stream(p1, go, off + 16);
    } else {
      const int v = (int)threadIdx.x + k * kThr;
      // Not streaming stores: the waves' stores meet inside cache lines here, which L2 should
      // merge (407 us against 416 us for the [8191, 50257] bf16 loss and gradient).
      if (v < nvec) {
        st16_any(gr + v * VE, p0);
        if constexpr (kGradBytes == 32) st16_any(gr + v * VE + 4, p1);
      }
    }
  };
  const bool has_tail = V % VE != 0;  // uniform: rows of whole vectors skip its code
  if (label == ignore_index) {
    const u32x4 zero = {0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < kKv; ++k) store(k, zero, zero);
    if (has_tail) {
      const int64_t ec = tail_col<VE>(V);
      if (ec >= 0) Elt<G>::store1(gr + ec, 0.f);
    }
    if (threadIdx.x == 0) {
      loss[row] = 0.f;
      lse_out[row] = 0.f;
    }
    return;
  }
  // The tail element goes out first: a wait for it later leaves the vectors' loads in
  // flight. Lanes without one read outside the resource, which touches no memory.
  const int64_t ec = has_tail ? tail_col<VE>(V) : -1;
  T xe;
  {
    const Rsrc xt = buf_rsrc(xr, (uint32_t)V * (uint32_t)sizeof(T));
    const int off = ec >= 0 ? (int)(ec * (int64_t)sizeof(T)) : kBufOob;
    if constexpr (sizeof(T) == 4) {
      const uint32_t q = __builtin_amdgcn_raw_buffer_load_b32(xt, off, 0, kBufNt);
      xe = __builtin_bit_cast(T, q);
    } else {
      const uint16_t q = __builtin_amdgcn_raw_buffer_load_b16(xt, off, 0, kBufNt);
      xe = __builtin_bit_cast(T, q);
    }
  }
  u32x4 buf[kKv];
  if constexpr (kAligned) {
    const Rsrc xi = buf_rsrc(xr, (uint32_t)nvec * 16u);
#pragma unroll
    for (int k = 0; k < kKv; ++k) buf[k] = buf_ld16_stream(xi, voff(k, 16));
  } else if (nvec > 0) {
    // unconditional, so that the loads have no branches between them: a lane past the
    // row's last vector loads its first one, which nothing uses
#pragma unroll
    for (int k = 0; k < kKv; ++k) {
      const int v = (int)threadIdx.x + k * kThr;
      buf[k] = ld16_any_stream(xr + (v < nvec ? v * VE : 0));
    }
  }
  // Each lane sums exp(z - m) over its vectors against one reference m, the
  // largest value of its first vector (0 if that vector is all -inf): per
  // element one unpack, one FMA, one exp and one add, with no running max or
  // rescale. Such a sum serves while it lies in [0.5, kLaneSumMax]: terms that
  // underflowed are then below its resolution, and settle brings it next to its
  // reference, so that no fold over the lanes overflows with it or loses it.
  // Other lanes (values far above m, a NaN, a reference past kRefMax, an all -inf
  // first vector that left a sum of values far below 0) fold their vectors again
  // from the registers with an exact online max and rescale: s in [1, VE * kKv]
  // against the largest value. Lanes without vectors keep m = -inf, s = 0.
  float m = -INFINITY, mb = 0.f, s = 0.f, sz = 0.f;
  auto sum_exp = [&](const float (&z)[VE], float bias) {
    float cs = fast_exp2(__builtin_fmaf(z[0], kLog2e, -bias));
#pragma unroll
    for (int i = 1; i < VE; ++i) cs += fast_exp2(__builtin_fmaf(z[i], kLog2e, -bias));
    return cs;
  };
  auto values = [&](const u32x4& q, float (&z)[VE]) {
    Elt<T>::unpack(q, z);
    xform_vec<kMode, VE>(z, xf);
  };
  auto vmax = [&](const float (&z)[VE]) {
    float cm = z[0];
#pragma unroll
    for (int i = 1; i < VE; ++i) cm = __builtin_fmaxf(cm, z[i]);
    return cm;
  };
  auto fold = [&](const u32x4& q, bool first) {
    float z[VE];
    values(q, z);
    if constexpr (kMode != kPlain) {
#pragma unroll
      for (int i = 0; i < VE; ++i) sz += z[i];
    }
    if (first) {
      const float cm = vmax(z);
      m = cm == -INFINITY ? 0.f : cm;
      mb = m * kLog2e;
    }
    s += sum_exp(z, mb);
  };
#pragma unroll
  for (int k = 0; k < kKv; ++k) {
    // Vectors every thread holds take a uniform branch; only the row's last
    // partial sweep tests each lane.
    // With transforms one copy of their code serves both.
    if (kMode != kGeneral && (k + 1) * kThr <= nvec) fold(buf[k], k == 0);
    else if ((int)threadIdx.x + k * kThr < nvec) fold(buf[k], k == 0);
  }
  if (s >= 0.5f && s <= kLaneSumMax && fabsf(m) < kRefMax) {
    settle(m, mb, s);
  } else if ((int)threadIdx.x < nvec) {
    m = -INFINITY;
    s = 0.f;
#pragma unroll
    for (int k = 0; k < kKv; ++k) {
      if ((int)threadIdx.x + k * kThr < nvec) {
        float z[VE];
        values(buf[k], z);
        // __builtin_fmaxf drops NaN, whose term makes s NaN, and s stays so
        const float mn = __builtin_fmaxf(m, vmax(z));
        s = (s == 0.f ? 0.f : s * fast_exp2((m - mn) * kLog2e)) + sum_exp_far<VE>(z, mn);
        m = mn;
      }
    }
  }
  if (has_tail && ec >= 0) {
    const float ze = xform1<kMode>(Elt<T>::load1(&xe), xf);
    fold1(ze, m, s);
    if constexpr (kMode != kPlain) sz += ze;
  }
  const float l = fused_lse<kMode, kNW>(m, s, sz, lds);
  // The gradient pass re-unpacks the stored vectors; this keeps the compiler
  // from carrying the first pass's unpacked floats (twice the registers).
#pragma unroll
  for (int k = 0; k < kKv; ++k) asm volatile("" : "+v"(buf[k]));
  if (threadIdx.x == 0) {
    loss[row] = row_loss<kMode>(xr, label, V, ignore_index, l, sz, smoothing, xf);
    lse_out[row] = l;
  }
  // One upstream gradient per row, moved to a scalar register: its sign below
  // is then a wave-uniform mask (one XOR per packed dword, no per-lane select).
  GradRow r;
  r.dl = __builtin_bit_cast(
      float, __builtin_amdgcn_readfirstlane(
                 __builtin_bit_cast(int, dloss[row * dloss_stride] * dloss_scale)));
  r.lse2 = l * kLog2e;
  set_smoothing(r, smoothing, V);
  if (has_tail && ec >= 0) Elt<G>::store1(gr + ec, grad1<kMode>(Elt<T>::load1(&xe), ec == label, r, xf));
  // The position of the label is uniform over the workgroup: its correction is a
  // uniform branch, and only the lane holding the label runs it.
  const bool lab_in = label >= 0 && label < (int64_t)nvec * VE;
  const int64_t la = lab_in ? label : 0;
  const int klab = lab_in ? (int)(la / VE / kThr) : -1;
  const int tlab = lab_in ? (int)(la / VE % kThr) : -1;
  const int elab = lab_in ? (int)(la % VE) : 0;
  const float adl = fabsf(r.dl);
  const float l2d = r.lse2 - __builtin_amdgcn_logf(adl);  // v_log_f32 is log2
  const uint32_t smask = kMode == kPlain && (__builtin_bit_cast(uint32_t, r.dl) >> 31) != 0
                             ? sign_bits<G>() : 0u;
#pragma unroll
  for (int k = 0; k < kKv; ++k) {
    float z[VE], g[VE];
    Elt<T>::unpack(buf[k], z);
    if constexpr (kMode == kPlain) {
#pragma unroll
      for (int i = 0; i < VE; ++i) g[i] = fast_exp2(__builtin_fmaf(z[i], kLog2e, -l2d));
      if (k == klab && (int)threadIdx.x == tlab) {
#pragma unroll
        for (int i = 0; i < VE; ++i)
          if (i == elab) g[i] = adl * (fast_exp2(__builtin_fmaf(z[i], kLog2e, -r.lse2)) - 1.f);
      }
    } else {
      grad_vec<kMode, VE>(z, g, -1, r, xf);
      if (k == klab && (int)threadIdx.x == tlab) {
        float zl = z[0];
#pragma unroll
        for (int i = 1; i < VE; ++i) zl = i == elab ? z[i] : zl;
        const float gl = grad1<kMode>(zl, true, r, xf);
#pragma unroll
        for (int i = 0; i < VE; ++i) g[i] = i == elab ? gl : g[i];
      }
    }
    if constexpr (kGradBytes == 32) {
      u32x4 p0 = Elt<float>::pack(g), p1 = Elt<float>::pack(g + 4);
      p0 ^= smask;
      p1 ^= smask;
      store(k, p0, p1);
    } else {
      u32x4 p = Elt<G>::pack(g);
      p ^= smask;
      store(k, p, p);
    }
  }
}

// The one-pass kernel for logits of one type (T) with gradients of that type, or fp32 ones of
// 16-bit logits (`wide`); false, and nothing launched, when no workgroup holds the row.
struct FusedArgs {
  const void* logits;
  int64_t ld;
  const int64_t* labels;
  int64_t N, V, ignore_index;
  Xform xf;
  Mode mode;
  float smoothing;
  const float* dloss;
  int64_t dloss_stride;
  float dloss_scale;
  float* loss;
  float* lse;
  void* grad;
  int64_t ld_grad;
  hipStream_t st;
};
bool fused_bf16(const FusedArgs& a, bool wide, ts_status* status);
bool fused_f16(const FusedArgs& a, bool wide, ts_status* status);
bool fused_f32(const FusedArgs& a, ts_status* status);

// Schedule B when the row fits the registers of one workgroup; returns false (nothing
// launched) otherwise.
template <typename T, typename G>
bool launch_fused(const FusedArgs& a, ts_status* status) {
  constexpr int VE = sizeof(T) == 4 ? 4 : 8;
  const ts_plan::CeFusedPlan plan = ts_plan::ce_fused_plan(a.V / VE, sizeof(G) != sizeof(T));
  if (plan.threads == 0 || a.N > INT32_MAX) return false;
  const bool aligned = ts_host::aligned16(a.logits) && ts_host::aligned16(a.grad) &&
                       a.ld * (int64_t)sizeof(T) % 16 == 0 &&
                       a.ld_grad * (int64_t)sizeof(G) % 16 == 0;
#define TS_CE_FUSED(M, THR, KV, AL)                                                            \
  if (a.mode == M && plan.threads == THR && plan.kv == KV && aligned == AL) {                  \
    hipLaunchKernelGGL((ce_fused_vec<T, G, M, THR, KV, AL>), dim3((unsigned)a.N), dim3(THR),   \
                       0, a.st, static_cast<const T*>(a.logits), a.ld, a.labels, a.V,          \
                       (int)(a.V / VE), a.ignore_index, a.xf, a.smoothing, a.dloss,            \
                       a.dloss_stride, a.dloss_scale, a.loss, a.lse, static_cast<G*>(a.grad),  \
                       a.ld_grad);                                                             \
    *status = ts_host::check_launch("ce_fused_vec");                                           \
    return true;                                                                               \
  }
#define TS_CE_FUSED_MODES(THR, KV)         \
  TS_CE_FUSED(kPlain, THR, KV, true)       \
  TS_CE_FUSED(kSmooth, THR, KV, true)      \
  TS_CE_FUSED(kGeneral, THR, KV, true)     \
  TS_CE_FUSED(kPlain, THR, KV, false)      \
  TS_CE_FUSED(kSmooth, THR, KV, false)     \
  TS_CE_FUSED(kGeneral, THR, KV, false)
  if constexpr (sizeof(G) == sizeof(T)) {
    TS_CE_FUSED_MODES(64, 4)
    TS_CE_FUSED_MODES(256, 4)
    TS_CE_FUSED_MODES(256, 8)
    TS_CE_FUSED_MODES(256, 16)
    TS_CE_FUSED_MODES(512, 16)
  }
  TS_CE_FUSED_MODES(1024, 16)
#undef TS_CE_FUSED_MODES
#undef TS_CE_FUSED
  *status = ts_host::fail(TS_ERR_INVALID_ARGUMENT, "ce_fwd_bwd: no kernel for %d x %d",
                          plan.threads, plan.kv);
  return true;
}

}  // namespace ts_ce
