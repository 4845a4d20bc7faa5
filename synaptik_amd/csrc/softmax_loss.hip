// Row softmax / log-softmax / log-sum-exp and the MSE loss.
//
// Softmax follows CpuSoftmaxReferenceKernel.evaluateFloat (reference/CpuSoftmaxReferenceKernel.java:104-146):
//   maximum by Math.max; a +inf maximum maps +inf entries to NaN and the rest to 0 (softmax) or
//   -inf (log-softmax); a row containing -inf (and no NaN) is evaluated unshifted (shift 0);
//   addends are (float)exp((double)(x - shift)); the result is (float)exp(shift)/sum or
//   shift - (float)log(sum). The GPU forms the addends with exp_f32 (fexp.h), which returns
//   that binary32 value or one of its neighbours (at most 1 ulp away; 0.46% of arguments), in its
//   range, and as the reference does elsewhere.
//   The reference sums addends with Kahan compensation in binary32 (error within about
//   2 ulp of the exact sum). All forms here round a sum once that is within a few binary32 ulps of
//   the exact one (reduction-order difference):
//   softmax_fwd_regs    16-byte aligned rows of 509 to 4096: one workgroup of 256 a row, held in
//                       registers. Each lane's 4V addends are summed pairwise in binary32 (positive
//                       addends: error within log2(4V) ulp), the lanes in binary64 through a fixed
//                       tree; the row is multiplied by a once-rounded reciprocal of the sum.
//   softmax_fwd_rows    other rows up to 32764 (aligned ones up to 32768): one wave or one workgroup
//                       of 256 to 1024 a row, held in registers, summed in binary64; the quotient is
//                       the correctly rounded one.
//   softmax_fwd_stream  wider rows: one workgroup of 256 a row, read three times, summed in binary64
//                       and divided.
#include "common.h"
#include "fexp.h"
#include "kernels.h"
#include "rowvec.h"
#include <algorithm>
#include <type_traits>

namespace shk {
namespace {

constexpr int SM_NT = 256;

__device__ __forceinline__ int block_or(int v, int* lds) {
  v = wave_or(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
  __syncthreads();
  int r = 0;
#pragma unroll
  for (int i = 0; i < SM_NT / 64; ++i) r |= lds[i];
  return r;
}

struct RowStats {
  float shift;
  float sum;
  bool pos_inf;
};

__device__ __forceinline__ float shifted_exp(float x, float shift) {
  return exp_f32(x - shift);
}

__device__ __forceinline__ int holds_nan(const float4& v) {
  return __builtin_isunordered(v.x, v.y) | __builtin_isunordered(v.z, v.w);
}

// V float4 per thread in registers (C <= V * 4 * SM_NT, C % 4 == 0).
//
// The row statistics use the hardware max / min (v_max_f32 / v_min_f32, which skip NaN and need
// not order signed zeros) and restore Math.max semantics where they differ: a NaN anywhere, which a
// flag of its own tells, makes the maximum and with it the shift NaN, and a zero maximum is +0 when
// any element is +0 (a branch taken only by rows whose maximum is a zero). A row holds -inf exactly
// when its minimum is -inf.
template <int V>
__global__ void __launch_bounds__(SM_NT) softmax_fwd_regs(const float* __restrict__ x,
                                                          float* __restrict__ y, float* lse,
                                                          int64_t C, int log_softmax) {
  __shared__ double dl[SM_NT / 64];
  __shared__ float fmx[SM_NT / 64], fmn[SM_NT / 64];
  __shared__ int il[SM_NT / 64], il2[SM_NT / 64];  // (NaN, +0)
  const int64_t r = blockIdx.x;
  const float4* xr = reinterpret_cast<const float4*>(x + r * C);
  float4* yr = reinterpret_cast<float4*>(y + r * C);
  const int C4 = (int)(C / 4);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  float4 v[V];
  float m = -INFINITY, mn = INFINITY;
  int nan = 0;
#pragma unroll
  for (int i = 0; i < V; ++i) {
    const int c = threadIdx.x + i * SM_NT;
    if (c < C4) {
      v[i] = ld_stream(&xr[c]);
      nan |= holds_nan(v[i]);
      m = fmaxf(m, fmaxf(fmaxf(v[i].x, v[i].y), fmaxf(v[i].z, v[i].w)));
      mn = fminf(mn, fminf(fminf(v[i].x, v[i].y), fminf(v[i].z, v[i].w)));
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    m = fmaxf(m, __shfl_xor(m, o, 64));
    mn = fminf(mn, __shfl_xor(mn, o, 64));
  }
  nan = __any(nan);
  if (lane == 0) { fmx[w] = m; fmn[w] = mn; il[w] = nan; }
  __syncthreads();
  m = fmx[0];
  mn = fmn[0];
  nan = il[0];
#pragma unroll
  for (int i = 1; i < SM_NT / 64; ++i) {
    m = fmaxf(m, fmx[i]);
    mn = fminf(mn, fmn[i]);
    nan |= il[i];
  }
  if (nan) {
    m = NAN;
  } else if (m == 0.0f) {  // block-uniform, rare
    int pos_zero = 0;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const int c = threadIdx.x + i * SM_NT;
      if (c < C4)
        pos_zero |= (__float_as_uint(v[i].x) == 0u) | (__float_as_uint(v[i].y) == 0u) |
                    (__float_as_uint(v[i].z) == 0u) | (__float_as_uint(v[i].w) == 0u);
    }
    pos_zero = __any(pos_zero);
    if (lane == 0) il2[w] = pos_zero;
    __syncthreads();
    pos_zero = 0;
#pragma unroll
    for (int i = 0; i < SM_NT / 64; ++i) pos_zero |= il2[i];
    m = pos_zero ? 0.0f : -0.0f;
  }
  if (m == INFINITY) {
    const float other = log_softmax ? -INFINITY : 0.0f;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const int c = threadIdx.x + i * SM_NT;
      if (c < C4) {
        float4 o;
        o.x = v[i].x == INFINITY ? NAN : other;
        o.y = v[i].y == INFINITY ? NAN : other;
        o.z = v[i].z == INFINITY ? NAN : other;
        o.w = v[i].w == INFINITY ? NAN : other;
        yr[c] = o;
      }
    }
    if (lse != nullptr && threadIdx.x == 0) lse[r] = INFINITY;
    return;
  }
  const bool neg_inf = mn == -INFINITY;
  const float shift = (neg_inf && m == m) ? 0.0f : m;
  // One exponential per element: softmax keeps the rounded addends in registers and scales
  // them by the sum; log-softmax only needs the sum and recomputes x - shift.
  //
  // Every argument x - shift of a row shifted by its finite maximum lies in
  // [fl(min - max), 0] (subtraction rounds monotonically), so when fl(min - max) >= -87 the
  // whole row takes the binary32 path of the exponential without a per-element range test.
  const bool in_range = shift == m && is_finite(m) && mn - m >= -87.0f;  // block-uniform
  float4 e[V];
  float part[V];
  if (in_range) {
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const int c = threadIdx.x + i * SM_NT;
      if (c < C4) {
        e[i].x = exp_f32_in_range(v[i].x - shift);
        e[i].y = exp_f32_in_range(v[i].y - shift);
        e[i].z = exp_f32_in_range(v[i].z - shift);
        e[i].w = exp_f32_in_range(v[i].w - shift);
        part[i] = (e[i].x + e[i].y) + (e[i].z + e[i].w);
      } else {
        part[i] = 0.0f;
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const int c = threadIdx.x + i * SM_NT;
      if (c < C4) {
        e[i].x = shifted_exp(v[i].x, shift);
        e[i].y = shifted_exp(v[i].y, shift);
        e[i].z = shifted_exp(v[i].z, shift);
        e[i].w = shifted_exp(v[i].w, shift);
        part[i] = (e[i].x + e[i].y) + (e[i].z + e[i].w);
      } else {
        part[i] = 0.0f;
      }
    }
  }
  // Pairwise over the lane's float4 groups (every part is >= 0 or NaN, so zero padding is exact).
#pragma unroll
  for (int h = 1; h < V; h <<= 1)
#pragma unroll
    for (int i = 0; i + h < V; i += 2 * h) part[i] += part[i + h];
  const float sum = (float)block_sum<SM_NT>((double)part[0], dl);
  // Every lane needs the binary64 logarithm of the sum only for log-softmax; softmax needs it
  // only for the LSE output, which lane 0 forms below.
  const float logsum = log_softmax ? (float)log((double)sum) : 0.0f;
  // Softmax scales by the reciprocal of the sum (one division per row; at most one extra
  // rounding per element against the reference's quotient). A sum whose reciprocal would leave
  // the normal range, or a non-finite one, keeps the per-element division.
  const bool recip = sum >= 0x1p-126f && sum <= 0x1p126f;
  const float inv = 1.0f / sum;
#pragma unroll
  for (int i = 0; i < V; ++i) {
    const int c = threadIdx.x + i * SM_NT;
    if (c < C4) {
      float4 o;
      if (log_softmax) {
        o.x = (v[i].x - shift) - logsum;
        o.y = (v[i].y - shift) - logsum;
        o.z = (v[i].z - shift) - logsum;
        o.w = (v[i].w - shift) - logsum;
      } else if (recip) {
        o.x = e[i].x * inv;
        o.y = e[i].y * inv;
        o.z = e[i].z * inv;
        o.w = e[i].w * inv;
      } else {
        o.x = e[i].x / sum;
        o.y = e[i].y / sum;
        o.z = e[i].z / sum;
        o.w = e[i].w / sum;
      }
      st_stream(&yr[c], o);
    }
  }
  if (lse != nullptr) {
    if (neg_inf && is_finite(m)) {
      // LOG_SUM_EXP keeps the maximum as its shift even when the row holds -inf
      // (CpuLogSumExpEmitter.java:4-9); only the softmax values use the unshifted form.
      double s2 = 0.0;
#pragma unroll
      for (int i = 0; i < V; ++i) {
        const int c = threadIdx.x + i * SM_NT;
        if (c < C4)
          s2 += ((double)shifted_exp(v[i].x, m) + (double)shifted_exp(v[i].y, m)) +
                ((double)shifted_exp(v[i].z, m) + (double)shifted_exp(v[i].w, m));
      }
      const float sum2 = (float)block_sum<SM_NT>(s2, dl);
      if (threadIdx.x == 0) lse[r] = m + (float)log((double)sum2);
    } else if (threadIdx.x == 0) {
      lse[r] = shift + (log_softmax ? logsum : (float)log((double)sum));
    }
  }
}

// Rows of any start and width in aligned 16-byte groups (rowvec.h), V of them a thread, held in
// registers from the load to the store; sums in binary64 throughout. One wave a row (NT = 64, four
// rows a workgroup, no barrier) up to 2044 columns, where a workgroup a row spends its time in
// barriers and a single load's latency; one workgroup of NT threads above. Aligned rows
// of 509 to 4096 keep softmax_fwd_regs (20000x1000 97 us against 119). Three passes of 4-byte loads
// before; us on MI355X, softmax with its gradient: 20000x1001 174 -> 103, 10000x4095 320 -> 204,
// 2000x32000 545 -> 302, 65536x100 152 -> 84; log-softmax 92 -> 55, 157 -> 93, 271 -> 131, 122 -> 62.
template <int NT>
struct RowTeam {  // the threads that share a row: a wave, or a workgroup
  static constexpr int WAVES = NT == 64 ? 4 : NT / 64;
  static constexpr int THREADS = NT == 64 ? 256 : NT;
  struct Shared {
    double d[WAVES];
    float a[WAVES], b[WAVES];
    int i[WAVES];
  };
  __device__ static __forceinline__ int lane() { return NT == 64 ? threadIdx.x & 63 : threadIdx.x; }
  __device__ static __forceinline__ double sum(double v, Shared& s) {
    v = wave_sum(v);
    if constexpr (NT == 64) return v;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) s.d[threadIdx.x >> 6] = v;
    __syncthreads();
    double r = 0.0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) r += s.d[w];
    return r;
  }
  // The row's hardware maximum and minimum (both skip NaN) and whether it holds a NaN.
  __device__ static __forceinline__ void extremes(float& mx, float& mn, int& nan, Shared& s) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      mx = fmaxf(mx, __shfl_xor(mx, o, 64));
      mn = fminf(mn, __shfl_xor(mn, o, 64));
    }
    nan = __any(nan);
    if constexpr (NT == 64) return;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) {
      s.a[threadIdx.x >> 6] = mx;
      s.b[threadIdx.x >> 6] = mn;
      s.i[threadIdx.x >> 6] = nan;
    }
    __syncthreads();
    mx = s.a[0];
    mn = s.b[0];
    nan = s.i[0];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) {
      mx = fmaxf(mx, s.a[w]);
      mn = fminf(mn, s.b[w]);
      nan |= s.i[w];
    }
  }
  __device__ static __forceinline__ int any(int a, Shared& s) {
    a = __any(a);
    if constexpr (NT == 64) return a;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) s.i[threadIdx.x >> 6] = a;
    __syncthreads();
    a = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) a |= s.i[w];
    return a;
  }
};

// exp(x - shift) with the binary64 evaluation of fexp64.h outside exp_f32's fast range.
__device__ __forceinline__ float row_exp(float x, float shift) {
  const float t = x - shift;
  return t >= -87.0f && t <= 88.0f ? exp_f32_in_range(t) : exp_rn(t);
}

template <int NT, int V, bool LOG>
__global__ void __launch_bounds__(RowTeam<NT>::THREADS)
__attribute__((amdgpu_waves_per_eu(NT == 1024 ? 4 : V <= 2 ? 5 : V == 4 ? 4 : 3)))
softmax_fwd_rows(const float* x, float* y, float* lse, int64_t R, int64_t C) {
  using Team = RowTeam<NT>;
  __shared__ typename Team::Shared sh;
  const int tid = Team::lane();
  const int64_t first_row = NT == 64 ? (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6) : blockIdx.x;
  const int64_t row_step = NT == 64 ? (int64_t)gridDim.x * 4 : gridDim.x;
  for (int64_t r = first_row; r < R; r += row_step) {
    const float* xr = x + r * C;
    float* yr = y + r * C;
    const RowGroups view(xr, (int)C);
    float4 v[V];
    float m = -INFINITY, mn = INFINITY;
    int nan = 0;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const int q = tid + i * NT;
      v[i] = q < view.groups ? view.load(xr, q, -INFINITY)
                             : make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
    }
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const int q = tid + i * NT;
      m = fmaxf(m, fmaxf(fmaxf(v[i].x, v[i].y), fmaxf(v[i].z, v[i].w)));
      nan |= holds_nan(v[i]);
      if (q < view.groups) {
        if (view.whole(q)) {
          mn = fminf(mn, fminf(fminf(v[i].x, v[i].y), fminf(v[i].z, v[i].w)));
        } else {
          if (view.holds(q, 0)) mn = fminf(mn, v[i].x);
          if (view.holds(q, 1)) mn = fminf(mn, v[i].y);
          if (view.holds(q, 2)) mn = fminf(mn, v[i].z);
          if (view.holds(q, 3)) mn = fminf(mn, v[i].w);
        }
      }
    }
    Team::extremes(m, mn, nan, sh);
    // Math.max: a NaN is the maximum, and so the shift. (It also keeps the row off the binary32
    // exponential, whose result is a finite number for most NaN patterns.)
    if (nan) {
      m = NAN;
    } else if (m == 0.0f) {  // uniform for the row, rare (see softmax_fwd_regs)
      int pos_zero = 0;
#pragma unroll
      for (int i = 0; i < V; ++i)
        pos_zero |= (__float_as_uint(v[i].x) == 0u) | (__float_as_uint(v[i].y) == 0u) |
                    (__float_as_uint(v[i].z) == 0u) | (__float_as_uint(v[i].w) == 0u);
      m = Team::any(pos_zero, sh) ? 0.0f : -0.0f;
    }
    if (m == INFINITY) {
      const float other = LOG ? -INFINITY : 0.0f;
#pragma unroll
      for (int i = 0; i < V; ++i) {
        const int q = tid + i * NT;
        if (q < view.groups)
          view.store(yr, q, make_float4(v[i].x == INFINITY ? NAN : other, v[i].y == INFINITY ? NAN : other,
                                        v[i].z == INFINITY ? NAN : other, v[i].w == INFINITY ? NAN : other));
      }
      if (lse != nullptr && tid == 0) lse[r] = INFINITY;
      continue;
    }
    const bool neg_inf = mn == -INFINITY;
    const float shift = (neg_inf && m == m) ? 0.0f : m;
    // every argument in the binary32 exponential's range (see softmax_fwd_regs)
    const bool in_range = shift == m && is_finite(m) && mn - m >= -87.0f;
    // (padding, -inf, lies outside that range: its terms are left out)
    auto add = [&](int i, const float4& e, double& s) {
      const int q = tid + i * NT;
      if (q >= view.groups) return;
      if (view.whole(q)) {
        s += ((double)e.x + (double)e.y) + ((double)e.z + (double)e.w);
      } else {
        if (view.holds(q, 0)) s += (double)e.x;
        if (view.holds(q, 1)) s += (double)e.y;
        if (view.holds(q, 2)) s += (double)e.z;
        if (view.holds(q, 3)) s += (double)e.w;
      }
    };
    float row_lse = 0.0f;
    const bool lse_apart = lse != nullptr && neg_inf && is_finite(m);
    if (lse_apart) {
      // LOG_SUM_EXP keeps the maximum as its shift even when the row holds -inf
      // (CpuLogSumExpEmitter.java:4-9); only the softmax values use the unshifted form.
      double s2 = 0.0;
#pragma unroll
      for (int i = 0; i < V; ++i) {
        add(i, make_float4(row_exp(v[i].x, m), row_exp(v[i].y, m), row_exp(v[i].z, m),
                           row_exp(v[i].w, m)), s2);
        __builtin_amdgcn_sched_barrier(0);
      }
      row_lse = m + (float)log((double)(float)Team::sum(s2, sh));
    }
    double s = 0.0;
    auto exps = [&](auto fast) {
#pragma unroll
      for (int i = 0; i < V; ++i) {
        float4 e;
        if constexpr (decltype(fast)::value) {
          e = make_float4(exp_f32_in_range(v[i].x - shift), exp_f32_in_range(v[i].y - shift),
                          exp_f32_in_range(v[i].z - shift), exp_f32_in_range(v[i].w - shift));
        } else {
          e = make_float4(row_exp(v[i].x, shift), row_exp(v[i].y, shift),
                          row_exp(v[i].z, shift), row_exp(v[i].w, shift));
        }
        add(i, e, s);
        if constexpr (!LOG) v[i] = e;
        __builtin_amdgcn_sched_barrier(0);  // four at a time keep the registers down
      }
    };
    if (in_range) exps(std::true_type{});
    else exps(std::false_type{});
    const float sum = (float)Team::sum(s, sh);
    // softmax needs the logarithm of the sum for the LSE output alone
    const float logsum = LOG || tid == 0 ? (float)log((double)sum) : 0.0f;
    // In range the sum lies in [1, C], and a reciprocal with a residual correction gives the
    // correctly rounded quotient; otherwise divide.
    const float inv = 1.0f / sum;
    auto quotient = [&](float e) {
      if (!in_range) return e / sum;
      const float q0 = e * inv;
      return fmaf(fmaf(-q0, sum, e), inv, q0);
    };
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const int q = tid + i * NT;
      if (q < view.groups) {
        float4 o;
        if constexpr (LOG)
          o = make_float4((v[i].x - shift) - logsum, (v[i].y - shift) - logsum,
                          (v[i].z - shift) - logsum, (v[i].w - shift) - logsum);
        else
          o = make_float4(quotient(v[i].x), quotient(v[i].y), quotient(v[i].z), quotient(v[i].w));
        view.store(yr, q, o);
      }
    }
    if (lse != nullptr && tid == 0) lse[r] = lse_apart ? row_lse : shift + logsum;
  }
}

// dX = y (.) (g - s) [+ k_r * y], s = sum(g (.) y), over the same row forms.
template <int NT, int V>
__global__ void __launch_bounds__(RowTeam<NT>::THREADS)
softmax_bwd_rows(const float* y, const float* g, float* dx, int64_t R, int64_t C,
                 const float* rowscale, float rsc) {
  using Team = RowTeam<NT>;
  __shared__ typename Team::Shared sh;
  const int tid = Team::lane();
  const int64_t first_row = NT == 64 ? (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6) : blockIdx.x;
  const int64_t row_step = NT == 64 ? (int64_t)gridDim.x * 4 : gridDim.x;
  const bool scaled = rowscale != nullptr || rsc != 0.0f;
  for (int64_t r = first_row; r < R; r += row_step) {
    const float* yr = y + r * C;
    const float* gr = g + r * C;
    const RowGroups view(yr, (int)C);
    float4 yv[V], gv[V];
    const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const int q = tid + i * NT;
      yv[i] = q < view.groups ? view.load(yr, q, 0.0f) : zero;
      gv[i] = q < view.groups ? view.load(gr, q, 0.0f) : zero;
    }
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      s += (double)(gv[i].x * yv[i].x);
      s += (double)(gv[i].y * yv[i].y);
      s += (double)(gv[i].z * yv[i].z);
      s += (double)(gv[i].w * yv[i].w);
    }
    const float sf = (float)Team::sum(s, sh);
    const float k = rowscale != nullptr ? rowscale[r] : rsc;
    auto out = [&](float a, float b) {
      const float o = a * (b - sf);
      return scaled ? o + k * a : o;
    };
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const int q = tid + i * NT;
      if (q < view.groups)
        view.store(dx + r * C, q, make_float4(out(yv[i].x, gv[i].x), out(yv[i].y, gv[i].y),
                                              out(yv[i].z, gv[i].z), out(yv[i].w, gv[i].w)));
    }
  }
}

// Any width: three streaming passes over the row.
__global__ void __launch_bounds__(SM_NT) softmax_fwd_stream(const float* __restrict__ x,
                                                            float* __restrict__ y, float* lse,
                                                            int64_t C, int log_softmax) {
  __shared__ double dl[SM_NT / 64];
  __shared__ float fl[SM_NT / 64];
  __shared__ int il[SM_NT / 64];
  const int64_t r = blockIdx.x;
  const float* xr = x + r * C;
  float* yr = y + r * C;
  float m = -INFINITY;
  int neg_inf = 0;
  for (int64_t c = threadIdx.x; c < C; c += SM_NT) {
    const float t = xr[c];
    m = java_max(m, t);
    neg_inf |= t == -INFINITY;
  }
  m = block_max<SM_NT>(m, fl);
  neg_inf = block_or(neg_inf, il);
  if (m == INFINITY) {
    const float other = log_softmax ? -INFINITY : 0.0f;
    for (int64_t c = threadIdx.x; c < C; c += SM_NT) yr[c] = xr[c] == INFINITY ? NAN : other;
    if (lse != nullptr && threadIdx.x == 0) lse[r] = INFINITY;
    return;
  }
  const float shift = (neg_inf && m == m) ? 0.0f : m;
  double s = 0.0;
  for (int64_t c = threadIdx.x; c < C; c += SM_NT) s += (double)shifted_exp(xr[c], shift);
  const float sum = (float)block_sum<SM_NT>(s, dl);
  const float logsum = (float)log((double)sum);
  for (int64_t c = threadIdx.x; c < C; c += SM_NT)
    yr[c] = log_softmax ? (xr[c] - shift) - logsum : shifted_exp(xr[c], shift) / sum;
  if (lse != nullptr) {
    float l = C == 0 ? -INFINITY : shift + logsum;
    if (neg_inf && is_finite(m)) {  // LOG_SUM_EXP shifts by the maximum (see above)
      double s2 = 0.0;
      for (int64_t c = threadIdx.x; c < C; c += SM_NT) s2 += (double)shifted_exp(xr[c], m);
      l = m + (float)log((double)(float)block_sum<SM_NT>(s2, dl));
    }
    if (threadIdx.x == 0) lse[r] = l;
  }
}

// dX = y (.) (g - s) [+ k_r * y], s = sum(g (.) y)  (ReductionGradientRules.java:84-90).
template <int V>
__global__ void __launch_bounds__(SM_NT) softmax_bwd_regs(const float* __restrict__ y,
                                                          const float* __restrict__ g,
                                                          float* __restrict__ dx, int64_t C,
                                                          const float* rowscale, float rsc) {
  __shared__ double dl[SM_NT / 64];
  const int64_t r = blockIdx.x;
  const float4* yr = reinterpret_cast<const float4*>(y + r * C);
  const float4* gr = reinterpret_cast<const float4*>(g + r * C);
  float4* dr = reinterpret_cast<float4*>(dx + r * C);
  const int C4 = (int)(C / 4);
  float4 yv[V], gv[V];
  double s = 0.0;
#pragma unroll
  for (int i = 0; i < V; ++i) {
    const int c = threadIdx.x + i * SM_NT;
    if (c < C4) {
      yv[i] = ld_stream(&yr[c]);
      gv[i] = ld_stream(&gr[c]);
      s += (double)(gv[i].x * yv[i].x);
      s += (double)(gv[i].y * yv[i].y);
      s += (double)(gv[i].z * yv[i].z);
      s += (double)(gv[i].w * yv[i].w);
    }
  }
  const float sf = (float)block_sum<SM_NT>(s, dl);
  const bool scaled = rowscale != nullptr || rsc != 0.0f;
  const float k = rowscale != nullptr ? rowscale[r] : rsc;
#pragma unroll
  for (int i = 0; i < V; ++i) {
    const int c = threadIdx.x + i * SM_NT;
    if (c < C4) {
      float4 o;
      o.x = yv[i].x * (gv[i].x - sf);
      o.y = yv[i].y * (gv[i].y - sf);
      o.z = yv[i].z * (gv[i].z - sf);
      o.w = yv[i].w * (gv[i].w - sf);
      if (scaled) {
        o.x = o.x + k * yv[i].x;
        o.y = o.y + k * yv[i].y;
        o.z = o.z + k * yv[i].z;
        o.w = o.w + k * yv[i].w;
      }
      st_stream(&dr[c], o);
    }
  }
}

__global__ void __launch_bounds__(SM_NT) softmax_bwd_stream(const float* __restrict__ y,
                                                            const float* __restrict__ g,
                                                            float* __restrict__ dx, int64_t C,
                                                            const float* rowscale, float rsc) {
  __shared__ double dl[SM_NT / 64];
  const int64_t r = blockIdx.x;
  const float* yr = y + r * C;
  const float* gr = g + r * C;
  float* dr = dx + r * C;
  double s = 0.0;
  for (int64_t c = threadIdx.x; c < C; c += SM_NT) s += (double)(gr[c] * yr[c]);
  const float sf = (float)block_sum<SM_NT>(s, dl);
  const bool scaled = rowscale != nullptr || rsc != 0.0f;
  const float k = rowscale != nullptr ? rowscale[r] : rsc;
  for (int64_t c = threadIdx.x; c < C; c += SM_NT) {
    float o = yr[c] * (gr[c] - sf);
    if (scaled) o = o + k * yr[c];
    dr[c] = o;
  }
}

// LOG_SUM_EXP gradient g_r * exp(x - lse_r) (ReductionGradientRules.java:213-224). Bound by the
// binary64 exponentials, each one dependent chain. Small inputs, whose waves hide it, and rows of
// less than four take an element a thread; LSE_BWD_GROUPED elements and more a group of four,
// evaluated side by side with one division for the group's row and, as rows follow each other
// without a gap, one 16-byte access wherever a row ends. [11537, 1756] 51 us a
// step on MI355X with an element a thread, 33 so; [300000, 6] 7.3 and 5.6; [1000, 400], below the
// line, 3.5 with an element a thread.
constexpr int64_t LSE_BWD_GROUPED = 1 << 19;
__global__ void __launch_bounds__(256) lse_bwd_kernel(const float* __restrict__ x,
                                                      const float* __restrict__ lse, const float* g,
                                                      float gconst, float* __restrict__ dx, int64_t R,
                                                      int64_t C) {
  const int64_t n = R * C;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = i / C;
    const float gr = g != nullptr ? g[r] : gconst;
    dx[i] = gr * exp_rn(x[i] - lse[r]);
  }
}
__global__ void __launch_bounds__(256) lse_bwd_groups(const float* __restrict__ x,
                                                      const float* __restrict__ lse, const float* g,
                                                      float gconst, float* __restrict__ dx, int64_t R,
                                                      int64_t C) {
  const int64_t n = R * C;
  for (int64_t i = 4 * ((int64_t)blockIdx.x * blockDim.x + threadIdx.x); i < n;
       i += 4 * (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = n <= 0xffffffffll ? (int64_t)((uint32_t)i / (uint32_t)C) : i / C;
    const int64_t next = min<int64_t>(r + 1, R - 1), left = C - (i - r * C);  // left: in row r
    const float l0 = lse[r], l1 = lse[next];
    const float g0 = g != nullptr ? g[r] : gconst, g1 = g != nullptr ? g[next] : gconst;
    auto element = [&](float v, int q) { return (q < left ? g0 : g1) * exp_rn(v - (q < left ? l0 : l1)); };
    if (i + 3 < n) {
      const float4u v = __builtin_nontemporal_load(reinterpret_cast<const float4u*>(x + i));
      const float4u o = {element(v[0], 0), element(v[1], 1), element(v[2], 2), element(v[3], 3)};
      __builtin_nontemporal_store(o, reinterpret_cast<float4u*>(dx + i));
    } else {
      for (int q = 0; i + q < n; ++q) dx[i + q] = element(x[i + q], q);
    }
  }
}

// ---- MSE (CpuLossReferenceKernel.java:67-87, LossGradientRules.java:77-97) ----
constexpr int MSE_BLOCKS = 1024;
// MEAN finalization divides the binary32 sum by the exact count before one final rounding.
__device__ __forceinline__ float mse_loss(double s, int64_t n, int reduction_sum) {
  const float sf = (float)s;
  return reduction_sum ? sf : (float)((double)sf / (double)n);
}
// Pass 1: block b's binary64 partial sum of squared differences (and the gradient). A launch of
// one block finishes the loss itself: its partial is the whole sum, which pass 2 would only
// return unchanged. Up to MSE_ONE_BLOCK elements one block of 1024 threads does so: its few loads a
// thread cost less than the second launch (8192 elements 9.2 us in two launches on MI355X, 4.4 in
// one).
constexpr int64_t MSE_ONE_BLOCK = 16384;
template <int NT>
__global__ void __launch_bounds__(NT) mse_pass1(const float* __restrict__ p,
                                                 const float* __restrict__ t,
                                                 float* __restrict__ grad, int64_t n, float gn,
                                                 double* part, float* loss, int reduction_sum) {
  __shared__ double dl[NT / 64];
  double s = 0.0;
  const int64_t stride = (int64_t)gridDim.x * NT;
  const bool vec = ((reinterpret_cast<uintptr_t>(p) | reinterpret_cast<uintptr_t>(t) |
                     reinterpret_cast<uintptr_t>(grad)) & 15u) == 0;
  int64_t head = 0;
  if (vec) {
    // four elements per thread and iteration, streaming 16-byte accesses
    const int64_t n4 = n / 4;
    for (int64_t q = (int64_t)blockIdx.x * NT + threadIdx.x; q < n4; q += stride) {
      const float4 pv = ld_stream(reinterpret_cast<const float4*>(p) + q);
      const float4 tv = ld_stream(reinterpret_cast<const float4*>(t) + q);
      const float d0 = pv.x - tv.x, d1 = pv.y - tv.y, d2 = pv.z - tv.z, d3 = pv.w - tv.w;
      const float q0 = d0 * d0, q1 = d1 * d1, q2 = d2 * d2, q3 = d3 * d3;
      s += ((double)q0 + (double)q1) + ((double)q2 + (double)q3);
      if (grad != nullptr) {
        const float t0 = d0 * 2.0f, t1 = d1 * 2.0f, t2 = d2 * 2.0f, t3 = d3 * 2.0f;
        st_stream(reinterpret_cast<float4*>(grad) + q, make_float4(t0 * gn, t1 * gn, t2 * gn, t3 * gn));
      }
    }
    head = n4 * 4;
  }
  for (int64_t i = head + (int64_t)blockIdx.x * NT + threadIdx.x; i < n; i += stride) {
    const float d = p[i] - t[i];
    const float sq = d * d;
    s += (double)sq;
    if (grad != nullptr) {
      const float twice = d * 2.0f;
      grad[i] = twice * gn;
    }
  }
  s = block_sum<NT>(s, dl);
  if (threadIdx.x == 0) {
    if (gridDim.x == 1) loss[0] = mse_loss(s, n, reduction_sum);
    else part[blockIdx.x] = s;
  }
}
__global__ void __launch_bounds__(256) mse_pass2(const double* part, int P, int64_t n,
                                                 int reduction_sum, float* loss) {
  __shared__ double dl[4];
  double s = 0.0;
  for (int i = threadIdx.x; i < P; i += 256) s += part[i];
  s = block_sum<256>(s, dl);
  if (threadIdx.x == 0) loss[0] = mse_loss(s, n, reduction_sum);
}

}  // namespace

namespace {
// One wave a row: four rows a workgroup; otherwise a row a workgroup (looping beyond 2^20).
template <int NT>
dim3 row_grid(int64_t R) {
  return dim3((unsigned)std::min<int64_t>(NT == 64 ? (R + 3) / 4 : R, 1 << 20));
}
template <int NT, int V>
void launch_fwd_rows(const float* x, float* y, float* lse, int64_t R, int64_t C, int log_softmax,
                     hipStream_t s) {
  const dim3 g = row_grid<NT>(R), b(RowTeam<NT>::THREADS);
  if (log_softmax) hipLaunchKernelGGL((softmax_fwd_rows<NT, V, true>), g, b, 0, s, x, y, lse, R, C);
  else hipLaunchKernelGGL((softmax_fwd_rows<NT, V, false>), g, b, 0, s, x, y, lse, R, C);
}
template <int NT, int V>
void launch_bwd_rows(const float* y, const float* g, float* dx, int64_t R, int64_t C,
                     const float* rowscale, float rsc, hipStream_t s) {
  hipLaunchKernelGGL((softmax_bwd_rows<NT, V>), row_grid<NT>(R), dim3(RowTeam<NT>::THREADS), 0, s,
                     y, g, dx, R, C, rowscale, rsc);
}
// Floats that V groups of each of NT threads hold, whatever the row's start.
constexpr int64_t row_capacity(int nt, int v) { return 4ll * nt * v - 4; }
// Backward, rows of at most 2044: up to this many rows a workgroup of 256 a row ends sooner than a
// wave a row, which holds ragged groups: the streamed form or, for aligned rows, the one in
// registers. us a step on MI355X, streamed and a wave a row: [16, 275] 3.2 and 4.3, [2048, 275] 4.6
// and 4.8, [2048, 907] 6.4 and 7.2, [512, 130] 3.2 and 3.4, [1024, 1691] 6.5 and 6.9; [4096, 275]
// 6.3 and 5.3, [1544, 130] 3.8 and 3.7, [1544, 1691] 8.6 and 8.5. Aligned rows of at most 252 take a
// wave each from the first ([16, 200] 3.1 and 2.9).
inline int64_t sb_few_rows(int64_t C) {
  return C > row_capacity(64, 1) && C <= row_capacity(64, 4) ? 2048 : 1024;
}
}  // namespace

hipError_t launch_softmax_fwd(const float* x, float* y, float* lse, int64_t R, int64_t C,
                              int log_softmax, hipStream_t s) {
  if (R <= 0) return hipSuccess;
  const bool vec = C % 4 == 0 && ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y)) & 15u) == 0;
  auto rows = [&](auto nt, auto v) {
    launch_fwd_rows<decltype(nt)::value, decltype(v)::value>(x, y, lse, R, C, log_softmax, s);
  };
  auto regs = [&](auto v) {
    hipLaunchKernelGGL(softmax_fwd_regs<decltype(v)::value>, dim3((unsigned)R), dim3(SM_NT), 0, s, x, y, lse, C, log_softmax);
  };
  using std::integral_constant;
  if (C <= 0)
    hipLaunchKernelGGL(softmax_fwd_stream, dim3((unsigned)R), dim3(SM_NT), 0, s, x, y, lse, C, log_softmax);
  else if (C <= row_capacity(64, 1)) rows(integral_constant<int, 64>{}, integral_constant<int, 1>{});
  else if (C <= row_capacity(64, 2)) rows(integral_constant<int, 64>{}, integral_constant<int, 2>{});
  else if (vec && C <= 1024) regs(integral_constant<int, 1>{});
  else if (vec && C <= 2048) regs(integral_constant<int, 2>{});
  else if (vec && C <= 4096) regs(integral_constant<int, 4>{});
  else if (C <= row_capacity(64, 4)) rows(integral_constant<int, 64>{}, integral_constant<int, 4>{});
  else if (C <= row_capacity(64, 8)) rows(integral_constant<int, 64>{}, integral_constant<int, 8>{});
  else if (C <= row_capacity(256, 4)) rows(integral_constant<int, 256>{}, integral_constant<int, 4>{});
  else if (C <= row_capacity(256, 8)) rows(integral_constant<int, 256>{}, integral_constant<int, 8>{});
  else if (C <= row_capacity(512, 8)) rows(integral_constant<int, 512>{}, integral_constant<int, 8>{});
  else if (C <= row_capacity(1024, 8) + (vec ? 4 : 0)) rows(integral_constant<int, 1024>{}, integral_constant<int, 8>{});
  else
    hipLaunchKernelGGL(softmax_fwd_stream, dim3((unsigned)R), dim3(SM_NT), 0, s, x, y, lse, C, log_softmax);
  return hipGetLastError();
}

hipError_t launch_softmax_bwd(const float* y, const float* g, float* dx, int64_t R, int64_t C,
                              const float* rowscale, float rowscale_const, hipStream_t s) {
  if (R <= 0) return hipSuccess;
  const bool vec = C % 4 == 0 &&
      ((reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(g) |
        reinterpret_cast<uintptr_t>(dx)) & 15u) == 0;
  auto rows = [&](auto nt, auto v) {
    launch_bwd_rows<decltype(nt)::value, decltype(v)::value>(y, g, dx, R, C, rowscale, rowscale_const, s);
  };
  auto regs = [&](auto v) {
    hipLaunchKernelGGL(softmax_bwd_regs<decltype(v)::value>, dim3((unsigned)R), dim3(SM_NT), 0, s, y, g, dx, C, rowscale,
                       rowscale_const);
  };
  using std::integral_constant;
  if (C <= 0) return hipSuccess;
  if ((!vec && C <= row_capacity(64, 8) && R <= sb_few_rows(C)) || C > row_capacity(1024, 8) + (vec ? 4 : 0))
    hipLaunchKernelGGL(softmax_bwd_stream, dim3((unsigned)R), dim3(SM_NT), 0, s, y, g, dx, C, rowscale,
                       rowscale_const);
  else if (C <= row_capacity(64, 1)) rows(integral_constant<int, 64>{}, integral_constant<int, 1>{});
  else if (vec && C <= 508 && R <= 1024) regs(integral_constant<int, 1>{});
  else if (C <= row_capacity(64, 2)) rows(integral_constant<int, 64>{}, integral_constant<int, 2>{});
  else if (vec && C <= 1024) regs(integral_constant<int, 1>{});
  else if (vec && C <= 2048) regs(integral_constant<int, 2>{});
  else if (vec && C <= 4096) regs(integral_constant<int, 4>{});
  else if (C <= row_capacity(64, 4)) rows(integral_constant<int, 64>{}, integral_constant<int, 4>{});
  else if (C <= row_capacity(64, 8)) rows(integral_constant<int, 64>{}, integral_constant<int, 8>{});
  else if (C <= row_capacity(256, 4)) rows(integral_constant<int, 256>{}, integral_constant<int, 4>{});
  else if (C <= row_capacity(256, 8)) rows(integral_constant<int, 256>{}, integral_constant<int, 8>{});
  else if (C <= row_capacity(512, 8)) rows(integral_constant<int, 512>{}, integral_constant<int, 8>{});
  else rows(integral_constant<int, 1024>{}, integral_constant<int, 8>{});
  return hipGetLastError();
}

hipError_t launch_lse_bwd(const float* x, const float* lse, const float* g, float gconst,
                          float* dx, int64_t R, int64_t C, hipStream_t s) {
  const int64_t n = R * C;
  if (n <= 0) return hipSuccess;
  const int each = n >= LSE_BWD_GROUPED && C >= 4 ? 4 : 1;
  const dim3 blocks((unsigned)std::min<int64_t>(65536, (n + 256 * each - 1) / (256 * each))), nt(256);
  if (each == 4) hipLaunchKernelGGL(lse_bwd_groups, blocks, nt, 0, s, x, lse, g, gconst, dx, R, C);
  else hipLaunchKernelGGL(lse_bwd_kernel, blocks, nt, 0, s, x, lse, g, gconst, dx, R, C);
  return hipGetLastError();
}

int64_t mse_partial_doubles(int64_t) { return MSE_BLOCKS; }
hipError_t launch_mse(const float* p, const float* t, float* loss, float* grad, int64_t n,
                      float g, int reduction_sum, double* partial, hipStream_t s) {
  const unsigned blocks = n <= MSE_ONE_BLOCK ? 1u : (unsigned)std::min<int64_t>(MSE_BLOCKS, (n + 1023) / 1024);
  // restore(g): MEAN divides g by the count (an exact binary32 sum of ones); SUM expands g.
  const float gn = reduction_sum ? g : g / (float)n;
  if (n > 1024 && blocks == 1)
    hipLaunchKernelGGL(mse_pass1<1024>, dim3(1), dim3(1024), 0, s, p, t, grad, n, gn, partial, loss,
                       reduction_sum);
  else
    hipLaunchKernelGGL(mse_pass1<256>, dim3(blocks), dim3(256), 0, s, p, t, grad, n, gn, partial, loss,
                       reduction_sum);
  if (blocks > 1)
    hipLaunchKernelGGL(mse_pass2, dim3(1), dim3(256), 0, s, (const double*)partial, (int)blocks,
                       n, reduction_sum, loss);
  return hipGetLastError();
}

}  // namespace shk
