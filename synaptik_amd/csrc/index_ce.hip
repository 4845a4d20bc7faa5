// Index categorical cross-entropy with logits: the loss (MEAN over the samples that are not
// ignored) and its gradient (CpuLossReferenceKernel.java:196-218,261-288;
// LossGradientRules.java:172-240).
//
// Bound: the logits are read once and the gradient is written once. One pass does both: a row is
// held in registers from its load to its gradient, so its exponentials (binary64, rounded once:
// exp_rn) are evaluated once and serve the loss, the sum and the probabilities. The former two
// kernels read each row five times, formed three exponentials for each element and gave every
// row to a single wave: [4096, 32003] with an ignore index took 1514 us on MI355X, now 245
// us (its 1.05 GB take 159 us at the card's copy rate).
//
// The gradient is scaled by the sample count, which is R without an ignore index. With one, up to
// a stated number of rows each workgroup counts the targets itself; beyond that a launch before
// counts them once. The mean counts the rows that it adds.
//
// Row statistics: the loss shifts by the maximum by '>' and the gradient by Math.max. A NaN
// logit makes both NaN through the sum, and the sign of a zero maximum changes no exponential,
// so the hardware maximum serves both; so does a row whose maximum is infinite (NaN throughout).
#include "common.h"
#include "kernels.h"
#include "rowvec.h"
#include <algorithm>

namespace shk {
namespace {

struct CeArgs {
  const float* logits;
  const void* target;
  float* grad;      // null: the loss alone
  float* row_loss;  // [R]: lse - logit of the target, CE_NO_LOSS where ignored or out of bounds
  const uint4* count;  // sample counts of four parts of the rows; null: counted here (with an
                       // ignore index) or R
  uint32_t* status;
  int64_t R, C, ignore;
  int has_ignore;
  float g;
};

// The loss of a row that is not a sample: -0, which the sum does not see and no sample's loss is (a
// difference is -0 only for -0 minus +0, and lse = m + log(sum), log(sum) >= +0, is never -0).
constexpr float CE_NO_LOSS = -0.0f;
__device__ __forceinline__ int ce_no_loss(float v) { return __float_as_uint(v) == 0x80000000u; }

template <typename T, int NT>
__device__ __forceinline__ double ce_count(const CeArgs& a, int64_t first, int64_t end, double* dl) {
  const T* target = static_cast<const T*>(a.target);
  int64_t n = 0;
#pragma unroll 8
  for (int64_t i = first + threadIdx.x; i < end; i += NT) {
    const int64_t t = (int64_t)target[i];
    n += !(a.has_ignore && t == a.ignore) && t >= 0 && t < a.C;
  }
  return block_sum<NT>((double)n, dl);  // whole numbers: exact in any order
}

// The gradient's divisor, for a block of NT threads.
template <typename T, int NT>
__device__ __forceinline__ float ce_divisor(const CeArgs& a, double* dl) {
  if (!a.has_ignore) return (float)(double)a.R;
  if (a.count == nullptr) return (float)ce_count<T, NT>(a, 0, a.R, dl);
  const uint4 n = *a.count;
  return (float)(((double)n.x + (double)n.y) + ((double)n.z + (double)n.w));
}

// e / s for the correctly rounded reciprocal `inv` of s >= 1: the quotient's residual corrects it
// to the correctly rounded quotient (Markstein's division) wherever that is a normal number.
__device__ __forceinline__ float ce_quotient(float e, float s, float inv) {
  const float q = e * inv;
  return fmaf(fmaf(-q, s, e), inv, q);
}

// ---- rows of at most 64 V classes: one wave a row, lane l holds classes l, l + 64, ... ----
// (a narrow row leaves most of a workgroup idle; a wave needs no barrier between its three steps)
template <typename T, int V>
__global__ void __launch_bounds__(256) ce_rows_wave(CeArgs a) {
  __shared__ double dl[4];
  const int lane = threadIdx.x & 63;
  const float divisor = a.grad != nullptr ? ce_divisor<T, 256>(a, dl) : 1.0f;
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= a.R) return;
  const int C = (int)a.C;
  const float* row = a.logits + r * a.C;
  const int64_t t = (int64_t)static_cast<const T*>(a.target)[r];
  const bool ignored = a.has_ignore && t == a.ignore;
  const bool in_range = t >= 0 && t < a.C;
  if (ignored) {  // (uniform for the wave) no loss, a zero gradient: the row is not read
    if (lane == 0) a.row_loss[r] = CE_NO_LOSS;
    if (a.grad != nullptr) {
#pragma unroll
      for (int i = 0; i < V; ++i)
        if (lane + 64 * i < C) a.grad[r * a.C + lane + 64 * i] = 0.0f;
    }
    return;
  }
  const int safe = (int)(t < 0 ? 0 : (t >= a.C ? a.C - 1 : t));
  const float xt = row[safe];
  float v[V];
  float m = -INFINITY;
#pragma unroll
  for (int i = 0; i < V; ++i) {
    const int c = lane + 64 * i;
    v[i] = c < C ? row[c] : -INFINITY;
    m = fmaxf(m, v[i]);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  double s = 0.0;
#pragma unroll
  for (int i = 0; i < V; ++i) {
    if (lane + 64 * i < C) {
      v[i] = exp_rn(v[i] - m);
      s += (double)v[i];
    }
  }
  const float sum = (float)wave_sum(s);
  if (lane == 0) {
    if (!in_range) atomicOr(a.status, (uint32_t)DEV_INDEX_OUT_OF_BOUNDS);
    const float lse = m + (float)log((double)sum);
    a.row_loss[r] = in_range ? lse - xt : CE_NO_LOSS;
  }
  if (a.grad == nullptr) return;
  float* gr = a.grad + r * a.C;
  const float scale = a.g / divisor;
#pragma unroll
  for (int i = 0; i < V; ++i) {
    const int c = lane + 64 * i;
    if (c < C) gr[c] = (v[i] / sum - (c == safe ? 1.0f : 0.0f)) * scale;
  }
}

// ---- wider rows: one workgroup of NT threads a row, V 16-byte groups a thread ----
// Four waves on each SIMD in every form: two workgroups of 512 on a CU, one of 1024.
template <typename T, int NT, int V>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4)))
ce_rows_block(CeArgs a) {
  __shared__ double dl[NT / 64];
  __shared__ float fm[NT / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const float scale = a.grad != nullptr ? a.g / ce_divisor<T, NT>(a, dl) : 0.0f;
  const int C = (int)a.C;
  for (int64_t r = blockIdx.x; r < a.R; r += gridDim.x) {
    const float* row = a.logits + r * a.C;
    const int64_t t = (int64_t)static_cast<const T*>(a.target)[r];
    const bool ignored = a.has_ignore && t == a.ignore;
    const bool in_range = t >= 0 && t < a.C;
    const int safe = (int)(t < 0 ? 0 : (t >= a.C ? a.C - 1 : t));
    const RowGroups view(row, C);
    if (ignored) {  // no loss, a zero gradient: the row is not read
      if (threadIdx.x == 0) a.row_loss[r] = CE_NO_LOSS;
      if (a.grad != nullptr)
        for (int q = threadIdx.x; q < view.groups; q += NT)
          view.store(a.grad + r * a.C, q, make_float4(0.f, 0.f, 0.f, 0.f));
      continue;
    }
    const float xt = row[safe];
    float4 v[V];
    float m = -INFINITY;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const int q = threadIdx.x + i * NT;
      v[i] = q < view.groups ? view.load(row, q, -INFINITY)
                             : make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
    }
#pragma unroll
    for (int i = 0; i < V; ++i)
      m = fmaxf(m, fmaxf(fmaxf(v[i].x, v[i].y), fmaxf(v[i].z, v[i].w)));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    __syncthreads();  // the last row's values in fm and dl have been read
    if (lane == 0) fm[w] = m;
    __syncthreads();
    m = fm[0];
#pragma unroll
    for (int i = 1; i < NT / 64; ++i) m = fmaxf(m, fm[i]);
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      if (threadIdx.x + i * NT < view.groups) {
        v[i].x = exp_rn(v[i].x - m);
        v[i].y = exp_rn(v[i].y - m);
        v[i].z = exp_rn(v[i].z - m);
        v[i].w = exp_rn(v[i].w - m);
        s += ((double)v[i].x + (double)v[i].y) + ((double)v[i].z + (double)v[i].w);
      }
      __builtin_amdgcn_sched_barrier(0);  // four exponentials at a time keep the registers down
    }
    const float sum = (float)block_sum<NT>(s, dl);
    if (threadIdx.x == 0) {
      if (!in_range) atomicOr(a.status, (uint32_t)DEV_INDEX_OUT_OF_BOUNDS);
      const float lse = m + (float)log((double)sum);
      a.row_loss[r] = in_range ? lse - xt : CE_NO_LOSS;
    }
    if (a.grad == nullptr) continue;
    const float inv = 1.0f / sum;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const int q = threadIdx.x + i * NT;
      if (q < view.groups) {
        const int c = view.first(q);
        float4 o;
        o.x = (ce_quotient(v[i].x, sum, inv) - (c == safe ? 1.0f : 0.0f)) * scale;
        o.y = (ce_quotient(v[i].y, sum, inv) - (c + 1 == safe ? 1.0f : 0.0f)) * scale;
        o.z = (ce_quotient(v[i].z, sum, inv) - (c + 2 == safe ? 1.0f : 0.0f)) * scale;
        o.w = (ce_quotient(v[i].w, sum, inv) - (c + 3 == safe ? 1.0f : 0.0f)) * scale;
        view.store(a.grad + r * a.C, q, o);
      }
    }
  }
}

// ---- rows too wide for registers: one workgroup a row, streamed ----
constexpr int CE_STREAM_NT = 1024;
template <typename T>
__global__ void __launch_bounds__(CE_STREAM_NT) ce_rows_stream(CeArgs a) {
  constexpr int NT = CE_STREAM_NT;
  __shared__ double dl[NT / 64];
  __shared__ float fm[NT / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const float scale = a.grad != nullptr ? a.g / ce_divisor<T, NT>(a, dl) : 0.0f;
  for (int64_t r = blockIdx.x; r < a.R; r += gridDim.x) {
    const float* row = a.logits + r * a.C;
    const int64_t t = (int64_t)static_cast<const T*>(a.target)[r];
    const bool ignored = a.has_ignore && t == a.ignore;
    const bool in_range = t >= 0 && t < a.C;
    if (ignored) {  // as in ce_rows_block
      if (threadIdx.x == 0) a.row_loss[r] = CE_NO_LOSS;
      if (a.grad != nullptr)
        for (int64_t c = threadIdx.x; c < a.C; c += NT) a.grad[r * a.C + c] = 0.0f;
      continue;
    }
    const int64_t safe = t < 0 ? 0 : (t >= a.C ? a.C - 1 : t);
    const float xt = row[safe];
    float m = -INFINITY;
    for (int64_t c = threadIdx.x; c < a.C; c += NT) m = fmaxf(m, row[c]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    __syncthreads();
    if (lane == 0) fm[w] = m;
    __syncthreads();
    m = fm[0];
#pragma unroll
    for (int i = 1; i < NT / 64; ++i) m = fmaxf(m, fm[i]);
    double s = 0.0;
    for (int64_t c = threadIdx.x; c < a.C; c += NT) s += (double)exp_rn(row[c] - m);
    const float sum = (float)block_sum<NT>(s, dl);
    if (threadIdx.x == 0) {
      if (!in_range) atomicOr(a.status, (uint32_t)DEV_INDEX_OUT_OF_BOUNDS);
      const float lse = m + (float)log((double)sum);
      a.row_loss[r] = in_range ? lse - xt : CE_NO_LOSS;
    }
    if (a.grad == nullptr) continue;
    const float inv = 1.0f / sum;
    for (int64_t c = threadIdx.x; c < a.C; c += NT)
      a.grad[r * a.C + c] =
          (ce_quotient(exp_rn(row[c] - m), sum, inv) - (c == safe ? 1.0f : 0.0f)) * scale;
  }
}

// Block b of four counts its part of the rows: [1000000, 10] with an ignore index and its gradient
// 1234 us on MI355X with one block, whose loads came one after the other, and the mean's loads so
// too; 540 with four and eight loads in flight in both.
template <typename T>
__global__ void __launch_bounds__(1024) ce_count_kernel(CeArgs a, uint32_t* count) {
  __shared__ double dl[16];
  const int64_t part = (a.R + 3) / 4, first = min(a.R, (int64_t)blockIdx.x * part);
  const double n = ce_count<T, 1024>(a, first, min(a.R, first + part), dl);
  if (threadIdx.x == 0) count[blockIdx.x] = (uint32_t)n;
}

// The MEAN: binary64 partials of rows 4i .. 4i+3 summed in a fixed order, one rounding, over the
// number of samples, which with an ignore index is counted from the same losses. Bound by latency:
// eight loads are in flight whatever the number of rows, those past the end reading the last group,
// and up to CE_FINISH_ROWS_WAVE rows, which one wave holds, no other wave is waited for.
// [5120, 140] with an ignore index, the loss alone: 15.6 us a step on MI355X when this block read the
// targets to count them, 8.5 so.
constexpr int64_t CE_FINISH_ROWS_WAVE = 252;
template <int NT>
__global__ void __launch_bounds__(NT) ce_finish_kernel(const float* __restrict__ row_loss, int64_t R,
                                                       int has_ignore, float* loss) {
  __shared__ double dl[NT / 64];
  __shared__ int kl[NT / 64];
  const int64_t whole = R / 4;
  const float4* quad = reinterpret_cast<const float4*>(row_loss);  // (16-byte aligned)
  double s = 0.0;
  int skipped = 0;
  for (int64_t i = threadIdx.x; i < whole; i += 8 * 256) {
    float4 v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = quad[min(i + u * 256, whole - 1)];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (i + u * 256 < whole) {
        s += (((double)v[u].x + (double)v[u].y) + (double)v[u].z) + (double)v[u].w;
        skipped += ce_no_loss(v[u].x) + ce_no_loss(v[u].y) + ce_no_loss(v[u].z) + ce_no_loss(v[u].w);
      }
    }
  }
  if (R % 4 != 0 && (int)threadIdx.x == (int)(whole % 256)) {  // the thread whose turn it is
    double q[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float v = 4 * whole + w < R ? row_loss[4 * whole + w] : 0.0f;
      q[w] = (double)v;
      skipped += ce_no_loss(v);
    }
    s += ((q[0] + q[1]) + q[2]) + q[3];
  }
  s = wave_sum(s);
  if (has_ignore) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) skipped += __shfl_xor(skipped, o, 64);
  }
  if constexpr (NT > 64) {
    if ((threadIdx.x & 63) == 0) { dl[threadIdx.x >> 6] = s; kl[threadIdx.x >> 6] = skipped; }
    __syncthreads();
    s = ((dl[0] + dl[1]) + dl[2]) + dl[3];
    skipped = (kl[0] + kl[1]) + (kl[2] + kl[3]);
  }
  if (threadIdx.x == 0) loss[0] = (float)s / (float)(double)(R - (has_ignore ? skipped : 0));
}

// Rows a workgroup counts by itself instead of a launch before: with one row a wave at most 1024
// workgroups each read 16 targets a thread (as much as a small launch takes); with one row a
// workgroup four times the workgroups do.
constexpr int64_t CE_COUNT_ROWS_WAVE = 4096, CE_COUNT_ROWS_BLOCK = 1024;
constexpr int64_t CE_WAVE_CLASSES = 1024;   // 16 floats a lane
constexpr int64_t CE_BLOCK_CLASSES = 65532; // 1024 threads x 16 groups, less a ragged lead

template <typename T, int V>
void launch_wave(const CeArgs& a, hipStream_t s) {
  hipLaunchKernelGGL((ce_rows_wave<T, V>), dim3((unsigned)((a.R + 3) / 4)), dim3(256), 0, s, a);
}
template <typename T, int NT, int V>
void launch_block(const CeArgs& a, hipStream_t s) {
  const unsigned g = (unsigned)std::min<int64_t>(a.R, 1 << 20);
  hipLaunchKernelGGL((ce_rows_block<T, NT, V>), dim3(g), dim3(NT), 0, s, a);
}

template <typename T>
hipError_t launch_typed(CeArgs a, float* loss, uint32_t* count, hipStream_t s) {
  const bool wave = a.C <= CE_WAVE_CLASSES;
  // (only a gradient is scaled before the mean is formed)
  if (a.has_ignore && a.grad != nullptr && a.R > (wave ? CE_COUNT_ROWS_WAVE : CE_COUNT_ROWS_BLOCK)) {
    hipLaunchKernelGGL(ce_count_kernel<T>, dim3(4), dim3(1024), 0, s, a, count);
    a.count = reinterpret_cast<const uint4*>(count);
  }
  // The smallest workgroup that holds the row, up to 16 groups (64 registers) a thread: 512
  // threads leave room for a second workgroup on the CU, whose loads run beside this one's
  // exponentials.
  if (a.C <= 64) launch_wave<T, 1>(a, s);
  else if (a.C <= 128) launch_wave<T, 2>(a, s);
  else if (a.C <= 256) launch_wave<T, 4>(a, s);
  else if (a.C <= 512) launch_wave<T, 8>(a, s);
  else if (wave) launch_wave<T, 16>(a, s);
  else if (a.C <= 256 * 4 * 2 - 4) launch_block<T, 256, 2>(a, s);
  else if (a.C <= 256 * 4 * 4 - 4) launch_block<T, 256, 4>(a, s);
  else if (a.C <= 256 * 4 * 8 - 4) launch_block<T, 256, 8>(a, s);
  else if (a.C <= 512 * 4 * 8 - 4) launch_block<T, 512, 8>(a, s);
  else if (a.C <= 512 * 4 * 16 - 4) launch_block<T, 512, 16>(a, s);
  else if (a.C <= CE_BLOCK_CLASSES) launch_block<T, 1024, 16>(a, s);
  else
    hipLaunchKernelGGL(ce_rows_stream<T>, dim3((unsigned)std::min<int64_t>(a.R, 1 << 20)),
                       dim3(CE_STREAM_NT), 0, s, a);
  if (a.R <= CE_FINISH_ROWS_WAVE)
    hipLaunchKernelGGL(ce_finish_kernel<64>, dim3(1), dim3(64), 0, s, a.row_loss, a.R, a.has_ignore, loss);
  else
    hipLaunchKernelGGL(ce_finish_kernel<256>, dim3(1), dim3(256), 0, s, a.row_loss, a.R, a.has_ignore, loss);
  return hipGetLastError();
}

}  // namespace

// R row losses (floats), then the four sample counts.
int64_t index_ce_partial_doubles(int64_t R) { return 2 * ((R + 3) / 4) + 2; }

hipError_t launch_index_ce(const float* logits, const void* target, int target_is_64,
                           float* loss, float* grad, int64_t R, int64_t C, int has_ignore,
                           int64_t ignore_index, float g, double* partial, uint32_t* status,
                           hipStream_t s) {
  if (R <= 0) return hipSuccess;
  CeArgs a{};
  a.logits = logits;
  a.target = target;
  a.grad = grad;
  a.row_loss = reinterpret_cast<float*>(partial);
  a.status = status;
  a.R = R;
  a.C = C;
  a.ignore = ignore_index;
  a.has_ignore = has_ignore;
  a.g = g;
  uint32_t* count = reinterpret_cast<uint32_t*>(partial + 2 * ((R + 3) / 4));
  return target_is_64 ? launch_typed<int64_t>(a, loss, count, s)
                      : launch_typed<int32_t>(a, loss, count, s);
}

}  // namespace shk
