// Fused elementwise chains and SUM/MEAN/MAX reductions for gfx950.
//
// Pointwise: the reference fuses elementwise/activation chains into one generated kernel per
// chain (CPU: CpuPointwiseGeneratedKernelTest; Metal: SynaptikPointwiseFusionKernelSource.h,
// a runtime-generated instruction-list unit). Here one precompiled kernel interprets a short
// register-machine program held in the kernel arguments: the opcode stream is wave-uniform, so
// every branch is scalar and the kernel stays HBM-bound with one read per input and one write
// per output, four elements per thread through 128-bit accesses.
//
// Reductions: SUM/MEAN/SUM_TO_SHAPE are exact in the reference (fixed-width limb accumulation
// rounded once, CpuExactSumEmitter.java:4-12, CpuAggregateEmitter.java:18-20). The GPU
// accumulates binary32 inputs in binary64 through a fixed-shape tree (wave shuffles, then LDS,
// then a second deterministic pass) and rounds once; that equals the exactly rounded sum
// unless the binary64 accumulation error crosses a binary32 rounding boundary. MAX follows
// Java Math.max (NaN wins, +0.0 beats -0.0).
#include "common.h"
#include "kernels.h"
#include "pw_divide.h"
#include "rowvec.h"
#include <algorithm>
#include <type_traits>

namespace shk {
namespace {

enum PwOp : uint8_t {
  PW_LOAD = 0,     // r[dst] = in[a]
  PW_CONST = 1,    // r[dst] = imm
  PW_ADD = 2, PW_SUB = 3, PW_MUL = 4, PW_DIV = 5,
  PW_NEG = 6,
  PW_RELU = 7, PW_TANH = 8, PW_SIGMOID = 9,
  PW_EXP = 10, PW_LOG = 11,
  PW_RELU_GRAD = 12,     // r[dst] = r[a] > 0 ? r[b] : 0          (WHERE(x > 0, g, 0))
  PW_TANH_GRAD = 13,     // r[dst] = r[b] * (1 - r[a]*r[a])      (a = y, b = g)
  PW_SIGMOID_GRAD = 14,  // r[dst] = (r[b] * r[a]) * (1 - r[a])  (a = y, b = g)
  PW_GT = 15,            // r[dst] = r[a] > r[b] ? 1 : 0
  PW_WHERE = 16,         // r[dst] = r[c] != 0 ? r[a] : r[b]
  PW_STORE = 17,         // out[dst] = r[a]
  PW_MAX = 18,           // Java Math.max
  PW_SQRT = 19,
};
constexpr int PW_REGS = 8;

// Library functions kept out of line: they are rare in chains, and inlining them into the
// interpreter inflates the register allocation of the whole kernel. (exp, tanh and sigmoid are
// short: fexp64.h.)
__device__ __noinline__ float pw_log(float a) { return (float)log((double)a); }
__device__ __noinline__ float pw_sqrt(float a) { return (float)sqrt((double)a); }

// One instruction's value from its operands (a, b, c registers; imm for CONST). Shared by the
// interpreter (op known at run time) and the single-op kernels (op a template constant).
__device__ __forceinline__ float pw_op(int op, float a, float b, float c, float imm) {
  switch (op) {
    case PW_CONST: return imm;
    case PW_ADD: return a + b;
    case PW_SUB: return a - b;
    case PW_MUL: return a * b;
    case PW_DIV: return a / b;
    case PW_NEG: return -a;
    case PW_RELU: return relu_f(a);
    case PW_TANH: return tanh_f(a);
    case PW_SIGMOID: return sigmoid_f(a);
    case PW_EXP: return exp_rn(a);
    case PW_LOG: return pw_log(a);
    case PW_RELU_GRAD: return act_grad(ACT_RELU, b, a);
    case PW_TANH_GRAD: return act_grad(ACT_TANH, b, a);
    case PW_SIGMOID_GRAD: return act_grad(ACT_SIGMOID, b, a);
    case PW_GT: return a > b ? 1.0f : 0.0f;
    case PW_WHERE: return (c != 0.0f) ? a : b;
    case PW_STORE: return a;
    case PW_MAX: return java_max(a, b);
    case PW_SQRT: return pw_sqrt(a);
    default: return 0.0f;
  }
}

constexpr bool pw_reads_b(int op) {
  return op == PW_ADD || op == PW_SUB || op == PW_MUL || op == PW_DIV || op == PW_MAX ||
         op == PW_GT || op == PW_RELU_GRAD || op == PW_TANH_GRAD || op == PW_SIGMOID_GRAD ||
         op == PW_WHERE;
}

// Single-op chains (LOAD x [, LOAD y], OP, STORE) over full-shape, 16-byte aligned operands (out
// may be one of them: each element is read before it is written): out
// = OP(x, y) element by element with the interpreter's arithmetic (pw_op), streaming 16-byte
// accesses, two groups of four per thread and iteration, no interpreter.
template <int OP, bool BIN>
__global__ void __launch_bounds__(256) pw_single_kernel(const float* x,
                                                        const float* y,
                                                        float* out, int64_t n) {
  const int64_t n4 = n / 4;
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x; q < n4; q += 2 * stride) {
    const bool two = q + stride < n4;
    const float4 xa = ld_stream(reinterpret_cast<const float4*>(x) + q);
    const float4 ya = BIN ? ld_stream(reinterpret_cast<const float4*>(y) + q) : xa;
    float4 xb = xa, yb = ya;
    if (two) {
      xb = ld_stream(reinterpret_cast<const float4*>(x) + q + stride);
      yb = BIN ? ld_stream(reinterpret_cast<const float4*>(y) + q + stride) : xb;
    }
    st_stream(reinterpret_cast<float4*>(out) + q,
              make_float4(pw_op(OP, xa.x, ya.x, 0.f, 0.f), pw_op(OP, xa.y, ya.y, 0.f, 0.f),
                          pw_op(OP, xa.z, ya.z, 0.f, 0.f), pw_op(OP, xa.w, ya.w, 0.f, 0.f)));
    if (two)
      st_stream(reinterpret_cast<float4*>(out) + q + stride,
                make_float4(pw_op(OP, xb.x, yb.x, 0.f, 0.f), pw_op(OP, xb.y, yb.y, 0.f, 0.f),
                            pw_op(OP, xb.z, yb.z, 0.f, 0.f), pw_op(OP, xb.w, yb.w, 0.f, 0.f)));
  }
  if (blockIdx.x == 0 && threadIdx.x < n - n4 * 4) {
    const int64_t i = n4 * 4 + threadIdx.x;
    out[i] = pw_op(OP, x[i], BIN ? y[i] : x[i], 0.f, 0.f);
  }
}

// The interpreter. A thread handles one group of four elements, whose register k lives in LDS at
// regs[k * PW_NT + t]: any register index is just an address (no dynamically indexed VGPR array, no
// scratch) and each operand access is one 128-bit LDS access per lane. A launch takes only as many
// registers as its chain uses.
//
// What bounds it is the instructions around the arithmetic -- decoding, branching on the operation
// and on each input's kind -- and how many waves share them: seven a SIMD for chains that name up
// to five registers; six and five for six and for seven or eight, whose workgroups take 24 to 32 KB
// of a CU's 160 KB of LDS. An ordinal is divided
// once, by multiplication; a broadcast operand within one row is one vector load; an instruction
// is read as words (read as bytes it would come through vector memory: scalar loads have none), the
// next one's ahead of time. Before: a 64-bit division and four loads for each broadcast operand,
// five workgroups a CU whatever the chain. [20000, 1001] on MI355X: x - row 75 -> 44 us;
// tanh(d / row * row + row) 176 -> 123. (Two groups a thread 56 and 153, four 107 and 180, for
// want of registers; one group with every input loaded ahead 70 to 77 and 145 to 151.)
constexpr int PW_NT = 256;

struct PwArgs {
  PwParams p;
  PwDivide div;
};

struct PwWords {
  uint32_t w0, w1, w2;  // op | dst << 8 | a << 16 | b << 24; c; imm
};
static_assert(sizeof(PwInstr) == sizeof(PwWords) && alignof(PwInstr) == 4, "three words");
__device__ __forceinline__ PwWords pw_fetch(const PwParams& p, int pc) {
  const uint32_t* w = reinterpret_cast<const uint32_t*>(p.code) + 3 * pc;
  return PwWords{w[0], w[1], w[2]};
}

__device__ __forceinline__ float4 pw_vec(const float* src) {
  const float4u v = *reinterpret_cast<const float4u*>(src);
  return make_float4(v[0], v[1], v[2], v[3]);
}

// Element by element: the group of four from e0 on, cnt of them valid, at (row, col).
__device__ __forceinline__ float4 pw_load_each(const float* src, int mode, int64_t C, int64_t e0,
                                               int cnt, int64_t row, int64_t col) {
  float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (q < cnt) {
      v[q] = src[mode == 0 ? e0 + q : mode == 1 ? col : mode == 2 ? row : 0];
      if (++col == C) { col = 0; ++row; }
    }
  }
  return make_float4(v[0], v[1], v[2], v[3]);
}

// BCAST: some input is a row or a column vector. WIDE: ordinals beyond 32 bits (or C == 1).
template <bool BCAST, bool WIDE>
__global__ void __launch_bounds__(PW_NT) __attribute__((amdgpu_waves_per_eu(7)))
pointwise_kernel(PwArgs a) {
  using Place = typename std::conditional<WIDE, int64_t, uint32_t>::type;
  extern __shared__ float4 regs[];
  const PwParams& p = a.p;
  const int64_t n = p.R * p.C;
  const int t = threadIdx.x;
  const Place C = (Place)p.C;
  constexpr int64_t TILE = (int64_t)PW_NT * 4;
  for (int64_t base = (int64_t)blockIdx.x * TILE; base < n; base += (int64_t)gridDim.x * TILE) {
    const bool whole = base + TILE <= n;  // uniform: every group has four elements
    const int64_t e0 = base + t * 4;
    auto count = [&]() { return (int)max<int64_t>(0, min<int64_t>(4, n - e0)); };
    Place row = 0, col = 0;
    if constexpr (BCAST) {
      if constexpr (WIDE) {
        row = e0 / C;
        col = e0 - row * C;
      } else {
        const uint32_t e = (uint32_t)e0;
        row = pw_quotient(a.div.mul, a.div.shift, e);
        col = e - row * C;
      }
    }
    // (stored after the whole chain: an output may be one of the inputs)
    float4 outv[PW_MAX_OUTPUTS];
    outv[0] = outv[1] = make_float4(0.f, 0.f, 0.f, 0.f);
    PwWords next = pw_fetch(p, 0);
    for (int pc = 0; pc < p.n_instr; ++pc) {
      const PwWords ins = next;
      if (pc + 1 < p.n_instr) next = pw_fetch(p, pc + 1);
      const int op = ins.w0 & 0xff, dst = (ins.w0 >> 8) & 0xff;
      const float imm = __uint_as_float(ins.w2);
      float4* const D = regs + (dst & (PW_REGS - 1)) * PW_NT + t;
      if (op == PW_LOAD) {
        const int k = ((ins.w0 >> 16) & 0xff) % PW_MAX_INPUTS;
        const float* src = p.in[k];
        const int mode = (int)p.in_mode[k];
        float4 v;
        if (mode == 3) {
          const float x = src[0];
          v = make_float4(x, x, x, x);
        } else if (mode == 0 && whole) {
          const float4u x = __builtin_nontemporal_load(reinterpret_cast<const float4u*>(src + e0));
          v = make_float4(x[0], x[1], x[2], x[3]);
        } else if (!whole) {
          v = pw_load_each(src, mode, p.C, e0, count(), row, col);
        } else if (col + 3 >= C) {  // spans rows
          v = pw_load_each(src, mode, p.C, e0, 4, row, col);
        } else if (mode == 1) {
          v = pw_vec(src + col);
        } else {
          const float x = src[row];
          v = make_float4(x, x, x, x);
        }
        *D = v;
        continue;
      }
      const float4* const A = regs + ((ins.w0 >> 16) & (PW_REGS - 1)) * PW_NT + t;
      const float4* const B = regs + ((ins.w0 >> 24) & (PW_REGS - 1)) * PW_NT + t;
      const float4* const Cc = regs + (ins.w1 & (PW_REGS - 1)) * PW_NT + t;
      float4 d;
#define PW_CASE(OP)                                                                             \
  case OP: {                                                                                    \
    const float4 x = *A;                                                                        \
    const float4 y = pw_reads_b(OP) ? *B : x;                                                   \
    const float4 z = OP == PW_WHERE ? *Cc : x;                                                  \
    d = make_float4(pw_op(OP, x.x, y.x, z.x, imm), pw_op(OP, x.y, y.y, z.y, imm),               \
                    pw_op(OP, x.z, y.z, z.z, imm), pw_op(OP, x.w, y.w, z.w, imm));              \
  } break;
      switch (op) {  // (uniform)
        PW_CASE(PW_CONST) PW_CASE(PW_ADD) PW_CASE(PW_SUB) PW_CASE(PW_MUL) PW_CASE(PW_DIV)
        PW_CASE(PW_NEG) PW_CASE(PW_RELU) PW_CASE(PW_TANH) PW_CASE(PW_SIGMOID) PW_CASE(PW_EXP)
        PW_CASE(PW_LOG) PW_CASE(PW_RELU_GRAD) PW_CASE(PW_TANH_GRAD) PW_CASE(PW_SIGMOID_GRAD)
        PW_CASE(PW_GT) PW_CASE(PW_WHERE) PW_CASE(PW_STORE) PW_CASE(PW_MAX) PW_CASE(PW_SQRT)
        default: d = make_float4(0.f, 0.f, 0.f, 0.f);
      }
#undef PW_CASE
      if (op == PW_STORE) {
        if (dst & 1) outv[1] = d;
        else outv[0] = d;
      } else {
        *D = d;
      }
    }
#pragma unroll
    for (int o = 0; o < PW_MAX_OUTPUTS; ++o) {
      if (p.out[o] == nullptr) continue;
      float* dst = p.out[o] + e0;
      const float4 v = outv[o];
      if (whole) {
        __builtin_nontemporal_store(float4u{v.x, v.y, v.z, v.w}, reinterpret_cast<float4u*>(dst));
      } else {
        const int cnt = count();
        if (cnt > 0) dst[0] = v.x;
        if (cnt > 1) dst[1] = v.y;
        if (cnt > 2) dst[2] = v.z;
        if (cnt > 3) dst[3] = v.w;
      }
    }
  }
}

__global__ void fill_kernel(float* x, int64_t n, float v) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    x[i] = v;
}
__global__ void fill_u32_kernel(uint32_t* x, int64_t n, uint32_t v) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    x[i] = v;
}
// One float4 per thread, streamed past the caches: many short workgroups keep the most bytes
// in flight per CU (measured on MI355X: 6.7 TB/s for a 1 GiB copy, against 5.2-5.8 TB/s for
// grid-stride loops and 5.2 TB/s for a device-to-device hipMemcpy).
__global__ void __launch_bounds__(256) copy_vec_kernel(const float4* __restrict__ s,
                                                       float4* __restrict__ d, int64_t n4) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n4) st_stream(&d[i], ld_stream(&s[i]));
}
__global__ void copy_kernel(const float* __restrict__ s, float* __restrict__ d, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    d[i] = s[i];
}

// Column sums, pass 1: block (cx, ry) sums a 64-column x `rows`-row panel; each of the 4 waves
// walks a quarter of the panel's rows with lanes on consecutive columns (coalesced 256 B rows).
// The panel height is chosen per call so that a launch has ~1024 blocks even for short inputs.
constexpr int CS_COLS = 64;
constexpr int64_t CS_TARGET_BLOCKS = 1024;
int64_t colsum_rows_per_panel(int64_t R, int64_t N) {
  const int64_t colblocks = (N + CS_COLS - 1) / CS_COLS;
  const int64_t panels = std::max<int64_t>(1, (CS_TARGET_BLOCKS + colblocks - 1) / colblocks);
  int64_t rows = (R + panels - 1) / panels;
  rows = std::max<int64_t>(64, ((rows + 3) / 4) * 4);
  return rows;
}
__global__ void __launch_bounds__(256) colsum_pass1(const float* __restrict__ x, double* part,
                                                   int64_t R, int64_t N, int64_t ldx, int64_t rows) {
  __shared__ double lds[4][CS_COLS];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t col = (int64_t)blockIdx.x * CS_COLS + lane;
  const int64_t r0 = (int64_t)blockIdx.y * rows;
  double s = 0.0;
  if (col < N) {
    const int64_t rend = min<int64_t>(R, r0 + rows);
    for (int64_t r = r0 + w; r < rend; r += 4) s += (double)x[r * ldx + col];
  }
  lds[w][lane] = s;
  __syncthreads();
  if (w == 0 && col < N)
    part[(int64_t)blockIdx.y * N + col] = ((lds[0][lane] + lds[1][lane]) + lds[2][lane]) + lds[3][lane];
}
// Pass 1 for wider inputs: each lane owns four adjacent columns and reads them with one streaming
// 16-byte load per row (at any float), so a wave moves 1 KiB per row and a block covers 256
// columns with 16 waves (rows r0 + w, r0 + w + 16, ..., four loads in flight each; a quarter of
// colsum_pass1's blocks, so four times its waves). With 4-byte loads too few bytes are in flight:
// [20000, 1001] 40.8 us on MI355X, 21.7 so. Up to CS_FEW_ROWS rows four waves do: the others
// would only be launched and waited for ([8, 1000000] 27.3 us a call against 33.4).
constexpr int64_t CS_FEW_ROWS = 32;
// Few unaligned rows go to colsum_pass1, whose four times as many blocks are done sooner than a
// lane's four ragged columns. us a step, there and here: [16, 301] 4.5 and 5.0, [32, 1001] 4.8 and
// 5.7, [33, 100001] 6.0 and 6.5, [2, 1000001] 12.1 and 14.0; [64, 301] 5.7 and 5.4, [16, 1000001]
// 24.6 and 22.2.
constexpr int64_t CS_FEW_UNALIGNED = 48, CS_FEW_COLS = 1 << 18;
template <int CS_WAVES>
__global__ void __launch_bounds__(64 * CS_WAVES) colsum_pass1_v4(const float* __restrict__ x,
                                                                double* part, int64_t R, int64_t N,
                                                                int64_t ldx, int64_t rows) {
  __shared__ double lds[CS_WAVES][4 * CS_COLS];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t col = ((int64_t)blockIdx.x * CS_COLS + lane) * 4;
  const int64_t r0 = (int64_t)blockIdx.y * rows;
  const int64_t rend = min<int64_t>(R, r0 + rows);
  double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
  if (col + 3 < N) {
#pragma unroll 4
    for (int64_t r = r0 + w; r < rend; r += CS_WAVES) {
      const float4u v = __builtin_nontemporal_load(reinterpret_cast<const float4u*>(x + r * ldx + col));
      s0 += (double)v[0];
      s1 += (double)v[1];
      s2 += (double)v[2];
      s3 += (double)v[3];
    }
  } else if (col < N) {  // the last one to three columns
    for (int64_t r = r0 + w; r < rend; r += CS_WAVES) {
      const float* src = x + r * ldx + col;
      s0 += (double)src[0];
      if (col + 1 < N) s1 += (double)src[1];
      if (col + 2 < N) s2 += (double)src[2];
    }
  }
  lds[w][4 * lane + 0] = s0;
  lds[w][4 * lane + 1] = s1;
  lds[w][4 * lane + 2] = s2;
  lds[w][4 * lane + 3] = s3;
  __syncthreads();
  const int c = threadIdx.x;  // one column of the block's 256 per thread
  const int64_t gc = (int64_t)blockIdx.x * 4 * CS_COLS + c;
  if (c < 4 * CS_COLS && gc < N) {
    double s = lds[0][c];
#pragma unroll
    for (int i = 1; i < CS_WAVES; ++i) s += lds[i][c];
    part[(int64_t)blockIdx.y * N + gc] = s;
  }
}
// Column sums of a narrow input in one launch (N <= CS_SMALL_MAX_N, R <= CS_SMALL_MAX_R): block
// x sums 64 columns over all R rows with 16 waves (wave w: rows w, w + 16, ..., eight loads in
// flight), the waves' binary64 sums are added in wave order through LDS and finished as
// colsum_pass2 does.
constexpr int64_t CS_SMALL_MAX_N = 256;
constexpr int64_t CS_SMALL_MAX_R = 32768;
__global__ void __launch_bounds__(1024) colsum_small(const float* __restrict__ x, float* out,
                                                    int64_t R, int64_t N, int64_t ldx,
                                                    double divisor, int accumulate) {
  __shared__ double lds[16][CS_COLS];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t col = (int64_t)blockIdx.x * CS_COLS + lane;
  double s = 0.0;
  if (col < N) {
    int64_t r = w;
    for (; r + 7 * 16 < R; r += 8 * 16) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = x[(r + u * 16) * ldx + col];
#pragma unroll
      for (int u = 0; u < 8; ++u) s += (double)v[u];
    }
    for (; r < R; r += 16) s += (double)x[r * ldx + col];
  }
  lds[w][lane] = s;
  __syncthreads();
  if (w == 0 && col < N) {
    double t = lds[0][lane];
#pragma unroll
    for (int i = 1; i < 16; ++i) t += lds[i][lane];
    float v = (float)(t / divisor);
    if (accumulate) v = out[col] + v;
    out[col] = v;
  }
}
// Many partial rows are folded first: block (x, y) adds rows y * chunk .. of 64 columns into the
// first of them (in the order rows w, w + 4, ... of wave w, then the waves), eight loads in flight.
// A single block of pass 2 per 64 columns takes 67 us for the 1876 rows that the bias gradient of
// 30001 rows leaves on MI355X; folded, both launches take 9.5.
constexpr int64_t CS_FOLD_ROWS = 256, CS_FOLD_CHUNK = 64;
__global__ void __launch_bounds__(256) colsum_fold(double* part, int64_t P, int64_t N) {
  __shared__ double lds[4][CS_COLS];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t col = (int64_t)blockIdx.x * CS_COLS + lane;
  const int64_t r0 = (int64_t)blockIdx.y * CS_FOLD_CHUNK, rend = min(P, r0 + CS_FOLD_CHUNK);
  double s = 0.0;
  if (col < N) {
#pragma unroll 8
    for (int64_t i = r0 + w; i < rend; i += 4) s += part[i * N + col];
  }
  lds[w][lane] = s;
  __syncthreads();  // (the block has read its rows)
  if (w == 0 && col < N)
    part[r0 * N + col] = ((lds[0][lane] + lds[1][lane]) + lds[2][lane]) + lds[3][lane];
}
// Column sums, pass 2: block x finishes 64 columns of P partial rows `step` apart; wave w adds
// partial rows w, w + 4, ... in two interleaved chains (independent loads in flight), then the
// chains and the four waves are combined in a fixed order, so results are run-to-run identical.
__global__ void __launch_bounds__(256) colsum_pass2(const double* part, float* out, int64_t P,
                                                    int64_t N, int64_t step, double divisor,
                                                    int accumulate) {
  __shared__ double lds[4][CS_COLS];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t col = (int64_t)blockIdx.x * CS_COLS + lane;
  double s0 = 0.0, s1 = 0.0;
  if (col < N) {
    int64_t i = w;
    for (; i + 4 < P; i += 8) {
      s0 += part[i * step + col];
      s1 += part[(i + 4) * step + col];
    }
    if (i < P) s0 += part[i * step + col];
  }
  lds[w][lane] = s0 + s1;
  __syncthreads();
  if (w == 0 && col < N) {
    const double s = ((lds[0][lane] + lds[1][lane]) + lds[2][lane]) + lds[3][lane];
    float v = (float)(s / divisor);
    if (accumulate) v = out[col] + v;
    out[col] = v;
  }
}

// Row reductions, binary64 accumulation for SUM/MEAN/LSE, one read of each row in aligned 16-byte
// groups (rowvec.h), V of them a thread held in registers (LOG_SUM_EXP looks at them twice). Rows of
// at most 2044 take one wave each: a workgroup a row spends its time in barriers and a single
// load's latency. Wider rows take a workgroup of 256. From 8189 on SUM and MEAN read 4 bytes at a
// time, eight loads in flight ([20000, 20000] 269 us a call, held by 1024 threads 363); MAX and
// LOG_SUM_EXP, which look at a value twice or have more to do for it, are held by 512 and from
// 16381 on by 1024 threads up to 32764, then read 4 bytes at a time (once more for LOG_SUM_EXP).
// MI355X, one workgroup of 256 a row with 4-byte loads before: [20000, 1001] MAX 39, MEAN 22,
// LOG_SUM_EXP 58 us, now 14, 16 and 30; LOG_SUM_EXP of [65536, 10000] 1465 us a call, now 843, of
// [3000, 30000] 259, now 151, of [64, 100000] 159, now 92.
constexpr int RR_NT = 256;

__device__ __forceinline__ float row_lse(float m, float shift, double s) {
  if (m != m) return m;
  if (m == INFINITY) return INFINITY;
  return shift + (float)log((double)(float)s);
}

// This thread's share of the row statistics (Math.max: a NaN anywhere gives NaN, +0 beats -0).
// The hardware maximum skips NaN and does not order zeros; a flag and, where the maximum is a
// zero, a second look put that right.
template <int V>
struct RowPart {
  float4 v[V];
  int n;  // groups held
  template <int STRIDE>
  __device__ __forceinline__ void load(const RowGroups& view, const float* row, int first, float fill) {
    n = 0;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const bool in = first + i * STRIDE < view.groups;
      v[i] = in ? view.load(row, first + i * STRIDE, fill) : make_float4(fill, fill, fill, fill);
      n += in;
    }
  }
  __device__ __forceinline__ float maximum(int& nan) const {
    float m = -INFINITY;
    nan = 0;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      m = fmaxf(m, fmaxf(fmaxf(v[i].x, v[i].y), fmaxf(v[i].z, v[i].w)));
      nan |= (v[i].x != v[i].x) | (v[i].y != v[i].y) | (v[i].z != v[i].z) | (v[i].w != v[i].w);
    }
    return m;
  }
  __device__ __forceinline__ int positive_zero() const {
    int z = 0;
#pragma unroll
    for (int i = 0; i < V; ++i)
      z |= (__float_as_uint(v[i].x) == 0u) | (__float_as_uint(v[i].y) == 0u) |
           (__float_as_uint(v[i].z) == 0u) | (__float_as_uint(v[i].w) == 0u);
    return z;
  }
  __device__ __forceinline__ double sum() const {
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      s0 += (double)v[i].x;
      s1 += (double)v[i].y;
      s2 += (double)v[i].z;
      s3 += (double)v[i].w;
    }
    return (s0 + s1) + (s2 + s3);
  }
  // (padding is -inf, whose exponential is 0)
  __device__ __forceinline__ double sum_exp(float shift) const {
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < V; ++i)
      if (i < n)
        s += ((double)exp_rn(v[i].x - shift) + (double)exp_rn(v[i].y - shift)) +
             ((double)exp_rn(v[i].z - shift) + (double)exp_rn(v[i].w - shift));
    return s;
  }
};

__device__ __forceinline__ float wave_fmax(float m) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  return m;
}

// One wave a row, four rows a workgroup.
template <int KIND, int V>
__global__ void __launch_bounds__(RR_NT) row_reduce_wave(const float* __restrict__ x, float* out,
                                                         int64_t R, int64_t C) {
  const int lane = threadIdx.x & 63;
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= R) return;
  const float* row = x + r * C;
  const RowGroups view(row, (int)C);
  RowPart<V> part;
  part.template load<64>(view, row, lane, KIND >= 2 ? -INFINITY : 0.0f);
  float result;
  if constexpr (KIND < 2) {
    const double s = wave_sum(part.sum());
    result = KIND == 1 ? (float)(s / (double)C) : (float)s;
  } else {
    int nan;
    float m = wave_fmax(part.maximum(nan));
    if (__any(nan)) m = NAN;
    else if (m == 0.0f) m = __any(part.positive_zero()) ? 0.0f : -0.0f;
    result = m;
    if constexpr (KIND == 3) {
      // LOG_SUM_EXP: shifted exponentials, one logarithm (CpuLogSumExpEmitter.java:4-9)
      const float shift = (m == INFINITY || m == -INFINITY) ? 0.0f : m;
      result = row_lse(m, shift, wave_sum(part.sum_exp(shift)));
    }
  }
  if (lane == 0) out[r] = result;
}

// One workgroup of NT threads a row; V = 0: any width.
template <int NT, int KIND, int V>
__global__ void __launch_bounds__(NT) row_reduce_block(const float* __restrict__ x, float* out,
                                                       int64_t R, int64_t C) {
  constexpr int NW = NT / 64;
  __shared__ double dl[NW];
  __shared__ float fl[NW];
  __shared__ int nl[NW];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  for (int64_t r = blockIdx.x; r < R; r += gridDim.x) {
    const float* row = x + r * C;
    __syncthreads();  // the shared values of the row before have been read
    if constexpr (V == 0) {
      if constexpr (KIND < 2) {
        double s = 0.0;
#pragma unroll 8
        for (int64_t c = tid; c < C; c += NT) s += (double)row[c];
        s = block_sum<NT>(s, dl);
        if (tid == 0) out[r] = KIND == 1 ? (float)(s / (double)C) : (float)s;
      } else {
        float m = -INFINITY;
        for (int64_t c = tid; c < C; c += NT) m = java_max(m, row[c]);
        m = block_max<NT>(m, fl);
        if constexpr (KIND == 2) {
          if (tid == 0) out[r] = m;
        } else {
          const float shift = (m == INFINITY || m == -INFINITY) ? 0.0f : m;
          double s = 0.0;
          for (int64_t c = tid; c < C; c += NT) s += (double)exp_rn(row[c] - shift);
          s = block_sum<NT>(s, dl);
          if (tid == 0) out[r] = row_lse(m, shift, s);
        }
      }
    } else {
      const RowGroups view(row, (int)C);
      RowPart<V> part;
      part.template load<NT>(view, row, tid, KIND >= 2 ? -INFINITY : 0.0f);
      if constexpr (KIND < 2) {
        const double s = block_sum<NT>(part.sum(), dl);
        if (tid == 0) out[r] = KIND == 1 ? (float)(s / (double)C) : (float)s;
      } else {
        int nan;
        float m = wave_fmax(part.maximum(nan));
        nan = __any(nan);
        auto any = [&]() {
          int a = nl[0];
#pragma unroll
          for (int i = 1; i < NW; ++i) a |= nl[i];
          return a;
        };
        if (lane == 0) { fl[w] = m; nl[w] = nan; }
        __syncthreads();
        m = fl[0];
#pragma unroll
        for (int i = 1; i < NW; ++i) m = fmaxf(m, fl[i]);
        if (any()) {
          m = NAN;
        } else if (m == 0.0f) {  // the same for the whole workgroup
          const int z = __any(part.positive_zero());
          __syncthreads();
          if (lane == 0) nl[w] = z;
          __syncthreads();
          m = any() ? 0.0f : -0.0f;
        }
        if constexpr (KIND == 2) {
          if (tid == 0) out[r] = m;
        } else {
          const float shift = (m == INFINITY || m == -INFINITY) ? 0.0f : m;
          const double s = block_sum<NT>(part.sum_exp(shift), dl);
          if (tid == 0) out[r] = row_lse(m, shift, s);
        }
      }
    }
  }
}

template <int KIND>
void launch_row_kind(const float* x, float* out, int64_t R, int64_t C, hipStream_t s) {
  const dim3 rows((unsigned)std::min<int64_t>(R, 1 << 20)), quads((unsigned)((R + 3) / 4)), nt(RR_NT);
  // V groups hold rows of at most 4 V (threads) - 4 floats: a ragged start takes up to three
  if (C <= 64 * 4 * 1 - 4) hipLaunchKernelGGL((row_reduce_wave<KIND, 1>), quads, nt, 0, s, x, out, R, C);
  else if (C <= 64 * 4 * 2 - 4) hipLaunchKernelGGL((row_reduce_wave<KIND, 2>), quads, nt, 0, s, x, out, R, C);
  else if (C <= 64 * 4 * 4 - 4) hipLaunchKernelGGL((row_reduce_wave<KIND, 4>), quads, nt, 0, s, x, out, R, C);
  else if (C <= 64 * 4 * 8 - 4) hipLaunchKernelGGL((row_reduce_wave<KIND, 8>), quads, nt, 0, s, x, out, R, C);
  else if (C <= 256 * 4 * 4 - 4) hipLaunchKernelGGL((row_reduce_block<256, KIND, 4>), rows, nt, 0, s, x, out, R, C);
  else if (C <= 256 * 4 * 8 - 4) hipLaunchKernelGGL((row_reduce_block<256, KIND, 8>), rows, nt, 0, s, x, out, R, C);
  else if constexpr (KIND < 2)
    hipLaunchKernelGGL((row_reduce_block<256, KIND, 0>), rows, nt, 0, s, x, out, R, C);
  else if (C <= 512 * 4 * 8 - 4) hipLaunchKernelGGL((row_reduce_block<512, KIND, 8>), rows, dim3(512), 0, s, x, out, R, C);
  else if (C <= 1024 * 4 * 8 - 4) hipLaunchKernelGGL((row_reduce_block<1024, KIND, 8>), rows, dim3(1024), 0, s, x, out, R, C);
  else hipLaunchKernelGGL((row_reduce_block<512, KIND, 0>), rows, dim3(512), 0, s, x, out, R, C);
}

// Whole-tensor reductions in two deterministic passes.
constexpr int RA_BLOCKS = 1024;
__global__ void __launch_bounds__(256) reduce_all_pass1(const float* __restrict__ x, int64_t n,
                                                       int kind, double* part) {
  __shared__ double dl[4];
  __shared__ float fl[4];
  const int64_t stride = (int64_t)gridDim.x * 256;
  if (kind == 2) {
    float m = -INFINITY;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) m = java_max(m, x[i]);
    m = block_max<256>(m, fl);
    if (threadIdx.x == 0) part[blockIdx.x] = (double)m;
    return;
  }
  // 16-byte loads, four a thread in flight ([20020000] SUM 24.4 us with 4-byte loads on MI355X,
  // 14.4 so)
  double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
  const int64_t n4 = n / 4;
#pragma unroll 4
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += stride) {
    const float4u v = __builtin_nontemporal_load(reinterpret_cast<const float4u*>(x) + i);
    s0 += (double)v[0];
    s1 += (double)v[1];
    s2 += (double)v[2];
    s3 += (double)v[3];
  }
  if (blockIdx.x == 0 && threadIdx.x < n - 4 * n4) s0 += (double)x[4 * n4 + threadIdx.x];
  const double s = block_sum<256>((s0 + s1) + (s2 + s3), dl);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}
__global__ void __launch_bounds__(256) reduce_all_pass2(const double* part, int P, int64_t n,
                                                       int kind, float* out) {
  __shared__ double dl[4];
  __shared__ float fl[4];
  if (kind == 2) {
    float m = -INFINITY;
    for (int i = threadIdx.x; i < P; i += 256) m = java_max(m, (float)part[i]);
    m = block_max<256>(m, fl);
    if (threadIdx.x == 0) out[0] = m;
    return;
  }
  double s = 0.0;
  for (int i = threadIdx.x; i < P; i += 256) s += part[i];
  s = block_sum<256>(s, dl);
  if (threadIdx.x == 0) out[0] = kind == 1 ? (float)(s / (double)n) : (float)s;
}

// Rank-2 transpose (PERMUTE [1,0] materialized): 32x32 tiles staged through LDS (padded pitch)
// so both the read of X and the write of Y are coalesced.
__global__ void __launch_bounds__(256) transpose_kernel(const float* __restrict__ x,
                                                        float* __restrict__ y, int64_t R,
                                                        int64_t C) {
  __shared__ float tile[32][33];
  const int64_t r0 = (int64_t)blockIdx.y * 32, c0 = (int64_t)blockIdx.x * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int k = ty; k < 32; k += 8) {
    const int64_t r = r0 + k, c = c0 + tx;
    if (r < R && c < C) tile[k][tx] = x[r * C + c];
  }
  __syncthreads();
  for (int k = ty; k < 32; k += 8) {
    const int64_t c = c0 + k, r = r0 + tx;
    if (r < R && c < C) y[c * R + r] = tile[tx][k];
  }
}

unsigned grid_for(int64_t n, int per_thread, int nt = 256) {
  int64_t g = (n + (int64_t)nt * per_thread - 1) / ((int64_t)nt * per_thread);
  if (g < 1) g = 1;
  if (g > 65536) g = 65536;
  return (unsigned)g;
}

}  // namespace

namespace {
// Recognizes a single-op chain: LOAD x -> rx [, LOAD y -> ry], OP (operands among rx, ry) -> rd,
// STORE rd -> out[o], every operand full-shape and 16-byte aligned. Fills the operand order the
// op reads (a, b) and returns the op, or -1.
int pw_single_op(const PwParams& p, const float** a, const float** b, float** out, bool* binary) {
  auto aligned = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15u) == 0; };
  const int n = p.n_instr;
  if (n != 3 && n != 4) return -1;
  const int nl = n - 2;
  int reg[2];
  const float* src[2];
  for (int i = 0; i < nl; ++i) {
    const PwInstr& l = p.code[i];
    if (l.op != PW_LOAD) return -1;
    const int k = l.a % PW_MAX_INPUTS;
    if (p.in[k] == nullptr || p.in_mode[k] != 0 || !aligned(p.in[k])) return -1;
    reg[i] = l.dst & (PW_REGS - 1);
    src[i] = p.in[k];
  }
  if (nl == 2 && reg[0] == reg[1]) return -1;
  const PwInstr& op = p.code[nl];
  const PwInstr& st = p.code[nl + 1];
  if (st.op != PW_STORE || (st.a & (PW_REGS - 1)) != (op.dst & (PW_REGS - 1))) return -1;
  float* o = p.out[st.dst & 1];
  if (o == nullptr || !aligned(o)) return -1;
  auto which = [&](int r) -> const float* {
    for (int i = 0; i < nl; ++i)
      if (reg[i] == (r & (PW_REGS - 1))) return src[i];
    return nullptr;
  };
  const bool bin = op.op == PW_ADD || op.op == PW_SUB || op.op == PW_MUL || op.op == PW_DIV ||
                   op.op == PW_MAX || op.op == PW_GT || op.op == PW_RELU_GRAD ||
                   op.op == PW_TANH_GRAD || op.op == PW_SIGMOID_GRAD;
  const bool un = op.op == PW_NEG || op.op == PW_RELU || op.op == PW_TANH ||
                  op.op == PW_SIGMOID || op.op == PW_EXP || op.op == PW_LOG || op.op == PW_SQRT;
  if (!bin && !un) return -1;
  *a = which(op.a);
  *b = bin ? which(op.b) : *a;
  if (*a == nullptr || *b == nullptr) return -1;
  *out = o;
  *binary = bin;
  return op.op;
}

template <int OP>
void launch_single(const float* a, const float* b, float* out, int64_t n, bool bin, hipStream_t s) {
  const unsigned g = grid_for(n, 8);
  if (bin) hipLaunchKernelGGL((pw_single_kernel<OP, true>), dim3(g), dim3(256), 0, s, a, b, out, n);
  else hipLaunchKernelGGL((pw_single_kernel<OP, false>), dim3(g), dim3(256), 0, s, a, b, out, n);
}
}  // namespace

hipError_t launch_pointwise(const PwParams& p, hipStream_t s) {
  const int64_t n = p.R * p.C;
  if (n <= 0) return hipSuccess;
  const float *a, *b;
  float* out;
  bool bin;
  switch (pw_single_op(p, &a, &b, &out, &bin)) {
    case PW_ADD: launch_single<PW_ADD>(a, b, out, n, bin, s); break;
    case PW_SUB: launch_single<PW_SUB>(a, b, out, n, bin, s); break;
    case PW_MUL: launch_single<PW_MUL>(a, b, out, n, bin, s); break;
    case PW_DIV: launch_single<PW_DIV>(a, b, out, n, bin, s); break;
    case PW_MAX: launch_single<PW_MAX>(a, b, out, n, bin, s); break;
    case PW_GT: launch_single<PW_GT>(a, b, out, n, bin, s); break;
    case PW_RELU_GRAD: launch_single<PW_RELU_GRAD>(a, b, out, n, bin, s); break;
    case PW_TANH_GRAD: launch_single<PW_TANH_GRAD>(a, b, out, n, bin, s); break;
    case PW_SIGMOID_GRAD: launch_single<PW_SIGMOID_GRAD>(a, b, out, n, bin, s); break;
    case PW_NEG: launch_single<PW_NEG>(a, b, out, n, bin, s); break;
    case PW_RELU: launch_single<PW_RELU>(a, b, out, n, bin, s); break;
    case PW_TANH: launch_single<PW_TANH>(a, b, out, n, bin, s); break;
    case PW_SIGMOID: launch_single<PW_SIGMOID>(a, b, out, n, bin, s); break;
    case PW_EXP: launch_single<PW_EXP>(a, b, out, n, bin, s); break;
    case PW_LOG: launch_single<PW_LOG>(a, b, out, n, bin, s); break;
    case PW_SQRT: launch_single<PW_SQRT>(a, b, out, n, bin, s); break;
    default:
      PwArgs a{p, pw_divide(p.R * p.C, p.C)};
      bool bcast = false;
      for (int k = 0; k < PW_MAX_INPUTS; ++k)
        bcast |= p.in[k] != nullptr && (p.in_mode[k] == 1 || p.in_mode[k] == 2);
      int regs = 1;  // registers the chain names (every operand field is read, used or not)
      for (int i = 0; i < p.n_instr; ++i) {
        const PwInstr& c = p.code[i];
        for (int r : {(int)c.dst, (int)c.a, (int)c.b, (int)c.c})
          regs = std::max(regs, (r & (PW_REGS - 1)) + 1);
      }
      const size_t lds = (size_t)regs * PW_NT * sizeof(float4);
      const dim3 g(grid_for(n, 4)), nt(PW_NT);
      if (!bcast) hipLaunchKernelGGL((pointwise_kernel<false, false>), g, nt, lds, s, a);
      else if (a.div.narrow) hipLaunchKernelGGL((pointwise_kernel<true, false>), g, nt, lds, s, a);
      else hipLaunchKernelGGL((pointwise_kernel<true, true>), g, nt, lds, s, a);
  }
  return hipGetLastError();
}

hipError_t launch_transpose(const float* x, float* y, int64_t R, int64_t C, hipStream_t s) {
  if (R <= 0 || C <= 0) return hipSuccess;
  dim3 g((unsigned)((C + 31) / 32), (unsigned)((R + 31) / 32));
  hipLaunchKernelGGL(transpose_kernel, g, dim3(256), 0, s, x, y, R, C);
  return hipGetLastError();
}

hipError_t launch_fill(float* x, int64_t n, float value, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(fill_kernel, dim3(grid_for(n, 4)), dim3(256), 0, s, x, n, value);
  return hipGetLastError();
}
hipError_t launch_fill_u32(uint32_t* x, int64_t n, uint32_t value, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(fill_u32_kernel, dim3(grid_for(n, 4)), dim3(256), 0, s, x, n, value);
  return hipGetLastError();
}
hipError_t launch_copy(const float* src, float* dst, int64_t n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const bool aligned =
      ((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) & 15u) == 0;
  const int64_t n4 = aligned ? n / 4 : 0;
  if (n4 > 0) {
    const int64_t blocks = (n4 + 255) / 256;
    if (blocks > INT32_MAX) return hipErrorInvalidValue;
    hipLaunchKernelGGL(copy_vec_kernel, dim3((unsigned)blocks), dim3(256), 0, s,
                       reinterpret_cast<const float4*>(src), reinterpret_cast<float4*>(dst), n4);
  }
  const int64_t rest = n - 4 * n4;
  if (rest > 0)
    hipLaunchKernelGGL(copy_kernel, dim3(grid_for(rest, 4)), dim3(256), 0, s, src + 4 * n4,
                       dst + 4 * n4, rest);
  return hipGetLastError();
}

int64_t colsum_partial_doubles(int64_t R, int64_t N) {
  if (R <= 0 || N <= 0) return 0;
  const int64_t rows = colsum_rows_per_panel(R, N);
  return ((R + rows - 1) / rows) * N;
}
hipError_t launch_colsum(const float* x, float* out, int64_t R, int64_t N, int64_t ldx,
                         double divisor, int accumulate, double* partial, hipStream_t s) {
  if (N <= 0) return hipSuccess;
  if (N <= CS_SMALL_MAX_N && R <= CS_SMALL_MAX_R) {
    hipLaunchKernelGGL(colsum_small, dim3((unsigned)((N + CS_COLS - 1) / CS_COLS)), dim3(1024), 0,
                       s, x, out, R, N, ldx, divisor, accumulate);
    return hipGetLastError();
  }
  const int64_t rows = colsum_rows_per_panel(R, N);
  const int64_t P = (R + rows - 1) / rows;
  if (P > 0) {
    const bool aligned = N % 4 == 0 && ldx % 4 == 0 && (reinterpret_cast<uintptr_t>(x) & 15u) == 0;
    // (64 columns fill colsum_pass1's lanes: [1000000, 33] 120 us, 144 in fours)
    if (N > CS_COLS && (aligned || R > CS_FEW_UNALIGNED || (R > 4 && N > CS_FEW_COLS))) {
      dim3 g1((unsigned)((N + 4 * CS_COLS - 1) / (4 * CS_COLS)), (unsigned)P);
      // (sixteen waves of 2^30 and more columns are more threads than a grid dimension holds)
      if (R <= CS_FEW_ROWS || N >= (1ll << 30) - 4 * CS_COLS)
        hipLaunchKernelGGL(colsum_pass1_v4<4>, g1, dim3(256), 0, s, x, partial, R, N, ldx, rows);
      else
        hipLaunchKernelGGL(colsum_pass1_v4<16>, g1, dim3(1024), 0, s, x, partial, R, N, ldx, rows);
    } else {
      dim3 g1((unsigned)((N + CS_COLS - 1) / CS_COLS), (unsigned)P);
      hipLaunchKernelGGL(colsum_pass1, g1, dim3(256), 0, s, x, partial, R, N, ldx, rows);
    }
  }
  hipLaunchKernelGGL(colsum_pass2, dim3((unsigned)((N + CS_COLS - 1) / CS_COLS)), dim3(256), 0, s,
                     partial, out, P, N, N, divisor, accumulate);
  return hipGetLastError();
}

hipError_t launch_colsum_finish(double* partial, float* out, int64_t P, int64_t N,
                                hipStream_t s) {
  if (N <= 0) return hipSuccess;
  const unsigned x = (unsigned)((N + CS_COLS - 1) / CS_COLS);
  int64_t step = N;
  // a fold's workgroups beyond the grid's second dimension: one pass reads them all, as it did
  const int64_t chunks = (P + CS_FOLD_CHUNK - 1) / CS_FOLD_CHUNK;
  if (P > CS_FOLD_ROWS && chunks < 65536) {
    hipLaunchKernelGGL(colsum_fold, dim3(x, (unsigned)chunks), dim3(256), 0, s, partial, P, N);
    P = chunks;
    step = CS_FOLD_CHUNK * N;
  }
  hipLaunchKernelGGL(colsum_pass2, dim3(x), dim3(256), 0, s, (const double*)partial, out, P, N, step,
                     1.0, 0);
  return hipGetLastError();
}

hipError_t launch_row_reduce(const float* x, float* out, int64_t R, int64_t C, int kind,
                             hipStream_t s) {
  if (R <= 0) return hipSuccess;
  switch (kind) {
    case 0: launch_row_kind<0>(x, out, R, C, s); break;
    case 1: launch_row_kind<1>(x, out, R, C, s); break;
    case 2: launch_row_kind<2>(x, out, R, C, s); break;
    default: launch_row_kind<3>(x, out, R, C, s); break;
  }
  return hipGetLastError();
}

int64_t reduce_all_partial_doubles(int64_t) { return RA_BLOCKS; }
hipError_t launch_reduce_all(const float* x, float* out, int64_t n, int kind, double* partial,
                             hipStream_t s) {
  const unsigned g = (unsigned)std::min<int64_t>(RA_BLOCKS, std::max<int64_t>(1, (n + 1023) / 1024));
  hipLaunchKernelGGL(reduce_all_pass1, dim3(g), dim3(256), 0, s, x, n, kind, partial);
  hipLaunchKernelGGL(reduce_all_pass2, dim3(1), dim3(256), 0, s, (const double*)partial, (int)g, n,
                     kind, out);
  return hipGetLastError();
}

}  // namespace shk
