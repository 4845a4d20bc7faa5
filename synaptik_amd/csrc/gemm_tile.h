// What the GEMM kernels share: the per-layout launch entry, compile-time loops, the optimizer update
// of one element and the workgroup-to-tile map.
//
// Replaces the reference's MATMUL routes for the Linear path:
//   forward  Z = X . W^T          (TensorLinearExpressions.java:97-146)        -> transB = 1
//   backward dX = dZ . W          (LinearAlgebraGradientRules.java:97-104)     -> NN
//   backward dW = PERMUTE(X^T.dZ) (LayoutGradientRules.java:114), written directly as
//            dW[out,in] = dZ^T . X                                             -> transA = 1
// The reference contract allows a backend to reassociate an operation's reduction and use
// FP32 FMA within one operation (docs/architecture/contracts/foundational-modules.md:423-425),
// which is what the matrix cores do; results differ from the sequential no-FMA CPU oracle only
// by reduction order (and are bit-identical when all partial sums are exact).
//
// Each operand layout (NN, NT, TN, TT) instantiates the kernels (gemm_v2.h, gemm_direct.h) in a
// translation unit of its own (gemm_nn.hip ... gemm_tt.hip); gemm.hip holds the dispatch, split-K
// and K == 1. Workgroup ids are remapped so that each of the 8 XCDs receives a contiguous,
// M-grouped block of output tiles: tiles that share A row-panels and B column-panels share an L2.
#pragma once
#include "common.h"
#include "kernels.h"
#include "optim_math.h"
#include <algorithm>
#include <cstdlib>
#include <type_traits>
#include <utility>

namespace shk {

// Partial rows the last fused-column-sum launch on this thread wrote.
extern thread_local int64_t g_colsum_rows;

// Launches an MFMA kernel for one operand layout (instantiated per layout).
//   va / vb: the A / B operand allows aligned float4 loads; p.kchunk > 0: split-K slices.
template <bool TA, bool TB>
hipError_t launch_layout(const GemmParams& p, bool va, bool vb, hipStream_t s);
extern template hipError_t launch_layout<false, false>(const GemmParams&, bool, bool, hipStream_t);
extern template hipError_t launch_layout<false, true>(const GemmParams&, bool, bool, hipStream_t);
extern template hipError_t launch_layout<true, false>(const GemmParams&, bool, bool, hipStream_t);
extern template hipError_t launch_layout<true, true>(const GemmParams&, bool, bool, hipStream_t);

namespace {

// Compile-time loop: f(std::integral_constant<int, I>) for I in [0, N). Keeps accumulator
// indexing static where a large #pragma unroll body would be left rolled (and the accumulator
// array demoted to scratch memory).
template <int... I, typename F>
__device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(std::make_integer_sequence<int, N>{}, f);
}

// Fused optimizer update of one element from its gradient g (GemmParams::upd): the candidate
// parameter and slots go to pn/mn/vn; returns false if an intermediate failed its check.
struct UpdateCtx {
  Coeffs k;
  bool first;
};
__device__ __forceinline__ UpdateCtx update_ctx(const GemmUpdate& u) {
  const int64_t completed = *u.completed_steps;
  UpdateCtx c;
  c.first = completed == 0;
  c.k = Coeffs{1.0f, 1.0f, 1.0f, true};
  if (u.kind != 0) c.k = adam_coeffs(u, completed + 1);
  return c;
}
__device__ __forceinline__ bool update_element(const GemmUpdate& u, const UpdateCtx& c,
                                               float pv, float g, float mv, float vv, int64_t e) {
  float pc, mc, vc = 0.0f, chk = 0.0f;
  if (u.kind == 0) sgd_element(u, c.first, pv, g, mv, pc, mc, chk);
  else adam_element(u, c.k, pv, g, mv, vv, pc, mc, vc, chk);
  const bool ok = chk == 0.0f;
  u.pn[e] = pc;
  if (u.mn != nullptr) u.mn[e] = mc;
  if (u.kind != 0) u.vn[e] = vc;
  return ok;
}
// Flags a failed update in the program status word (one atomic per wave).
__device__ __forceinline__ void update_flag(const GemmUpdate& u, const UpdateCtx& c, bool ok) {
  const int bad = wave_or(ok ? 0 : 1);
  if (bad && (threadIdx.x & 63) == 0)
    atomicOr(u.status, c.k.ok ? (uint32_t)DEV_NON_FINITE : (uint32_t)DEV_NOT_POSITIVE);
}
__device__ __forceinline__ bool update_scalar(const GemmUpdate& u, const UpdateCtx& c, int64_t e,
                                              float g) {
  const float mv = u.m != nullptr ? u.m[e] : 0.0f;
  const float vv = u.kind != 0 ? u.v[e] : 0.0f;
  return update_element(u, c, u.p[e], g, mv, vv, e);
}

// Maps the linear workgroup id to an output tile: XCD-contiguous, then grouped along M.
__device__ __forceinline__ void tile_of(int id, int tilesM, int tilesN, int& tm, int& tn) {
  const int total = tilesM * tilesN;
  if ((total & 7) == 0) id = (id & 7) * (total >> 3) + (id >> 3);
  constexpr int GROUP = 8;
  const int per_group = GROUP * tilesN;
  const int g = id / per_group;
  const int first = g * GROUP;
  const int gsize = min(tilesM - first, GROUP);
  const int in_group = id - g * per_group;
  tm = first + in_group % gsize;
  tn = in_group / gsize;
}

}  // namespace
}  // namespace shk
