// fp32 MFMA GEMM straight from memory to registers, for gfx950: the problems with too few tiles
// for the direct-to-LDS kernel (gemm_v2.h), and the few with more that it does not take
// (direct_wide).
//
// Such a problem is bound by latency: a 128 x 1024 x 512 product is 1 us of matrix work. A wave
// owns a WT x WT tile (WT = 16 NB) as NB x NB blocks of v_mfma_f32_16x16x4_f32 and loads its operand
// fragments from global memory itself, 16 bytes a lane at any float: no LDS stage and no barrier
// in the main loop, D steps of loads in flight from the start, and the K groups of a workgroup
// (KW) each walk their own part of K, so that a 32 x 32 tile has eight waves' loads in flight. The
// register-staged kernel before it had one 16-deep k-tile of one workgroup in flight, on 128 x 128
// tiles split along K with a reduction pass. us on MI355X, before and after (NT unless said):
//   128x1024x512 19.7 -> 7.9; 64x4096x1024 24.3 -> 11.6; 500x509x1021 (odd) 29.1 -> 12.2;
//   500x101x509 23.9 -> 7.2; 100x300x700 21.4 -> 7.8; NN 500x509x101 10.6 -> 5.1;
//   TN 64x512x128 9.5 -> 5.2.
// Waves of a workgroup that share rows of A or columns of B load them twice; the second load hits
// the CU's L1.
//
// Configurations <NB, MW, NW, KW> (tile 16 NB MW x 16 NB NW, MW x NW x KW waves): <2, 2, 2, 2>
// 64 x 64, K in two groups; <2, 1, 1, 8> 32 x 32, K in eight. direct_wide chooses.
//
// Fragments (as gemm_v2.h): MFMA s of a 16-deep step takes k = 4 g + s from lane group g = lane / 16
// for both operands. A K-contiguous operand's lane loads four k of row 16 b + l16 (one vector per
// block b); an M/N-contiguous operand's lane loads the NB adjacent rows NB l16 .. at one k (one
// vector per s), its blocks interleaved by row. Rows beyond the operand are clamped into it and
// their results dropped; the last step of K is loaded element by element with zeros beyond K.
//
// Epilogue: the accumulators are staged in LDS (16-byte chunks XOR-swizzled by row), the K groups'
// partial tiles added in group order, and every global access of the epilogue is a 16-byte segment
// of a row. Reduction order: k within a step is permuted as above, steps in order within a K
// group, then the groups in order (a fixed order; foundational-modules.md:423-425 allows it).
#pragma once
#include "gemm_tile.h"

namespace shk {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float float2u __attribute__((ext_vector_type(2), aligned(4)));

constexpr int DK = 16;  // depth of a step
// Tiles in the grid's first dimension, which holds fewer than 2^32 threads; the rest go to planes
// along z.
constexpr uint32_t DIRECT_GRID_X = 1 << 20;

// One operand's fragments of a wave tile.
template <bool KMAJ, int NB>
struct DirectOperand {
  const float* p[KMAJ ? NB : 1];
  int64_t ld, row0, rows;
  bool edge;  // M/N-contiguous: the wave tile runs past the operand (wave-uniform)
  __device__ __forceinline__ void init(const float* base, int64_t ld_, int64_t r0, int64_t R) {
    const int l16 = threadIdx.x & 15, g = (threadIdx.x >> 4) & 3;
    ld = ld_;
    rows = R;
    edge = r0 + 16 * NB > R;
    if constexpr (KMAJ) {
      row0 = r0;
#pragma unroll
      for (int b = 0; b < NB; ++b) p[b] = base + min(r0 + 16 * b + l16, R - 1) * ld + 4 * g;
    } else {
      row0 = r0 + NB * l16;
      p[0] = base + 4 * g * ld;
    }
  }
  // The step [k, k + 16), all of it inside K.
  __device__ __forceinline__ void load(floatx4 (&f)[NB], int64_t k) const {
    if constexpr (KMAJ) {
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const float4u v = *reinterpret_cast<const float4u*>(p[b] + k);
        f[b] = floatx4{v[0], v[1], v[2], v[3]};
      }
    } else {
      // the step's offset is opaque, or the compiler keeps a pointer of its own for every load of
      // the unrolled steps (some 60 registers, and spills)
      int64_t step = k * ld;
      asm volatile("" : "+s"(step));
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const float* src = p[0] + step + s * ld;
        if (!edge) {
          static_assert(NB == 2, "two adjacent rows a lane");
          const float2u v = *reinterpret_cast<const float2u*>(src + row0);
          f[0][s] = v[0];
          f[1][s] = v[1];
        } else {
#pragma unroll
          for (int b = 0; b < NB; ++b) f[b][s] = src[min(row0 + b, rows - 1)];
        }
      }
    }
  }
  // The step that starts at k < ke and runs past ke: zeros from ke on.
  __device__ __forceinline__ void load_last(floatx4 (&f)[NB], int64_t k, int64_t ke) const {
    const int g = (threadIdx.x >> 4) & 3;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const bool in = k + 4 * g + s < ke;
      const int64_t ks = in ? k + s : ke - 1 - 4 * g;  // (relative to this lane's group)
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const float v = KMAJ ? p[KMAJ ? b : 0][ks] : p[0][ks * ld + min(row0 + b, rows - 1)];
        f[b][s] = in ? v : 0.0f;
      }
    }
  }
};

template <int NB, int MW, int NW, int KW>
struct DirectCfg {
  static constexpr int WT = 16 * NB, TM = WT * MW, TN = WT * NW;
  static constexpr int NT = 64 * MW * NW * KW;
  static constexpr int D = 4;                      // steps in flight
  static constexpr int CH = TN / 4;                // 16-byte chunks per tile row
  static constexpr int SW = (CH < 16 ? CH : 16) - 1;
  static constexpr int RP = NT / CH;               // rows per epilogue pass
  static constexpr int T = TM > RP ? TM / RP : 1;  // epilogue passes
  static constexpr int EC = T < 4 ? T : 4;         // passes whose loads go out together
};

// PLANES: the tiles beyond DIRECT_GRID_X lie in further planes of the grid (of their own, because
// the test costs a product of a million short rows 1%).
template <bool KA, bool KB, int NB, int MW, int NW, int KW, bool PLANES>
__global__ void __launch_bounds__(64 * MW * NW * KW) __attribute__((amdgpu_waves_per_eu(2)))
gemm_direct(GemmParams p) {
  using Cfg = DirectCfg<NB, MW, NW, KW>;
  constexpr int WT = Cfg::WT, TM = Cfg::TM, TN = Cfg::TN, D = Cfg::D, CH = Cfg::CH, SW = Cfg::SW;
  __shared__ __attribute__((aligned(16))) float stage[KW * TM * TN];

  const int tilesM = (int)((p.M + TM - 1) / TM), tilesN = (int)((p.N + TN - 1) / TN);
  const int id = (int)(blockIdx.x + (PLANES ? blockIdx.z * DIRECT_GRID_X : 0u));
  if (PLANES && id >= tilesM * tilesN) return;  // the last plane ends short
  int tm, tn;
  tile_of(id, tilesM, tilesN, tm, tn);
  const int64_t m0 = (int64_t)tm * TM, n0 = (int64_t)tn * TN;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int kw = wave / (MW * NW), wm = (wave / NW) % MW, wn = wave % NW;
  const int l16 = threadIdx.x & 15, g = (threadIdx.x >> 4) & 3;

  // K range of this workgroup (split-K slice) and of this wave's K group, in whole steps
  const int64_t k_begin = p.kchunk > 0 ? (int64_t)blockIdx.y * p.kchunk : 0;
  const int64_t k_end = p.kchunk > 0 ? min(p.K, k_begin + p.kchunk) : p.K;
  const int64_t steps = k_end > k_begin ? (k_end - k_begin + DK - 1) / DK : 0;
  const int64_t per = (steps + KW - 1) / KW;
  const int64_t s0 = min(steps, kw * per);
  int64_t s1 = min(steps, s0 + per);
  const int64_t rm = m0 + wm * WT, rn = n0 + wn * WT;
  if (rm >= p.M || rn >= p.N) s1 = s0;  // a wave tile beyond the result
  const int64_t kb = k_begin + s0 * DK;
  const int64_t whole = min(s1, (k_end - k_begin) / DK);
  const int nfull = (int)(whole > s0 ? whole - s0 : 0);

  floatx4 acc[NB][NB];
  static_for<NB>([&](auto i) {
    static_for<NB>([&](auto j) {
      acc[decltype(i)::value][decltype(j)::value] = floatx4{0.f, 0.f, 0.f, 0.f};
    });
  });
  auto mfma_step = [&](const floatx4 (&fa)[NB], const floatx4 (&fb)[NB])
      __attribute__((always_inline)) {
    static_for<4>([&](auto sc) {
      constexpr int S = decltype(sc)::value;
      static_for<NB * NB>([&](auto n) {
        constexpr int N = decltype(n)::value;
        // consecutive MFMAs share their first operand
        constexpr int I = KB ? N % NB : N / NB, J = KB ? N / NB : N % NB;
        if constexpr (KB)
          acc[I][J] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[J][S], fa[I][S], acc[I][J], 0, 0, 0);
        else
          acc[I][J] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[I][S], fb[J][S], acc[I][J], 0, 0, 0);
      });
    });
  };

  if (s1 > s0) {
    DirectOperand<KA, NB> A;
    DirectOperand<KB, NB> B;
    A.init(p.A, p.lda, rm, p.M);
    B.init(p.B, p.ldb, rn, p.N);
    floatx4 fa[D][NB], fb[D][NB];
    static_for<D>([&](auto jc) __attribute__((always_inline)) {
      constexpr int J = decltype(jc)::value;
      if (J < nfull) {
        A.load(fa[J], kb + J * DK);
        B.load(fb[J], kb + J * DK);
      }
    });
    int t = 0;
    for (; t + 2 * D <= nfull; t += D) {
      static_for<D>([&](auto jc) __attribute__((always_inline)) {
        constexpr int J = decltype(jc)::value;
        mfma_step(fa[J], fb[J]);
        __builtin_amdgcn_sched_barrier(0);
        A.load(fa[J], kb + (int64_t)(t + J + D) * DK);
        B.load(fb[J], kb + (int64_t)(t + J + D) * DK);
        __builtin_amdgcn_sched_barrier(0);
      });
    }
    // fewer than 2 D steps left, D of them in flight
    static_for<2 * D - 1>([&](auto jc) __attribute__((always_inline)) {
      constexpr int J = decltype(jc)::value;
      if (t + J < nfull) {
        mfma_step(fa[J % D], fb[J % D]);
        if (J + D < 2 * D - 1 && t + J + D < nfull) {
          A.load(fa[J % D], kb + (int64_t)(t + J + D) * DK);
          B.load(fb[J % D], kb + (int64_t)(t + J + D) * DK);
        }
      }
    });
    if (nfull < s1 - s0) {
      A.load_last(fa[0], kb + (int64_t)nfull * DK, k_end);
      B.load_last(fb[0], kb + (int64_t)nfull * DK, k_end);
      mfma_step(fa[0], fb[0]);
    }
  }

  // Stage: with a K-contiguous B the operands go into the MFMA swapped, and a lane holds four
  // consecutive columns of one row; otherwise NB adjacent columns of four rows.
  {
    float* st = stage + kw * (TM * TN);
    auto at = [&](int row, int col) {
      const int r = wm * WT + row, c = wn * WT + col;
      return st + r * TN + (((c >> 2) ^ (r & SW)) << 2) + (c & 3);
    };
    if constexpr (KB) {
      static_for<NB>([&](auto i) {
        static_for<NB>([&](auto j) {
          constexpr int I = decltype(i)::value, J = decltype(j)::value;
          *reinterpret_cast<floatx4*>(at(KA ? 16 * I + l16 : NB * l16 + I, 16 * J + 4 * g)) =
              acc[I][J];
        });
      });
    } else {
      static_for<NB>([&](auto i) {
        static_for<4>([&](auto r) {
          constexpr int I = decltype(i)::value, R = decltype(r)::value;
          float* dst = at(KA ? 16 * I + 4 * g + R : NB * (4 * g + R) + I, NB * l16);
          typedef float floatx2 __attribute__((ext_vector_type(2)));
          *reinterpret_cast<floatx2*>(dst) = floatx2{acc[I][0][R], acc[I][1][R]};
        });
      });
    }
  }
  __syncthreads();

  constexpr int RP = Cfg::RP, T = Cfg::T, EC = Cfg::EC;
  const int q = threadIdx.x % CH, r0 = threadIdx.x / CH;
  const int64_t col = n0 + 4 * q;
  const int cols = (int)min<int64_t>(4, p.N - col);  // columns of this lane's segments (<= 0: none)
  auto row_of = [&](int t) { return m0 + r0 + RP * t; };
  auto live = [&](int t) { return cols > 0 && r0 + RP * t < TM && row_of(t) < p.M; };
  auto sum_of = [&](int t) -> floatx4 {
    const int r = r0 + RP * t;
    const float* s = stage + r * TN + ((q ^ (r & SW)) << 2);
    floatx4 v = *reinterpret_cast<const floatx4*>(s);
#pragma unroll
    for (int w = 1; w < KW; ++w) {
      const floatx4 u = *reinterpret_cast<const floatx4*>(s + w * (TM * TN));
      v = floatx4{v[0] + u[0], v[1] + u[1], v[2] + u[2], v[3] + u[3]};
    }
    return v;
  };
  auto seg_load = [&](const float* src) -> floatx4 {
    if (cols >= 4) {
      const float4u v = *reinterpret_cast<const float4u*>(src);
      return floatx4{v[0], v[1], v[2], v[3]};
    }
    floatx4 v = floatx4{0.f, 0.f, 0.f, 0.f};
    if (cols > 0) v[0] = src[0];
    if (cols > 1) v[1] = src[1];
    if (cols > 2) v[2] = src[2];
    return v;
  };
  auto seg_store = [&](float* dst, const floatx4& v) {
    if (cols >= 4) {
      *reinterpret_cast<float4u*>(dst) = float4u{v[0], v[1], v[2], v[3]};
      return;
    }
    if (cols > 0) dst[0] = v[0];
    if (cols > 1) dst[1] = v[1];
    if (cols > 2) dst[2] = v[2];
  };
  const floatx4 zero = floatx4{0.f, 0.f, 0.f, 0.f};

  if (p.partial != nullptr) {  // split-K slice: reduced by gemm_splitk_reduce
    float* part = p.partial + (int64_t)blockIdx.y * p.M * p.N;
    for (int t = 0; t < T; ++t)
      if (live(t)) seg_store(part + row_of(t) * p.N + col, sum_of(t));
    return;
  }
  if (p.upd.pn != nullptr) {
    const GemmUpdate& u = p.upd;
    const UpdateCtx uc = update_ctx(u);
    bool ok = uc.k.ok;
    float chk = 0.0f;
    auto update_rows = [&](auto kindc) {
      constexpr bool SGD = decltype(kindc)::value == 0;
      for (int t0 = 0; t0 < T; t0 += EC) {
        floatx4 pv[EC], mv[EC], vv[EC];
        static_for<EC>([&](auto ic) {
          constexpr int I = decltype(ic)::value;
          const bool in = live(t0 + I);
          const int64_t e = row_of(t0 + I) * p.N + col;
          pv[I] = in ? seg_load(u.p + e) : zero;
          mv[I] = in && u.m != nullptr ? seg_load(u.m + e) : zero;
          vv[I] = !SGD && in ? seg_load(u.v + e) : zero;
        });
        static_for<EC>([&](auto ic) {
          constexpr int I = decltype(ic)::value;
          if (!live(t0 + I)) return;
          const int64_t e = row_of(t0 + I) * p.N + col;
          const floatx4 gv = sum_of(t0 + I);
          floatx4 pc, mc, vc = zero;
          static_for<4>([&](auto c) {
            constexpr int C = decltype(c)::value;
            float pe, me, ve = 0.0f, ce = 0.0f;
            if constexpr (SGD) sgd_element(u, uc.first, pv[I][C], gv[C], mv[I][C], pe, me, ce);
            else adam_element(u, uc.k, pv[I][C], gv[C], mv[I][C], vv[I][C], pe, me, ve, ce);
            if (C < cols) chk += ce;  // +0, or NaN once a check failed
            pc[C] = pe;
            mc[C] = me;
            vc[C] = ve;
          });
          seg_store(u.pn + e, pc);
          if (u.mn != nullptr) seg_store(u.mn + e, mc);
          if constexpr (!SGD) seg_store(u.vn + e, vc);
        });
      }
    };
    if (u.kind == 0) update_rows(std::integral_constant<int, 0>{});
    else update_rows(std::integral_constant<int, 1>{});
    update_flag(u, uc, ok && chk == 0.0f);
    return;
  }
  const bool has_bias = p.bias != nullptr;
  const floatx4 bias = has_bias && cols > 0 ? seg_load(p.bias + col) : zero;
  double cs[4] = {0.0, 0.0, 0.0, 0.0};
  auto store_rows = [&](auto modec, auto actc) {
    constexpr int MODE = decltype(modec)::value, ACT = decltype(actc)::value;
    for (int t0 = 0; t0 < T; t0 += EC) {
      floatx4 ya[EC], old[EC];
      static_for<EC>([&](auto ic) {
        constexpr int I = decltype(ic)::value;
        const bool in = live(t0 + I);
        ya[I] = MODE != 0 && in ? seg_load(p.aux + row_of(t0 + I) * p.ldaux + col) : zero;
        old[I] = p.accumulate && in ? seg_load(p.C + row_of(t0 + I) * p.ldc + col) : zero;
      });
      static_for<EC>([&](auto ic) {
        constexpr int I = decltype(ic)::value;
        if (!live(t0 + I)) return;
        const int64_t row = row_of(t0 + I);
        floatx4 v = sum_of(t0 + I);
        static_for<4>([&](auto c) {
          constexpr int C = decltype(c)::value;
          if constexpr (MODE != 1) {
            if (has_bias) v[C] = v[C] + bias[C];
            v[C] = apply_act(ACT, v[C]);
          } else {
            v[C] = act_grad(ACT, v[C], ya[I][C]);
          }
          if (p.accumulate) v[C] = old[I][C] + v[C];
        });
        seg_store(p.C + row * p.ldc + col, v);
        if constexpr (MODE == 2) {
          static_for<4>([&](auto c) {
            constexpr int C = decltype(c)::value;
            v[C] = act_grad(ACT, ya[I][C], v[C]);
          });
          seg_store(p.dz + row * p.ldaux + col, v);
        }
        static_for<4>([&](auto c) { cs[decltype(c)::value] += (double)v[decltype(c)::value]; });
      });
    }
  };
  auto by_act = [&](auto modec) {
    switch (p.act) {
      case ACT_RELU: store_rows(modec, std::integral_constant<int, ACT_RELU>{}); break;
      case ACT_TANH: store_rows(modec, std::integral_constant<int, ACT_TANH>{}); break;
      case ACT_SIGMOID: store_rows(modec, std::integral_constant<int, ACT_SIGMOID>{}); break;
      default: store_rows(modec, std::integral_constant<int, ACT_NONE>{}); break;
    }
  };
  if (p.mode == 0) by_act(std::integral_constant<int, 0>{});
  else if (p.mode == 1) by_act(std::integral_constant<int, 1>{});
  else by_act(std::integral_constant<int, 2>{});
  if (p.colsum_partial != nullptr) {
    // one binary64 partial row per tile row: the lanes' sums added over the row phases in order
    static_assert(KW * TM * TN * 4 >= RP * TN * 8, "the stage holds the phases' sums");
    double* red = reinterpret_cast<double*>(stage);
    __syncthreads();  // the staged tile has been read
    static_for<4>([&](auto c) {
      red[r0 * TN + 4 * q + decltype(c)::value] = cs[decltype(c)::value];
    });
    __syncthreads();
    for (int c = threadIdx.x; c < TN; c += Cfg::NT) {
      if (n0 + c >= p.N) continue;
      double s = 0.0;
      for (int r = 0; r < RP; ++r) s += red[r * TN + c];
      p.colsum_partial[(int64_t)tm * p.N + n0 + c] = s;
    }
  }
}

template <int NB, int MW, int NW, int KW, bool PLANES, bool TA, bool TB>
hipError_t launch_direct_cfg(const GemmParams& p, hipStream_t s) {
  using Cfg = DirectCfg<NB, MW, NW, KW>;
  const int64_t tm = (p.M + Cfg::TM - 1) / Cfg::TM, tn = (p.N + Cfg::TN - 1) / Cfg::TN;
  const int64_t slices = p.kchunk > 0 ? (p.K + p.kchunk - 1) / p.kchunk : 1;
  g_colsum_rows = tm;
  const int64_t x = PLANES ? DIRECT_GRID_X : tm * tn;
  hipLaunchKernelGGL((gemm_direct<!TA, TB, NB, MW, NW, KW, PLANES>),
                     dim3((unsigned)x, (unsigned)slices, (unsigned)((tm * tn + x - 1) / x)),
                     dim3(Cfg::NT), 0, s, p);
  return hipGetLastError();
}

// 64x64 tiles once they give every CU a workgroup, 32x32 below. Problems with that many tiles come
// here where gemm_v2.h refuses them: unaligned products of 17 to 32 rows or columns (whole calls:
// 200001x25x33 NN 39.3 us on 64x64 tiles, 48.9 on 32x32; 200001x25x200 78.6 and 79.5; TN
// 200001x25x33 52.9 and 62.1; fewer tiles 8200x19x300 NN 22.0 and 19.9), or of 33 to 63 with little K
// (30001x63x33 NN 19.6 and 25.0); leading dimensions beyond its offsets; K < 4.
inline bool direct_wide(const GemmParams& p) {
  const int64_t slices = p.kchunk > 0 ? (p.K + p.kchunk - 1) / p.kchunk : 1;
  return ((p.M + 63) / 64) * ((p.N + 63) / 64) * slices >= 256;
}

template <bool TA, bool TB>
hipError_t launch_direct(const GemmParams& p, hipStream_t s) {
  if (!direct_wide(p)) return launch_direct_cfg<2, 1, 1, 8, false, TA, TB>(p, s);
  return ((p.M + 63) / 64) * ((p.N + 63) / 64) <= DIRECT_GRID_X
             ? launch_direct_cfg<2, 2, 2, 2, false, TA, TB>(p, s)
             : launch_direct_cfg<2, 2, 2, 2, true, TA, TB>(p, s);
}

}  // namespace
}  // namespace shk
