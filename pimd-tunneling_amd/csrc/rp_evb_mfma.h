// rp_evb_mfma.h -- the EVB double well on the matrix cores, from registers, and the lane moves
// its callers share: the batched step kernel and the ring action.
#pragma once
#include <utility>

#include "rp_dispatch.h"
#include "rp_nm.h"

namespace rp {

// f(integral_constant<int, 0..N-1>) expanded at compile time: the state's register indices
// stay constants even where a loop body is too large for the unroller, so the state never
// falls back to scratch memory.
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

__device__ __forceinline__ d4 mfma_f64(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// DPP moves inside each row of 16 lanes; a lane without a source keeps `old`, or gets zero
template <int CTRL>
__device__ __forceinline__ double row_mov(double old, double v) {
  return __builtin_amdgcn_update_dpp(old, v, CTRL, 0xF, 0xF, false);
}
template <int CTRL>
__device__ __forceinline__ double row_mov0(double v) {
  return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xF, 0xF, true);
}
// The sum over the four lane groups of 16, in every lane: swaps of rows and of halves between
// two registers that hold the same value leave both addends in every lane (vector moves; a
// shuffle through LDS waits twice)
__device__ __forceinline__ double sum_groups(double v) {
  auto join = [](unsigned lo, unsigned hi) __attribute__((always_inline)) {
    return __hiloint2double((int)hi, (int)lo);
  };
  unsigned lo = __double2loint(v), hi = __double2hiint(v);
  auto l16 = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
  auto h16 = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
  v = join(l16[0], h16[0]) + join(l16[1], h16[1]);
  lo = __double2loint(v);
  hi = __double2hiint(v);
  auto l32 = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
  auto h32 = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
  return join(l32[0], h32[0]) + join(l32[1], h32[1]);
}
constexpr int kShr = 0x110, kShl = 0x100;  // row_shr:n, row_shl:n

// The EVB block as evb_gradient reads it from LDS, for DC = 16 DT padded
// dofs: [kappa, 0 | cA | cB | lam | cub (DC each) | WA (DC rows of stride DC + 1) | WB - WA],
// zero beyond the potential's own stride, so no operand load needs a clamp or a select.  The
// difference has columns up to the last dof tile in which the wells' permutation moves a dof
// (evb_moved), in rows of stride evb_diff_stride.
__host__ __device__ inline int evb_diff_stride(uint32_t moved) { return moved >> 4 ? 33 : 17; }
__host__ __device__ inline int evb_kick_lds_size(int DC, uint32_t moved) {
  return 2 + 4 * DC + DC * (DC + 1) + (moved ? DC * evb_diff_stride(moved) : 0);
}

// K-chunks of 4 dofs with a dof whose column differs between the wells, one bit each: those of
// an atom that the map does not send to itself, or that another atom (of a map which is no
// permutation) or no atom is sent to, as rp_pes_create inverts it
inline uint32_t evb_moved(const rp_pes* pes) {
  const int na = pes->natom, nd = pes->ndim;
  uint32_t moved = 0;
  for (int a = 0; a < na; ++a) {
    int from = -1;  // the last atom sent to a
    for (int k = 0; k < na; ++k)
      if (pes->ip[k] == a) from = k;
    if (from != a)
      for (int d = a * nd; d < (a + 1) * nd; ++d) moved |= 1u << (d / 4);
  }
  return moved;
}

// The EVB parameter block (evb_eval_at's layout, stride M) -> the kick's LDS layout
// (evb_kick_lds_size): vectors and matrices zero-padded to DC = 16 DT, matrix rows of
// stride DC + 1 (the y GEMM reads a column of 16 rows per lane group: an odd stride puts
// them in distinct banks).  The second matrix is the difference WtB - WtA: the wells differ by
// a permutation of atoms, so its columns are zero at every atom the permutation leaves (evb_moved).
template <int M, int DT>
__device__ __forceinline__ void stage_evb_kick(const double* __restrict__ dp, double* PL, uint32_t moved,
                                               int tid, int nthreads) {
  constexpr int DC = DT * 16, LW = DC + 1, NV = 2 + 4 * DC;
  const double* WA = dp + 1;
  const double* cA = WA + M * M;
  const double* WB = cA + M;
  const double* cB = WB + M * M;
  const double* lam = cB + M;
  const double* cub = lam + M;
  const int ld = evb_diff_stride(moved);
  for (int e = tid; e < evb_kick_lds_size(DC, moved); e += nthreads) {
    double v = 0.0;
    if (e == 0) {
      v = dp[0];
    } else if (e >= 2 && e < NV) {
      const int k = (e - 2) / DC, i = (e - 2) - k * DC;
      const double* vec = k == 0 ? cA : k == 1 ? cB : k == 2 ? lam : cub;
      if (i < M) v = vec[i];
    } else if (e >= NV) {
      const int f = e - NV, w = f >= DC * LW, r = f - w * (DC * LW);
      const int i = r / (w ? ld : LW), j = r - i * (w ? ld : LW);
      if (i < M && j < M) v = w ? WB[i * M + j] - WA[i * M + j] : WA[i * M + j];
    }
    PL[e] = v;
  }
}

// The EVB on the matrix cores, 16 beads of a wave, from registers to registers: returns the
// energy of bead m (in each of its four lanes) and puts scale dV/dx into ag.  Both wells'
// coordinates are y_A = WtA x - cA (one GEMM whose B operand is x as the state holds it: item
// j of dof tile d is dof 16 d + g + 4 j of bead m, the operand of K-chunk 4 d + j) and
// y_B = y_A + cA - cB + (WtB - WtA) x, over the K-chunks in `moved` only: those with a dof that
// the wells' permutation moves.  The mixed gradient is likewise
// WtA^T (wa hA + wb hB) + (WtB - WtA)^T wb hB, the second product for the dof tiles with a
// moved dof; its B operand is the first GEMMs' accumulators, scaled in place, and its result
// has the layout of x.  With two hydrogens exchanged (dofs 0-5 of 27) that is 39 MFMAs per 16
// beads; both wells in full take 56.  K-chunks beyond M are left out.  The per-bead well
// energies are reduced over the four lane groups (sum_groups).
template <int M, int DT>
__device__ __forceinline__ double evb_gradient(const double* PL, int m, int g, uint32_t moved,
                                               double scale, const double (&x)[DT][4],
                                               d4 (&ag)[DT]) {
  constexpr int DC = DT * 16, LW = DC + 1;
  const double kappa = PL[0];
  const double* cA = PL + 2 + g;
  const double* cB = cA + DC;
  const double* lam = cB + DC;
  const double* cub = lam + DC;
  const double* WA = PL + 2 + 4 * DC;
  const double* WD = WA + DC * LW;
  const int ld = evb_diff_stride(moved);
  d4 ya[DT], yb[DT];
#pragma unroll
  for (int r = 0; r < DT; ++r) ya[r] = d4{0.0, 0.0, 0.0, 0.0};
  static_for<4 * DT>([&](auto K) __attribute__((always_inline)) {
    constexpr int kc = decltype(K)::value;
    if constexpr (4 * kc < M) {
#pragma unroll
      for (int r = 0; r < DT; ++r)
        ya[r] = mfma_f64(WA[(r * 16 + m) * LW + 4 * kc + g], x[kc / 4][kc % 4], ya[r]);
    }
  });
#pragma unroll
  for (int r = 0; r < DT; ++r) yb[r] = ya[r];
  static_for<4 * DT>([&](auto K) __attribute__((always_inline)) {
    constexpr int kc = decltype(K)::value;
    if constexpr (4 * kc < M) {
      if ((moved >> kc) & 1) {  // wave-uniform
#pragma unroll
        for (int r = 0; r < DT; ++r)
          yb[r] = mfma_f64(WD[(r * 16 + m) * ld + 4 * kc + g], x[kc / 4][kc % 4], yb[r]);
      }
    }
  });
  // h = lam y + 3 c y^2 and the well energies, per bead m
  double va = 0.0, vb = 0.0;
#pragma unroll
  for (int r = 0; r < DT; ++r)
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      if (r * 16 + 4 * jj >= M) continue;  // padded rows
      const int i = r * 16 + 4 * jj;
      const double li = lam[i], ci = cub[i];
      auto well = [&](double y, double& v, double& h) __attribute__((always_inline)) {
        const double t = ci * y;
        v += (y * y) * fma(0.5, li, t);
        h = y * fma(3.0, t, li);
      };
      double ha, hb;
      well(ya[r][jj] - cA[i], va, ha);
      well(yb[r][jj] - cB[i], vb, hb);
      ya[r][jj] = ha;
      yb[r][jj] = hb;
    }
  va = sum_groups(va);
  vb = sum_groups(vb);
  const double dl = va - vb, R = sqrt(0.25 * dl * dl + kappa * kappa), f = dl / (4.0 * R);
  const double wa = scale * (0.5 - f), wb = scale * (0.5 + f);
#pragma unroll
  for (int r = 0; r < DT; ++r) {
    yb[r] *= wb;
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) ya[r][jj] = fma(wa, ya[r][jj], yb[r][jj]);
  }
#pragma unroll
  for (int d = 0; d < DT; ++d) ag[d] = d4{0.0, 0.0, 0.0, 0.0};
  static_for<4 * DT>([&](auto K) __attribute__((always_inline)) {
    constexpr int kc = decltype(K)::value;
    if constexpr (4 * kc < M) {
#pragma unroll
      for (int d = 0; d < DT; ++d)
        ag[d] = mfma_f64(WA[(4 * kc + g) * LW + d * 16 + m], ya[kc / 4][kc % 4], ag[d]);
    }
  });
#pragma unroll
  for (int d = 0; d < DT; ++d)
    if ((moved >> (4 * d)) & 15u) {  // wave-uniform
      static_for<4 * DT>([&](auto K) __attribute__((always_inline)) {
        constexpr int kc = decltype(K)::value;
        if constexpr (4 * kc < M)
          ag[d] = mfma_f64(WD[(4 * kc + g) * ld + d * 16 + m], yb[kc / 4][kc % 4], ag[d]);
      });
    }
  return 0.5 * (va + vb) - R;
}

// W x of both wells on the matrix cores, 16 beads of a wave: y_A = WtA x is one GEMM whose B
// operand is x as the state holds it (item j of dof tile d is dof 16 d + g + 4 j of bead m, the
// operand of K-chunk 4 d + j), and y_B = y_A + (WtB - WtA) x, over the K-chunks in `moved` only:
// those with a dof that the wells' permutation moves.  K-chunks beyond M are left out.
// (evb_gradient holds this and evb_back in its own body: by way of these functions the step
// kernel for small batches spills 12 VGPRs, 49 -> 52 us per 8 steps of 44 polymers, N = 32.)
template <int M, int DT>
__device__ __forceinline__ void evb_modes(const double* WA, const double* WD, int ld, int m, int g,
                                          uint32_t moved, const double (&x)[DT][4], d4 (&ya)[DT],
                                          d4 (&yb)[DT]) {
  constexpr int LW = 16 * DT + 1;
#pragma unroll
  for (int r = 0; r < DT; ++r) ya[r] = d4{0.0, 0.0, 0.0, 0.0};
  static_for<4 * DT>([&](auto K) __attribute__((always_inline)) {
    constexpr int kc = decltype(K)::value;
    if constexpr (4 * kc < M) {
#pragma unroll
      for (int r = 0; r < DT; ++r)
        ya[r] = mfma_f64(WA[(r * 16 + m) * LW + 4 * kc + g], x[kc / 4][kc % 4], ya[r]);
    }
  });
#pragma unroll
  for (int r = 0; r < DT; ++r) yb[r] = ya[r];
  static_for<4 * DT>([&](auto K) __attribute__((always_inline)) {
    constexpr int kc = decltype(K)::value;
    if constexpr (4 * kc < M) {
      if ((moved >> kc) & 1) {  // wave-uniform
#pragma unroll
        for (int r = 0; r < DT; ++r)
          yb[r] = mfma_f64(WD[(r * 16 + m) * ld + 4 * kc + g], x[kc / 4][kc % 4], yb[r]);
      }
    }
  });
}

// ag = WtA^T u + (WtB - WtA)^T w, the second product for the dof tiles with a moved dof: B
// operands in the accumulator layout of evb_modes, the result in the layout of x
template <int M, int DT>
__device__ __forceinline__ void evb_back(const double* WA, const double* WD, int ld, int m, int g,
                                         uint32_t moved, const d4 (&u)[DT], const d4 (&w)[DT],
                                         d4 (&ag)[DT]) {
  constexpr int LW = 16 * DT + 1;
#pragma unroll
  for (int d = 0; d < DT; ++d) ag[d] = d4{0.0, 0.0, 0.0, 0.0};
  static_for<4 * DT>([&](auto K) __attribute__((always_inline)) {
    constexpr int kc = decltype(K)::value;
    if constexpr (4 * kc < M) {
#pragma unroll
      for (int d = 0; d < DT; ++d)
        ag[d] = mfma_f64(WA[(4 * kc + g) * LW + d * 16 + m], u[kc / 4][kc % 4], ag[d]);
    }
  });
#pragma unroll
  for (int d = 0; d < DT; ++d)
    if ((moved >> (4 * d)) & 15u) {  // wave-uniform
      static_for<4 * DT>([&](auto K) __attribute__((always_inline)) {
        constexpr int kc = decltype(K)::value;
        if constexpr (4 * kc < M)
          ag[d] = mfma_f64(WD[(4 * kc + g) * ld + d * 16 + m], w[kc / 4][kc % 4], ag[d]);
      });
    }
}

}  // namespace rp
