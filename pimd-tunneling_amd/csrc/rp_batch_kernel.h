// rp_batch_kernel.h -- the fused persistent step kernel of the batched engine.
// Included by the per-potential instantiation units (rp_batch_k_*.hip).
#pragma once
#include "rp_batch.h"
#include "rp_evb_mfma.h"

namespace rp {

// inclusive sums over each row of 16 lanes, toward higher / lower lanes
__device__ __forceinline__ double row_prefix(double v) {
  v += row_mov0<kShr + 1>(v);
  v += row_mov0<kShr + 2>(v);
  v += row_mov0<kShr + 4>(v);
  v += row_mov0<kShr + 8>(v);
  return v;
}
__device__ __forceinline__ double row_suffix(double v) {
  v += row_mov0<kShl + 1>(v);
  v += row_mov0<kShl + 2>(v);
  v += row_mov0<kShl + 4>(v);
  v += row_mov0<kShl + 8>(v);
  return v;
}

__device__ __forceinline__ bool nonfinite(double v) { return !(fabs(v) < INFINITY); }

// The kernel's arguments in the constant segment they arrive in.  A phase reads them through
// an opaque copy of the segment's address (refresh), so they are scalar loads where they are
// used: as ordinary arguments the compiler kept all of them, and every lane's LDS addresses,
// in registers across the step loop, and spilled (160 SGPRs and, on the 27-dof EVB, 200
// VGPRs beyond the 256 of two waves per SIMD).
typedef const __attribute__((address_space(4))) BatchArgs KernArgs;

// One polymer group's place in the workgroup: pointers into LDS (batch_lds, rp_batch.h), the
// wave's half and tile, and the lane's bead.  The half h = 0 counts beads l = 0, 1, ... from
// the start of the chain, h = 1 from its end; both meet in the middle (the lower half has
// the middle bead of an odd chain).
struct Lane {
  double *Z, *E, *Tot, *Row, *Own;
  int N;               // beads of the chain
  int h, tile, nt;     // wave-uniform: the wave's half and bead tile, tiles per half
  int own;             // doubles of a wave's own area
  int wtid, wthreads;  // this thread among the group's threads
  int m, g;            // MFMA lane coordinates
  int l, bead;         // bead l of the half, bead N-1-l or l of the chain
  bool on, last;       // l is a bead of the half; its last one
};

// LDS place of normal `col` (row of the state) of mode 2 r + half.  The column's bit 4 is
// flipped on odd r: the four mode rows an MFMA operand load reads then fall in distinct banks.
template <int DC>
__device__ __forceinline__ int z_at(int HP, int half, int r, int col) {
  return (half * HP + r) * DC + (DC > 16 ? col ^ ((r & 1) << 4) : col);
}

// The normals of one O-step (or, `resample`, of a momentum resample: blocks of N in (dim
// outer, atom inner) order, verletmodule.f90:102-106, 211-215) into Z.  A thread makes the
// Philox blocks of one row: both normals of a block belong to consecutive modes.  Lanes run
// over the rows, so the LDS writes of a wave are consecutive.  N draws from position s take
// N/2 blocks when N and s are even (`whole`, in every row), else N/2 + 1.  PACK: cur counts
// from each polymer's own position.
template <int DC, bool PACK>
__device__ __forceinline__ void make_noise(KernArgs& A, const Lane& L, int R, int64_t cur,
                                           uint64_t strm, int64_t noff, bool whole,
                                           bool resample) {
  const int N = A.N, D = A.D, HP = 16 * L.nt;
  const int NB = whole ? N >> 1 : (N >> 1) + 1;
  int row = L.wtid % R, q = L.wtid / R;
  const int drow = L.wthreads % R, dq = L.wthreads / R;
  while (q < NB) {
    int d = row;
    int64_t c = cur;
    uint64_t st = strm;
    if constexpr (PACK) {
      const int pol = row / D;
      d = row - pol * D;
      const int64_t* ci = reinterpret_cast<const int64_t*>(L.Row + RW_CUR * DC);
      c = ci[pol] + cur;
      st = (uint64_t)ci[DC + pol];
    }
    const int blk = resample ? (d % A.ndim) * A.natom + d / A.ndim : d;
    const int64_t s = c + (int64_t)blk * N;
    const uint64_t b = (uint64_t)(s >> 1) + (uint64_t)q;
    const int i0 = (int)(2 * (int64_t)b - s), i1 = i0 + 1;  // -1 <= i0 <= N
    double z0, z1;
    if (A.noise) {
      z0 = (i0 >= 0 && i0 < N) ? A.noise[noff + s + i0] : 0.0;
      z1 = (i1 < N) ? A.noise[noff + s + i1] : 0.0;
    } else {
      philox_normal2(A.seed, st, b, z0, z1);
    }
    if (i0 >= 0 && i0 < N) L.Z[z_at<DC>(HP, i0 & 1, i0 >> 1, row)] = z0;
    if (i1 < N) L.Z[z_at<DC>(HP, i1 & 1, i1 >> 1, row)] = z1;
    row += drow;
    q += dq;
    if (row >= R) {
      row -= R;
      ++q;
    }
  }
}

// r = T (lambda z) for this wave's beads.  sin(i (N+1-l) pi/(N+1)) = -(-1)^i sin(i l pi/(N+1))
// splits the product into its odd modes P and even modes Q, half the multiply-adds: the lower
// half's beads get P + Q, the upper half's P - Q.  The two waves of a tile share that work:
// each makes P and Q of half the dof tiles (of one dof tile, the lower wave P and the upper
// Q) and hands over the other wave's part through LDS.  The tables carry the factor lambda_i;
// their fragments (L2) are loaded one K-chunk ahead of the MFMAs.
template <int DT>
__device__ __forceinline__ void noise_gemm(KernArgs& A, const Lane& L, double (&r)[DT][4]) {
  constexpr int DC = 16 * DT, ND = DT == 1 ? 1 : DT / 2, NQ = DT == 1 ? 1 : 2;
  const int HP = 16 * L.nt, lane = L.g * 16 + L.m;
  const double* __restrict__ T0 = A.Tf + (DT == 1 ? (size_t)L.h * HP * HP : 0);
  const int toff = L.g * HP + L.tile * 16 + L.m;
  // operand address of the first K-chunk: z_at's column swizzle is the same in every chunk
  const double* z0 = L.Z + z_at<DC>(HP, DT == 1 ? L.h : 0, L.g, (DT == 1 ? 0 : 16 * ND * L.h) + L.m);
  d4 acc[ND][NQ];
#pragma unroll
  for (int e = 0; e < ND; ++e)
#pragma unroll
    for (int q = 0; q < NQ; ++q) acc[e][q] = d4{0.0, 0.0, 0.0, 0.0};
  const int nk = HP >> 2;  // a multiple of 4
  double b[2][NQ];
  auto load = [&](int set, int kc) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) b[set][q] = (T0 + (size_t)(q * HP + 4 * kc) * HP)[toff];
  };
  auto mma = [&](int set, int kc) __attribute__((always_inline)) {
    const double* z = z0 + 4 * kc * DC;
#pragma unroll
    for (int e = 0; e < ND; ++e)
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        // dof tile 16 e further: bit 4 of the column flips with e when the swizzle is on
        const double* ze = z + q * HP * DC;
        const double a = ND == 1 ? ze[0] : ze[(L.g & 1) ? (e ^ 1) * 16 - 16 : e * 16];
        acc[e][q] = mfma_f64(a, b[set][q], acc[e][q]);
      }
  };
  load(0, 0);
  for (int kc = 0; kc < nk; kc += 2) {
    load(1, kc + 1);
    __builtin_amdgcn_sched_barrier(0);
    mma(0, kc);
    __builtin_amdgcn_sched_barrier(0);
    load(0, kc + 2 < nk ? kc + 2 : kc + 1);  // the last prefetch re-reads a valid chunk
    __builtin_amdgcn_sched_barrier(0);
    mma(1, kc + 1);
    __builtin_amdgcn_sched_barrier(0);
  }
  double* out = L.Own + lane;
  const double* in = L.Own + (L.h ? -L.own : L.own) + lane;  // the tile's other wave
#pragma unroll
  for (int e = 0; e < ND; ++e)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const double P = acc[e][0][j], Q = acc[e][NQ - 1][j];
      out[(e * 4 + j) * 64] = DT == 1 ? P : L.h ? P + Q : P - Q;
      r[e][j] = DT == 1 ? P : L.h ? P - Q : P + Q;
    }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < ND; ++e)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const double own = r[e][j], got = in[(e * 4 + j) * 64];
      if constexpr (DT == 1) {
        r[e][j] = L.h ? got - own : own + got;
      } else {
        r[e][j] = L.h ? got : own;
        r[ND + e][j] = L.h ? own : got;
      }
    }
}

// The same for one tile and dof tile, both halves, into the step's source R[half][row][bead]
// (kWide: helper waves)
template <int DT>
__device__ __forceinline__ void noise_gemm_to(KernArgs& A, const Lane& L, int tile, int dt, double* R) {
  constexpr int DC = 16 * DT;
  const int HP = 16 * L.nt;
  const double* __restrict__ T0 = A.Tf;
  const double* __restrict__ T1 = A.Tf + (size_t)HP * HP;
  const int toff = L.g * HP + tile * 16 + L.m;
  const double* z0 = L.Z + z_at<DC>(HP, 0, L.g, 16 * dt + L.m);
  const double* z1 = z0 + HP * DC;
  d4 P = {0.0, 0.0, 0.0, 0.0}, Q = P;
  for (int kc = 0; kc < HP >> 2; kc += 4) {  // HP/4 is a multiple of 4: four chunks' loads at once
    double b0[4], b1[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      b0[u] = (T0 + (size_t)(4 * (kc + u)) * HP)[toff];
      b1[u] = (T1 + (size_t)(4 * (kc + u)) * HP)[toff];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      P = mfma_f64(z0[4 * (kc + u) * DC], b0[u], P);
      Q = mfma_f64(z1[4 * (kc + u) * DC], b1[u], Q);
    }
  }
  double* r = R + (tile * 2 * DC + 16 * dt + L.g) * 16 + L.m;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    r[4 * j * 16] = P[j] + Q[j];
    r[(DC + 4 * j) * 16] = P[j] - Q[j];
  }
}

// The wave's edge beads, for the neighbours of the adjacent tiles: slot tile + 1 holds
// [lower m = 0 | lower m = 15 | upper m = 0 | upper m = 15]; slot 0 holds the fixed ends at
// the places of m = 15, slot nt + 1 each half's last bead, where the halves meet.
template <int DT>
__device__ __forceinline__ void publish_edges(const Lane& L, const double (&x)[DT][4]) {
  constexpr int DC = 16 * DT;
  auto put = [&](int slot) __attribute__((always_inline)) {
    double* e = L.E + slot * DC + L.g;
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int j = 0; j < 4; ++j) e[16 * d + 4 * j] = x[d][j];
  };
  if (L.m == 0 || L.m == 15) put((L.tile + 1) * 4 + 2 * L.h + (L.m == 15));
  if (L.last) put((L.nt + 1) * 4 + L.h);
}

// First part of the linear step (Linear, rp_batch.h): p', and x' without the other tiles'
// share of K^-1; the tile's sums go to Tot.  K^-1 in closed form, with k = 1..N the bead and
// G = N + 1:
//   (K^-1 u)_k = betan^2 / G [ (G - k) sum_{j<=k} j u_j + k sum_{j>k} (G - j) u_j ].
// With w = l + 1 the lower half's bead is k = w and the upper half's k = G - w, so each half
// takes a prefix sum of w u and a suffix sum of (G - w) u over its own beads, and the other
// half enters as one number, the total of its w u.  Every term enters with its own sign only:
// no difference of large partial sums.
template <int DT, bool NOISE>
__device__ __forceinline__ void linear_local(KernArgs& A, const Lane& L,
                                             const __attribute__((address_space(4))) Linear& C,
                                             double (&x)[DT][4], double (&p)[DT][4], const double (&r)[DT][4]) {
  constexpr int DC = 16 * DT;
  const double w = (double)(L.l + 1), v = (double)(L.N - L.l), wf = w * A.iG;
  const double* ea = L.E + (2 * L.h + 1) * DC + L.g;  // this half's fixed end
  const double* eb = L.E + (3 - 2 * L.h) * DC + L.g;  // the other one
  // Where a lane's row moves have no source: the bead before the tile (m = 0), the one after it
  // (m = 15), or, for the half's last bead, the other half's, which the lanes past it also hold
  // and so pass to a last bead with m < 15.  One read for every lane, and the tile's sums go out
  // once per dof tile: a branch per element leaves each element waiting for its own LDS reads
  // (8 steps of the 27-dof EVB: 44 polymers, N = 32, 63 us with branches, 57 without; 5632,
  // N = 128, 2.12 and 2.07 ms).
  const double* en = L.E + (L.m == 0               ? L.tile * 4 + 1 + 2 * L.h
                            : L.last || !L.on ? (L.nt + 1) * 4 + (L.h ^ 1)
                                                   : (L.tile + 2) * 4 + 2 * L.h) * DC + L.g;
  const double* Row = L.Row + L.g;
  double* tot = L.Tot + (L.tile * 2 + L.h) * DC * 2 + 2 * L.g + (L.m ? 0 : 1);
  static_for<DT>([&](auto Dx) __attribute__((always_inline)) {
    constexpr int d = decltype(Dx)::value;
    double sum[4];
    static_for<4>([&](auto J) __attribute__((always_inline)) {
      constexpr int j = decltype(J)::value, row = 16 * d + 4 * j;
      const double xi = x[d][j], pi = p[d][j];
      double ri = 0.0;
      if constexpr (NOISE) ri = Row[RW_SK * DC + row] * r[d][j];
      // neighbours l - 1 and l + 1; the halves meet at their last beads
      const double e = en[row];
      const double prev = row_mov<kShr + 1>(e, xi);
      const double next = row_mov<kShl + 1>(e, L.on ? xi : e);
      // K^-1 of the tile's own beads
      const double u = L.on ? (NOISE ? fma(C.cu, pi, ri) : pi) : 0.0;
      const double f = v * u;
      const double a = row_prefix(w * u), b = row_suffix(f);
      sum[j] = L.m ? a : b;  // prefix total in lane 15, suffix total in lane 0
      const double s = v * a + w * (b - f);
      const double xa = ea[row], xeq = xa + (eb[row] - xa) * wf;
      double xn = xeq + C.cy * (xi - xeq) + (C.gx * Row[RW_IM * DC + row]) * s;
      double pn = C.cp * pi - (C.ck * Row[RW_M * DC + row]) * ((xi - prev) + (xi - next));
      if constexpr (NOISE) pn += C.cr * ri;
      // computed here: sunk past the next element's they would hold its inputs
      asm volatile("" : "+v"(xn), "+v"(pn));
      x[d][j] = xn;
      p[d][j] = pn;
      if constexpr (j & 1) __builtin_amdgcn_sched_barrier(0);  // two elements at a time: bounded registers
    });
    if (L.m == 0 || L.m == 15)
#pragma unroll
      for (int j = 0; j < 4; ++j) tot[2 * (16 * d + 4 * j)] = sum[j];
  });
}

// Second part: the other tiles' share of K^-1.  Each wave sums the tiles' totals for its own
// place: prefix totals of the tiles before it, suffix totals of those after it plus the other
// half's total, one (row, kind) per lane, through a wave-private LDS area.
template <int DT>
__device__ __forceinline__ void linear_carry(KernArgs& A, const Lane& L,
                                             const __attribute__((address_space(4))) Linear& C,
                                             double (&x)[DT][4]) {
  constexpr int DC = 16 * DT;
  const int lane = L.g * 16 + L.m;
  double* car = L.Own;
#pragma unroll
  for (int q = 0; q < (DT + 1) / 2; ++q) {
    const int c = lane + 64 * q;  // of 2 DC columns (row, kind)
    if (c < 2 * DC) {
      double s = 0.0;
      for (int t = 0; t < L.nt; ++t) {
        const double* T = L.Tot + (2 * t + L.h) * DC * 2 + c;
        const double* To = L.Tot + (2 * t + (L.h ^ 1)) * DC * 2 + c;
        if (c & 1) {
          s += (t > L.tile ? T[0] : 0.0) + To[-1];  // suffix, and the other half's prefix total
        } else if (t < L.tile) {
          s += T[0];
        }
      }
      car[c] = s;
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  const double w = (double)(L.l + 1), v = (double)(L.N - L.l);
  const double* Row = L.Row + L.g;
  const double* k = car + 2 * L.g;
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int row = 16 * d + 4 * j;
      x[d][j] += (C.gx * Row[RW_IM * DC + row]) * (v * k[2 * row] + w * k[2 * row + 1]);
    }
}

// ---------------------------------------------------------------- the kick, p -= dt grad V
// (verletmodule.f90:565-585)

// The EVB (evb_gradient), 16 beads of a wave, from registers to registers.
template <int M, int DT>
__device__ __forceinline__ void evb_kick(const double* PL, const Lane& L, double dt, uint32_t moved,
                                         const double (&x)[DT][4], double (&p)[DT][4]) {
  d4 ag[DT];
  evb_gradient<M, DT>(PL, L.m, L.g, moved, -dt, x, ag);
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) p[d][jj] += ag[d][jj];
}

// Elementwise potentials, one state element at a time.  COUPLED2D pairs row 2 q (x) with row
// 2 q + 1 (y), which sits 16 lanes away.
template <int KIND, int DT>
__device__ __forceinline__ void simple_kick(KernArgs& A, const Lane& L,
                                            const double (&x)[DT][4], double (&p)[DT][4]) {
  constexpr int DC = 16 * DT;
  const double* dp = A.pes.dp;
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const double xi = x[d][j];
      double gr;
      if constexpr (KIND == PES_QUARTIC) {
        const double h = dp[0], x0 = dp[1], ix2 = 1.0 / (x0 * x0);
        gr = (xi * xi * ix2 - 1.0) * (4.0 * h) * xi * ix2;
      } else if constexpr (KIND == PES_HARMONIC) {
        const int row = 16 * d + L.g + 4 * j;
        gr = L.Row[RW_K * DC + row] * (xi - L.Row[RW_C * DC + row]);
      } else {
        static_assert(KIND == PES_COUPLED2D, "elementwise potentials only");
        const double V0 = dp[0], a = dp[1], mm = dp[2], om = dp[3], c = dp[4];
        const double ia2 = 1.0 / (a * a), mw2 = mm * om * om;
        const double xo = __shfl_xor(xi, 16);
        const bool isy = L.g & 1;
        const double x0 = isy ? xo : xi, x1 = isy ? xi : xo;
        const double s = x1 + c * x0 * x0, t = x0 * x0 * ia2 - 1.0;
        gr = isy ? mw2 * s : (4.0 * V0) * t * x0 * ia2 + mw2 * s * (2.0 * c) * x0;
      }
      p[d][j] -= gr * A.dt;
    }
}

// 1/sqrt(x), x > 0: the hardware estimate y (about 26 bits) and one third-order step on the
// residual 1 - x y^2, taken with the product's rounding error: within an ulp, in place of a
// division and a square root
__device__ __forceinline__ double rsqrt_ref(double x) {
  const double y = __builtin_amdgcn_rsq(x), t = x * y, tl = fma(x, y, -t);
  const double e = fma(-tl, y, fma(-t, y, 1.0));
  return fma(y * e, fma(e, 0.375, 0.5), y);
}

// The water cluster for the 16 beads of a wave, positions in the wave's own part of LDS: a
// lane takes bead m and, round by round, the atoms g, g + 4, ... for the terms with the other
// molecules (charges, and Lennard-Jones between oxygens; each pair is made by both of its
// atoms, but a lane holds one atom's three components: nothing spills), then the molecules
// g, g + 4 for the Morse bonds and the HOH bend.  The gradients of a lane's atoms stay in
// registers until the positions are done with, then replace them, so the kick needs no
// barrier.  (A thread per (bead, atom) that made its molecule's own terms three times over,
// between barriers: 15.9 ms per 8-step launch of 11,264 polymers of 6 molecules and 128
// beads; this 11.4.)  The terms are those of water_eval (rp_pes.h); X: [16][DX].
template <int NMOL, int DT>
__device__ __forceinline__ void water_kick(KernArgs& A, const Lane& L, double* X,
                                           const double (&x)[DT][4], double (&p)[DT][4]) {
  constexpr int NA = 3 * NMOL, D = 3 * NA, DX = water_stride(D), NR = (NA + 3) / 4;
  auto wave_sync = [] {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  double* xb = X + L.m * DX;
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int row = 16 * d + 4 * j + L.g;
      if (row < D) xb[row] = x[d][j];
    }
  wave_sync();
  const double* dp = A.pes.dp;
  double gp[NR][3];
  if constexpr (NMOL > 1) {
    const double eps = dp[5], sig2 = dp[6] * dp[6], q2 = dp[7] * dp[7];
    static_for<NR>([&](auto Rr) __attribute__((always_inline)) {
      constexpr int r = decltype(Rr)::value;
      const int i = min(4 * r + L.g, NA - 1), mol = i / 3;
      const bool oxy = i == 3 * mol;
      const double x0 = xb[3 * i], x1 = xb[3 * i + 1], x2 = xb[3 * i + 2];
      const double qo = oxy ? -4.0 * q2 : 2.0 * q2, qh = oxy ? 2.0 * q2 : -q2;  // -q_i q_O, -q_i q_H
      double g0 = 0.0, g1 = 0.0, g2 = 0.0;
#pragma unroll 1
      for (int k = 1; k < NMOL; ++k) {
        const int mj = mol + k < NMOL ? mol + k : mol + k - NMOL;
        const double* y = xb + 9 * mj;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const double d0 = x0 - y[3 * a], d1 = x1 - y[3 * a + 1], d2 = x2 - y[3 * a + 2];
          const double ir = rsqrt_ref(d0 * d0 + d1 * d1 + d2 * d2), ir2 = ir * ir;
          double f = (a ? qh : qo) * ir;  // r dE/dr
          if (a == 0) {
            const double s2 = sig2 * ir2, s6 = s2 * s2 * s2;
            const double lj = (24.0 * eps) * (s6 - 2.0 * s6 * s6);
            f += oxy ? lj : 0.0;
          }
          f *= ir2;
          g0 += f * d0;
          g1 += f * d1;
          g2 += f * d2;
        }
      }
      gp[r][0] = g0;
      gp[r][1] = g1;
      gp[r][2] = g2;
      __builtin_amdgcn_sched_barrier(0);
    });
  }
  constexpr int NM = (NMOL + 3) / 4;
  double gm[NM][9];
  const double De = dp[0], al = dp[1], re = dp[2], kb = dp[3], th0 = dp[4];
  static_for<NM>([&](auto Rr) __attribute__((always_inline)) {
    constexpr int r = decltype(Rr)::value;
    const double* xm = xb + 9 * min(4 * r + L.g, NMOL - 1);
    double u[2][3], rr[2], dEdr[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      double s = 0.0;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        u[h][d] = xm[3 * (h + 1) + d] - xm[d];
        s += u[h][d] * u[h][d];
      }
      rr[h] = sqrt(s);
      const double e = exp(-al * (rr[h] - re)), om = 1.0 - e;
      dEdr[h] = (2.0 * De * al) * om * e / rr[h];
    }
    const double dot = u[0][0] * u[1][0] + u[0][1] * u[1][1] + u[0][2] * u[1][2];
    const double ir01 = 1.0 / (rr[0] * rr[1]);
    const double cs = dot * ir01;
    const double dth = acos(cs) - th0;
    const double dEdc = -kb * dth / sqrt(1.0 - cs * cs);
    const double i00 = cs / (rr[0] * rr[0]), i11 = cs / (rr[1] * rr[1]);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double a = dEdr[0] * u[0][d] + dEdc * (u[1][d] * ir01 - i00 * u[0][d]);
      const double b = dEdr[1] * u[1][d] + dEdc * (u[0][d] * ir01 - i11 * u[1][d]);
      gm[r][d] = -(a + b);
      gm[r][3 + d] = a;
      gm[r][6 + d] = b;
    }
  });
  wave_sync();  // every lane has read the positions
  if constexpr (NMOL > 1) {
#pragma unroll
    for (int r = 0; r < NR; ++r)
      if (4 * r + L.g < NA)
#pragma unroll
        for (int d = 0; d < 3; ++d) xb[3 * (4 * r + L.g) + d] = gp[r][d];
    wave_sync();
  }
#pragma unroll
  for (int r = 0; r < NM; ++r)
    if (4 * r + L.g < NMOL)
#pragma unroll
      for (int d = 0; d < 9; ++d) {
        double* o = xb + 9 * (4 * r + L.g) + d;
        *o = (NMOL > 1 ? *o : 0.0) + gm[r][d];
      }
  wave_sync();
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int row = 16 * d + 4 * j + L.g;
      if (row < D) p[d][j] -= A.dt * xb[row];
    }
}

// ---------------------------------------------------------------- the step kernel
enum : int { kPile = 0, kLimit, kPack, kAndersen, kWide };

// One workgroup holds a.groups polymer groups of 2 nt waves each; a group is one polymer, or
// (PACK, at most 8 dofs) a.pack polymers side by side in the 16 rows of an MFMA tile.  The
// state x, p lives in registers in the MFMA accumulator layout for all nsteps steps: item
// (d, j) of lane (m, g) is row 16 d + g + 4 j (a dof, or PACK a polymer's dof) of bead
// l = 16 tile + m of the wave's half.
//
// Langevin (time_step_pile): kick, normals -> LDS | T (lambda z) | linear step | carries.
// Andersen (time_step_nm): [resample] A(dt/2), kick, A(dt/2).  Bars are barriers.
//
// MODE: kPile, kLimit (with dHdrlimit re-initialisations), kPack, kAndersen, or kWide: kPile for
// batches that leave most of the GPU idle, where a step's latency is what counts.  A.helpers
// more waves make the next step's normals while the polymer's own waves take the kick, and the
// next step's T (lambda z), into LDS, while those take the linear step.  us per 8-step launch of
// 44 polymers of the 27-dof EVB, without and with: N = 32 89 and 64, 64 94 and 70, 128 128 and
// 109 (57, 65 and 105 since linear_local lost its branches); where it stops paying stands at launch_batch_kind.
//
// FP64 MFMAs and FP64 vector instructions share one pipe (256 workgroups of 8 waves: MFMA
// alone 2.29 ms, as many FMAs alone 2.90 ms, both on different waves 5.29 ms), so the step's
// bound is the sum of both; the normals' integer rounds do overlap the kick's MFMAs, so half
// of the waves take the two in the other order.
template <int KIND, int MAXD, int DT, int MODE>
__global__ void __launch_bounds__(DT > 2 ? 512 : 1024, DT > 2 ? 2 : 4) batch_kernel(BatchArgs) {
  extern __shared__ double S[];
  constexpr int DC = DT * 16;
  constexpr bool LANGEVIN = MODE != kAndersen, PACK = MODE == kPack, WIDE = MODE == kWide;
  KernArgs* const args = (KernArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  const int tid = threadIdx.x;
  // wave-uniform values, in SGPRs
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nwave = 2 * batch_tiles(args->N);
  const int grp0 = WIDE ? 0 : wave / nwave, wave0 = wave - grp0 * nwave;  // kWide: helpers from nwave up
  // all that a lane's place needs of the arguments, in two SGPRs: no phase waits for a scalar
  // load before it can address LDS
  const int nbeads = args->N;
  const int nshared = batch_lds(nbeads, DT, KIND == PES_EVB ? evb_kick_lds_size(DC, args->moved) : 0,
                                KIND == PES_WATER ? args->D : 0).shared;
  const double* PL = S;  // EVB block (stage_evb_kick's layout), KIND == PES_EVB only
  // the lane's place, derived afresh from opaque copies in each phase of a step
  auto place = [&](KernArgs& A) __attribute__((always_inline)) -> Lane {
    int lane = tid & 63, grp = grp0, wv = wave0;
    asm volatile("" : "+v"(lane));
    asm volatile("" : "+s"(grp), "+s"(wv));
    int N = nbeads, shared = nshared;
    asm volatile("" : "+s"(N), "+s"(shared));
    const BatchLds B = batch_lds(N, DT, shared, KIND == PES_WATER ? MAXD : 0);
    Lane L;
    L.N = N;
    L.nt = batch_tiles(N);
    L.h = wv & 1;
    L.tile = wv >> 1;
    L.wthreads = L.nt * 128;
    L.wtid = wv * 64 + lane;
    L.m = lane & 15;
    L.g = lane >> 4;
    L.l = L.tile * 16 + L.m;
    L.bead = L.h ? N - 1 - L.l : L.l;
    const int nh = L.h ? N >> 1 : (N + 1) >> 1;  // beads of this half
    L.on = L.l < nh;
    L.last = L.l == nh - 1;
    double* base = S + B.shared + grp * B.group;
    L.Z = base;
    L.E = base + B.e;
    L.Tot = base + B.tot;
    L.Row = base + B.row;
    L.own = wave_lds(DT, KIND == PES_WATER ? MAXD : 0);
    L.Own = base + B.ex + wv * L.own;
    if (WIDE && wv >= 2 * L.nt) {  // a helper: no beads of its own
      L.wtid -= L.wthreads;
      L.wthreads = A.helpers * 64;
      L.on = L.last = false;
    }
    return L;
  };
  auto refresh = [&]() __attribute__((always_inline)) -> KernArgs& {
    KernArgs* a = args;
    asm volatile("" : "+s"(a));
    return *a;
  };
  // the group's polymers; a group past the family's last polymer repeats it without storing
  const int npk = PACK ? args->pack : 1;
  const int want = ((int)blockIdx.x * args->groups + grp0) * npk;
  const bool live = want < args->count;
  const int q0 = live ? want : args->count - 1;                // first polymer of the group
  const int npol = PACK ? min(npk, args->count - q0) : 1;
  const int poly = args->first + q0;
  const int R = PACK ? npol * args->D : args->D;               // rows in use
  const uint64_t strm = args->stream[poly];
  int64_t* const pi = args->pi64 + (size_t)poly * kPI64;
  const int64_t noff = pi[PI_NOISE_OFF];
  int64_t cur = PACK ? 0 : pi[PI_CURSOR];  // PACK: draws since the launch began
  bool whole = !(args->N & 1);
  for (int k = 0; k < npol; ++k) whole &= !(pi[(size_t)k * kPI64 + PI_CURSOR] & 1);
  auto each = [&](const Lane& L, auto&& f) __attribute__((always_inline)) {
    static_for<DT>([&](auto Dx) __attribute__((always_inline)) {
      static_for<4>([&](auto J) __attribute__((always_inline)) {
        constexpr int d = decltype(Dx)::value, j = decltype(J)::value;
        f(std::integral_constant<int, d>{}, std::integral_constant<int, j>{}, 16 * d + L.g + 4 * j);
      });
    });
  };
  // x column of a row in use, in the state's global memory
  auto state_of = [&](KernArgs& A, int row) __attribute__((always_inline)) -> double* {
    const int pol = PACK ? row / A.D : 0, d = row - pol * A.D;
    return A.state + A.pi64[(size_t)(poly + pol) * kPI64 + PI_STATE_OFF] + (size_t)d * A.N;
  };
  double x[DT][4], p[DT][4];
  {
    // staging: the EVB block, zeroed normals and edges, row tables; state -> registers
    KernArgs& A = refresh();
    const Lane L = place(A);
    const int N = A.N, D = A.D;
    if constexpr (KIND == PES_EVB) stage_evb_kick<MAXD, DT>(A.pes.dp, S, A.moved, tid, blockDim.x);
    const int ngrp = WIDE ? blockDim.x : L.wthreads;
    for (int e = WIDE ? tid : L.wtid; e < (int)(L.Tot - L.Z); e += ngrp) L.Z[e] = 0.0;  // Z and E
    __syncthreads();
    for (int row = WIDE ? tid : L.wtid; row < DC; row += ngrp) {
      const int pol = PACK ? row / D : 0, d = row - pol * D;
      const bool real = row < R;
      const double* pa = A.pdata + (size_t)(poly + (real ? pol : 0)) * 3 * DC;
      const double mass = real ? A.massd[d] : 1.0;
      L.Row[RW_M * DC + row] = mass;
      L.Row[RW_IM * DC + row] = 1.0 / mass;
      L.Row[RW_SK * DC + row] = real ? sqrt(mass) * A.kappa : 0.0;
      L.Row[RW_SV * DC + row] = real ? sqrt(mass) * A.stdev0 * A.tau : 0.0;
      L.Row[RW_MDB * DC + row] = real ? mass * pa[2 * DC + d] : 0.0;
      L.E[1 * DC + row] = real ? pa[d] : 0.0;       // fixed start a
      L.E[3 * DC + row] = real ? pa[DC + d] : 0.0;  // fixed end b
      if constexpr (KIND == PES_HARMONIC) {
        L.Row[RW_K * DC + row] = real ? A.pes.dp[d] : 0.0;
        L.Row[RW_C * DC + row] = real ? A.pes.dp[D + d] : 0.0;
      }
      if constexpr (PACK) {  // one entry per polymer
        int64_t* ci = reinterpret_cast<int64_t*>(L.Row + RW_CUR * DC);
        const int k = min(row, npol - 1);
        ci[row] = A.pi64[(size_t)(poly + k) * kPI64 + PI_CURSOR];
        ci[DC + row] = (int64_t)A.stream[poly + k];
      }
    }
    each(L, [&](auto Dx, auto J, int row) __attribute__((always_inline)) {
      constexpr int d = decltype(Dx)::value, j = decltype(J)::value;
      const bool real = row < R && L.on;
      const double* st = state_of(A, row < R ? row : 0) + (L.on ? L.bead : 0);
      x[d][j] = real ? st[0] : 0.0;
      p[d][j] = real ? st[(size_t)D * N] : 0.0;
    });
  }
  bool bad = false;
  auto check = [&]() __attribute__((always_inline)) {  // NaN or infinity in the real beads
    const Lane L = place(refresh());
    each(L, [&](auto Dx, auto J, int row) __attribute__((always_inline)) {
      constexpr int d = decltype(Dx)::value, j = decltype(J)::value;
      bad |= L.on && row < R && (nonfinite(x[d][j]) || nonfinite(p[d][j]));
    });
  };
  double tisum = 0.0;
  d4 tirow[DT];  // PACK: one running sum per row
#pragma unroll
  for (int d = 0; d < DT; ++d) tirow[d] = d4{0.0, 0.0, 0.0, 0.0};
  int64_t ticnt = 0, nre = 0;
  int64_t acount = 0, rkick = 0, kcur = 0;
  if constexpr (!LANGEVIN) {
    acount = pi[PI_ACOUNT];
    rkick = pi[PI_RKICK];
    kcur = pi[PI_KCURSOR];
  }
  const bool lead = wave0 == 1;  // the wave that holds bead N (upper half, l = 0): it keeps the TI sums
  const int64_t need = (int64_t)args->N * args->D;  // draws per O-step / resample / re-init

  auto kick = [&]() __attribute__((always_inline)) {
    KernArgs& A = refresh();
    const Lane L = place(A);
    if constexpr (KIND == PES_EVB) {
      evb_kick<MAXD, DT>(PL, L, A.dt, A.moved, x, p);
    } else if constexpr (KIND == PES_WATER) {
      water_kick<MAXD / 9, DT>(A, L, L.Own, x, p);
    } else {
      simple_kick<KIND, DT>(A, L, x, p);
    }
  };
  auto noise = [&](bool resample) __attribute__((always_inline)) {
    KernArgs& A = refresh();
    make_noise<DC, PACK>(A, place(A), R, cur, strm, noff, whole, resample);
  };
  // p = sqrt(1/betan) z sqrt(beadmass) in normal modes, transformed back (:102-115, 211-228)
  auto resample_p = [&]() __attribute__((always_inline)) {
    noise(true);
    KernArgs& A = refresh();
    const Lane L = place(A);
    __syncthreads();
    double r[DT][4];
    noise_gemm<DT>(A, L, r);
    each(L, [&](auto Dx, auto J, int row) __attribute__((always_inline)) {
      constexpr int d = decltype(Dx)::value, j = decltype(J)::value;
      p[d][j] = L.Row[RW_SV * DC + row] * r[d][j];
    });
    cur += need;
  };
  // the linear step: A(dt/2) O A(dt/2) with the normals in Z (AOA), or A(dt/2) alone
  auto linear = [&](auto AOA) __attribute__((always_inline)) {
    constexpr bool aoa = decltype(AOA)::value;
    {
      const Lane L = place(refresh());
      publish_edges<DT>(L, x);
      __syncthreads();
    }
    double r[DT][4];
    if constexpr (aoa) {
      KernArgs& A = refresh();
      noise_gemm<DT>(A, place(A), r);
    }
    {
      KernArgs& A = refresh();
      linear_local<DT, aoa>(A, place(A), aoa ? A.aoa : A.rot, x, p, r);
      __syncthreads();
    }
    KernArgs& A = refresh();
    linear_carry<DT>(A, place(A), aoa ? A.aoa : A.rot, x);
  };

  // kWide: R, after the row tables; the step after the current one's source
  double* const Rn = S + batch_lds(args->N, DT, KIND == PES_EVB ? evb_kick_lds_size(DC, args->moved) : 0,
                                   KIND == PES_WATER ? args->D : 0).wide();
  const int hw = WIDE ? wave - nwave : 0;  // helper number, negative in the polymer's own waves
  auto helper_gemm = [&]() __attribute__((always_inline)) {
    KernArgs& A = refresh();
    const Lane L = place(A);
    for (int u = hw; u < L.nt * DT; u += A.helpers) noise_gemm_to<DT>(A, L, u / DT, u % DT, Rn);
  };
  __syncthreads();
  if constexpr (WIDE) {  // the first step's source
    if (hw >= 0) noise(false);
    __syncthreads();
    if (hw >= 0) helper_gemm();
    __syncthreads();
  }
  bool stop = false;
  const int64_t step0 = args->step0p ? *args->step0p : args->step0;
#pragma unroll 1
  for (int s = 0; s < args->nsteps; ++s) {
    const int64_t ii = step0 + s + 1;  // the reference's step counter
    if constexpr (WIDE) {
      cur += need;
      double r[DT][4];
      if (hw >= 0) {
        if (s + 1 < args->nsteps) noise(false);
        __syncthreads();
        if (s + 1 < args->nsteps) helper_gemm();
        __syncthreads();
        continue;
      }
      kick();
      {
        const Lane L = place(refresh());
        const double* q = Rn + ((L.tile * 2 + L.h) * DC + L.g) * 16 + L.m;
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
          for (int j = 0; j < 4; ++j) r[d][j] = q[(16 * d + 4 * j) * 16];
        publish_edges<DT>(L, x);
        __syncthreads();
      }
      {
        KernArgs& A = refresh();
        linear_local<DT, true>(A, place(A), A.aoa, x, p, r);
        __syncthreads();
      }
      KernArgs& A = refresh();
      linear_carry<DT>(A, place(A), A.aoa, x);
    } else if constexpr (LANGEVIN) {
      KernArgs& A = refresh();
      if (A.noise && cur + need > A.noise_cap) {
        stop = true;
        break;
      }
#pragma unroll 1
      for (int k = 0; k < 2; ++k) {
        if ((k ^ (wave >> 2)) & 1)
          noise(false);
        else
          kick();
      }
      linear(std::true_type{});
      cur += need;
    } else {
      // propagate_pimd_nm (verletmodule.f90:202-234): Poisson-timed resample first
      KernArgs& A = refresh();
      auto interval = [&]() -> int64_t {
        const int64_t k = kcur++;
        return A.kicks ? A.kicks[pi[PI_KICK_OFF] + k]
                       : philox_poisson(A.seed, strm, k, (double)A.noutput);
      };
      if (rkick < 0) {
        if (A.kicks && kcur >= A.kick_cap) {
          stop = true;
          break;
        }
        rkick = interval();
      }
      acount = acount + 1;
      if (acount >= rkick) {
        if ((A.noise && cur + need > A.noise_cap) || (A.kicks && kcur >= A.kick_cap)) {
          stop = true;
          break;
        }
        resample_p();
        rkick = interval();
        acount = 0;
      }
      linear(std::false_type{});
      kick();
      linear(std::false_type{});
    }
    // TI estimator after the step (verletmodule.f90:397-410, 236-244): sum over dofs of
    // m (-x_N) db/dxi; bead N is the upper bead of l = 0 (the sum's order differs from the
    // reference's only in rounding)
    KernArgs& A = refresh();
    if (ii > A.imin) {
      const Lane L = place(A);
      if constexpr (PACK) {
        each(L, [&](auto Dx, auto J, int row) __attribute__((always_inline)) {
          constexpr int d = decltype(Dx)::value, j = decltype(J)::value;
          tirow[d][j] -= L.Row[RW_MDB * DC + row] * x[d][j];
        });
        ++ticnt;
      } else {
        double contr = 0.0;
        if (lead) {
          each(L, [&](auto Dx, auto J, int row) __attribute__((always_inline)) {
            constexpr int d = decltype(Dx)::value, j = decltype(J)::value;
            contr -= L.Row[RW_MDB * DC + row] * x[d][j];
          });
          contr = sum_groups(contr);
        }
        if constexpr (MODE == kLimit) {
          // dHdrlimit: a step whose term is too large is not counted and the path is
          // re-initialised (:398-408)
          int* flag = reinterpret_cast<int*>(L.Row + RW_FLAG * DC);
          if (lead && (tid & 63) == 0) *flag = fabs(contr) < A.limit ? 0 : 1;
          __syncthreads();
          if (!*flag) {
            tisum += contr;
            ++ticnt;
          } else {
            if (A.noise && cur + need > A.noise_cap) {
              stop = true;
              break;
            }
            ++nre;
            check();
            resample_p();
            // init_path positions: x_k = splint(path, (k-1) xi/(n-1)) (:40-48)
            const double xi = A.pf64[(size_t)poly * kPF64 + PF_XI];
            const double* lam = A.pathd;
            const int N = A.N, np = A.npath;
            each(L, [&](auto Dx, auto J, int row) __attribute__((always_inline)) {
              constexpr int d = decltype(Dx)::value, j = decltype(J)::value;
              if (row < A.D && L.on) {
                const double* yy = lam + np + (size_t)row * np;
                const double* y2 = lam + np * (1 + A.D) + (size_t)row * np;
                x[d][j] = splint_dev(lam, yy, y2, np, (double)L.bead * xi / (double)(N - 1));
              }
            });
          }
          __syncthreads();
        } else {
          tisum += contr;
          ++ticnt;
        }
      }
    }
  }
  if (WIDE && hw >= 0) return;
  check();
  if (!live) return;
  KernArgs& A = refresh();
  const Lane L = place(A);
  const int N = A.N, D = A.D;
  if (stop && L.wtid == 0) atomicOr(&A.flags[1], 1);
  if (bad) atomicOr(&A.flags[0], 1);
  // registers -> state
  each(L, [&](auto Dx, auto J, int row) __attribute__((always_inline)) {
    constexpr int d = decltype(Dx)::value, j = decltype(J)::value;
    if (row < R && L.on) {
      double* st = state_of(A, row) + L.bead;
      st[0] = x[d][j];
      st[(size_t)D * N] = p[d][j];
    }
  });
  if constexpr (PACK) {
    // each polymer's rows summed by one lane
    if (!lead) return;
    if (L.m == 0)
      each(L, [&](auto Dx, auto J, int row) __attribute__((always_inline)) {
        L.Z[row] = tirow[decltype(Dx)::value][decltype(J)::value];
      });
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int q = tid & 63;
    if (q < npol) {
      double t = 0.0;
      for (int d = 0; d < D; ++d) t += L.Z[q * D + d];
      A.pf64[(size_t)(poly + q) * kPF64 + PF_TISUM] += t;
      pi[(size_t)q * kPI64 + PI_TICNT] += ticnt;
      pi[(size_t)q * kPI64 + PI_CURSOR] += cur;
    }
  } else if (lead && (tid & 63) == 0) {
    A.pf64[(size_t)poly * kPF64 + PF_TISUM] += tisum;
    pi[PI_TICNT] += ticnt;
    pi[PI_NREINIT] += nre;
    pi[PI_CURSOR] = cur;
    if constexpr (!LANGEVIN) {
      pi[PI_ACOUNT] = acount;
      pi[PI_RKICK] = rkick;
      pi[PI_KCURSOR] = kcur;
    }
  }
}

// How a family is dealt to workgroups.  A polymer takes one wave per 16 beads of each half.
//  * PACK (Langevin without re-initialisation, at most 8 dofs): as many polymers share the 16
//    rows of a tile as fit, but no more than leaves a workgroup for every CU.
//  * Groups per workgroup, for plain Langevin, where every group of a workgroup runs the same
//    steps: the fewest that keep a CU busiest by the score below, or a.waves (set_launch) over
//    the tiles of a half; and no more than leaves a workgroup for every CU.  Otherwise one:
//    resamples and re-initialisations fall differently.
//  * kWide (plain Langevin, no wave budget set, few polymers): helper waves, one group.
template <int KIND, int MAXD, int DT>
int launch_batch_kind(const BatchArgs& a0, int thermostat, int npoly, hipStream_t s) {
  BatchArgs a = a0;
  const bool lang = thermostat == RP_THERMO_LANGEVIN, plain = lang && a.limit < 0.0 && !a.noise;
  const int nt = batch_tiles(a.N);
  a.count = npoly;
  a.pack = a.groups = 1;
  constexpr bool packs =
      DT == 1 && (KIND == PES_QUARTIC || KIND == PES_HARMONIC || KIND == PES_COUPLED2D);
  if (packs && plain && a.D <= 8)
    a.pack = std::max(1, std::min(16 / a.D, (npoly + a.ncu - 1) / a.ncu));
  const BatchLds B = batch_lds(a.N, DT, KIND == PES_EVB ? evb_kick_lds_size(DT * 16, a.moved) : 0,
                               KIND == PES_WATER ? a.D : 0);
  const int units = (npoly + a.pack - 1) / a.pack;
  // kWide: enough helpers for the transform's tiles and the normals, a wave per 64 blocks of
  // them, as far as a workgroup has waves left.  Both lines measured, us per 8-step launch
  // without and with: past one workgroup per CU the helpers only take the kick's time (264
  // polymers of the 27-dof EVB, N = 32: 91 and 113; 1012: 126 and 217); with fewer than half as
  // many helpers as tiles they are waited for (44 polymers, N = 160, 6 helpers for 10 tiles: 167
  // and 141; N = 192, 4 for 12: 176 and 180; 88 quartic, N = 224, 2 for 7: 92 and 120).
  const int free_waves = (DT > 2 ? 8 : 16) - 2 * nt, tiles = nt * DT;
  a.helpers = std::min(free_waves, std::max(tiles, (a.D * ((a.N >> 1) + 1) + 63) / 64));
  const size_t wide_lds = (B.wide() + (size_t)2 * 16 * nt * 16 * DT) * sizeof(double);
  const bool wide = plain && a.pack == 1 && !a.waves && units <= a.ncu &&
                    2 * a.helpers >= tiles && wide_lds <= kBatchLds;
  constexpr int kWaves = DT > 2 ? 8 : 16;  // of a workgroup (launch bound)
  auto go = [&](auto kern) -> int {
    auto lds_of = [&](int g) { return (B.shared + (size_t)g * B.group) * sizeof(double); };
    RP_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)std::min(kBatchLds, lds_of(kWaves))));
    if (plain) {
      const int most = std::min({kWaves / (2 * nt), (units + a.ncu - 1) / a.ncu,
                                 a.waves ? std::max(1, a.waves / nt) : kWaves});
      double best = 0.0;
      for (int g = 1; g <= most && lds_of(g) <= kBatchLds; ++g) {
        int per_cu = 0;
        const int w = 2 * nt * g;
        RP_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, w * 64, lds_of(g)));
        // waves of a CU, less where a workgroup is alone on it (nothing fills its barriers) and
        // where its waves do not divide over the four SIMDs.  Measured on the 27-dof EVB, ms
        // per 8-step launch of 5632 polymers: N = 32, 2 groups (3 workgroups, 12 waves) 0.52,
        // 7 groups (1 workgroup, 14 waves) 0.72; N = 96, 2 groups (1 workgroup, 12 waves) 1.74,
        // 1 group (2 workgroups of 6 waves) 2.03; N = 64, 2 groups (2 workgroups, 16 waves)
        // 1.00, 1 group (3 workgroups, 12 waves) 1.30
        const double score = per_cu * w * (per_cu > 1 ? 1.0 : 0.74) * (w % 4 ? 0.7 : 1.0);
        if (a.waves || score > best) {
          a.groups = g;
          best = score;
        }
      }
    }
    const size_t lds = lds_of(a.groups);
    RP_REQUIRE(lds <= kBatchLds, "batch: n=%d with %d dof needs %zu bytes of LDS", a.N, a.D, lds);
    kern<<<(units + a.groups - 1) / a.groups, nt * a.groups * 128, lds, s>>>(a);
    RP_HIP(hipGetLastError());
    return RP_OK;
  };
  if (!lang) return go(batch_kernel<KIND, MAXD, DT, kAndersen>);
  if constexpr (packs) {
    if (a.pack > 1) return go(batch_kernel<KIND, MAXD, DT, kPack>);
  }
  if (a.limit >= 0.0) return go(batch_kernel<KIND, MAXD, DT, kLimit>);
  if (wide) {
    auto kern = batch_kernel<KIND, MAXD, DT, kWide>;
    RP_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)wide_lds));
    kern<<<units, (2 * nt + a.helpers) * 64, wide_lds, s>>>(a);
    RP_HIP(hipGetLastError());
    return RP_OK;
  }
  return go(batch_kernel<KIND, MAXD, DT, kPile>);
}

}  // namespace rp
