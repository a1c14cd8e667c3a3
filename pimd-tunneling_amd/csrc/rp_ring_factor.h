// rp_ring_factor.h -- block LDL^T of the ring Hessian on the matrix cores, ndof <= 32.
// Included by rp_ring.hip.
//
// The chain is eliminated from both ends toward its middle bead h = (n - 1) / 2, a wave per
// side: S_i = A_i - c^2 S_{i-1}^-1 for i < h, S'_i = A_i - c^2 S'_{i+1}^-1 for i > h, and
// S_h = A_h - c^2 S_{h-1}^-1 - c^2 S'_{h+1}^-1 (c = 1/betan^2; bead 0 is not coupled to bead 1,
// instantonmod.f90:203).  log|det| and the inertia are the sums over all blocks, in whatever
// order the beads are eliminated (Haynsworth).
//
// A block is inverted by the symmetric sweep operator, four pivots K at a time, in the
// registers of one wave: with P = M[K][K]^-1,
//   M[r][c] -= M[r][K] P M[K][c],  M[K][c] = P M[K][c],  M[r][K] = M[r][K] P,  M[K][K] = -P,
// and after every pivot M = -S^-1, which is what the next bead adds c^2 times.  M sits in
// RT x RT MFMA accumulator tiles: item j of lane (m, g) of tile (rt, ct) is row 16 rt + 4 j + g,
// column 16 ct + m.  Item j of the tiles of one row is then four consecutive rows, as the B
// operand of a 16x16x4 MFMA (k = g, column m), and by symmetry those four columns as an A
// operand: a pivot step moves no data, and the update is one MFMA per tile.  The pivot rows
// times P are another MFMA, whose A operand repeats P in every fourth row.
//
// No pivoting: the blocks' 2 x 2 leading minors are divided by in turn, so their signs give
// the inertia (Sylvester) and their product the determinant, kept as mantissa and exponent.
//
// Bound by the latency of a pivot step: ten lane reads, the 4 x 4 inverse with its two
// reciprocals, one MFMA for P M[K][.], then the update.  The 256 EVB instanton chains of 64 to
// 1024 beads (ndof 27), one factorisation each: 1.64 ms, and 3.4 ms for seven shifts of every
// chain, against 6.8 and 11.5 ms for a workgroup of 4 waves per chain that swept two pivots
// per barrier through LDS.  At 3 waves per SIMD the registers spill: 1.79 and 4.1 ms.
#pragma once

template <int RT>
__global__ void __launch_bounds__(128, 2) ring_factor_kernel(
    int D, const int* __restrict__ nn, const int64_t* __restrict__ boff,
    const double* __restrict__ betan, const double* __restrict__ massd,
    const double* __restrict__ blocks, const double* __restrict__ shift, double* __restrict__ sinv,
    double* __restrict__ logdet, int* __restrict__ nneg, const int* __restrict__ chain_of) {
  constexpr int DC = 16 * RT;
  __shared__ double wt[DC * DC];          // 1/sqrt(m_r m_c), zero in the padding
  __shared__ double other[RT * RT * 256];  // the far side's -S'^-1 next to the middle bead
  __shared__ double slg;
  __shared__ int sng;
  // one task per workgroup: chain c (task t of a chain_of map, else chain t) factored at
  // the shift of task t; outputs per task
  const int task = blockIdx.x, c = chain_of ? chain_of[task] : task;
  const int n = nn[c], tid = threadIdx.x, lane = tid & 63, m = lane & 15, g = lane >> 4;
  const int side = __builtin_amdgcn_readfirstlane(tid >> 6);  // 0: from bead 0, 1: from bead n-1
  const int h = (n - 1) >> 1, DD8 = D * D * 8;
  const double bn2 = betan[c] * betan[c], c2 = 1.0 / (bn2 * bn2);
  const double dv = 2.0 / bn2 - (shift ? shift[task] : 0.0);  // factor H - shift I
  for (int e = tid; e < DC * DC; e += 128) {
    const int r = e / DC, q = e - r * DC;
    wt[e] = r < D && q < D ? 1.0 / sqrt(massd[r] * massd[q]) : 0.0;
  }
  __syncthreads();
  const double* const chain = blocks + (size_t)boff[c] * D * D;
  int vo[RT][4], co[RT];  // byte offsets of the lane's rows and columns, clamped to the block
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    co[t] = min(16 * t + m, D - 1) * 8;
#pragma unroll
    for (int j = 0; j < 4; ++j) vo[t][j] = min(16 * t + 4 * j + g, D - 1) * D * 8;
  }
  d4 acc[RT][RT], nxt[RT][RT];
  // a buffer per block: a chain's blocks may take more than its 32-bit offsets reach
  auto load = [&](int bead) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t Bb = raw_buffer(chain + (size_t)bead * D * D, DD8);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < RT; ++ct)
#pragma unroll
        for (int j = 0; j < 4; ++j) nxt[rt][ct][j] = buffer_ld(Bb, vo[rt][j] + co[ct], 0);
  };
  double mant = 1.0;  // the determinant so far: mant 2^ex, and the negative pivots
  int ex = 0, neg = 0;
  // the lane's entry (q, g) of a 4 x 4 pivot block: unit factors that pick it out of the sums
  // below without a branch or a select
  const int q = m & 3;
  const double q0 = q == 0, q1 = q == 1, q2 = -(double)(q == 2), q3 = -(double)(q == 3);
  const double g0 = g == 0, g1 = g == 1, g2 = -(double)(g == 2), g3 = -(double)(g == 3);
  const double b00 = q0 * g0, b01 = -(q0 * g1 + q1 * g0), b11 = q1 * g1;

  // A_i + c2c acc -> acc
  auto form = [&](double c2c) __attribute__((always_inline)) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < RT; ++ct) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int r = 16 * rt + 4 * j + g;
          double a = nxt[rt][ct][j] * wt[r * DC + 16 * ct + m];
          if (rt == ct) a += m == 4 * j + g ? dv : 0.0;
          a = fma(c2c, acc[rt][ct][j], a);
          if (rt == ct && rt == RT - 1) a = r >= D ? (m == 4 * j + g ? 1.0 : 0.0) : a;  // padding
          acc[rt][ct][j] = a;
        }
      }
  };
  // negative pivots of a 2 x 2 minor with determinant det and leading entry a: one where det
  // is negative, else two or none with the sign of a
  auto negative = [](double det, double a) __attribute__((always_inline)) {
    const uint32_t sd = (uint32_t)__double2hiint(det) >> 31, sa = (uint32_t)__double2hiint(a) >> 31;
    return (int)(sd + ((sa & ~sd) << 1));
  };
  auto sweep = [&]() __attribute__((always_inline)) {
    const int before = neg;
    static_for<4 * RT>([&](auto Sx) __attribute__((always_inline)) {
      constexpr int s = decltype(Sx)::value, t = s / 4, j = s % 4;
      if (4 * s >= D) return;  // uniform
      double W[RT];
#pragma unroll
      for (int ct = 0; ct < RT; ++ct) W[ct] = acc[t][ct][j];
      auto at = [&](int a, int b) __attribute__((always_inline)) {
        return read_lane(W[t], 16 * a + 4 * j + b);
      };
      const double a00 = at(0, 0), a01 = at(0, 1), a11 = at(1, 1), a02 = at(0, 2), a03 = at(0, 3),
                   a12 = at(1, 2), a13 = at(1, 3), a22 = at(2, 2), a23 = at(2, 3), a33 = at(3, 3);
      // P by 2 x 2 blocks: A = [a00 a01; a01 a11], X = A^-1 B, S = C - B^T X
      const double dA = fma(a00, a11, -a01 * a01), iA = pivot_recip(dA);
      const double x00 = (a11 * a02 - a01 * a12) * iA, x01 = (a11 * a03 - a01 * a13) * iA;
      const double x10 = (a00 * a12 - a01 * a02) * iA, x11 = (a00 * a13 - a01 * a03) * iA;
      const double s00 = a22 - (a02 * x00 + a12 * x10), s01 = a23 - (a02 * x01 + a12 * x11);
      const double s11 = a33 - (a03 * x01 + a13 * x11);
      const double dS = fma(s00, s11, -s01 * s01), iS = pivot_recip(dS);
      const double t00 = s11 * iS, t01 = -s01 * iS, t11 = s00 * iS;
      neg += negative(dA, a00) + negative(dS, s00);
      mant = mant * dA * dS;
      ex += __builtin_amdgcn_frexp_exp(mant);
      mant = __builtin_amdgcn_frexp_mant(mant);
      // P = [A^-1 0; 0 0] + U S^-1 U^T with U = [X; -1]: the lane's entry (q, g)
      const double uq0 = fma(x00, q0, fma(x10, q1, q2)), uq1 = fma(x01, q0, fma(x11, q1, q3));
      const double ug0 = fma(x00, g0, fma(x10, g1, g2)), ug1 = fma(x01, g0, fma(x11, g1, g3));
      const double base = fma(a11, b00, fma(a01, b01, a00 * b11)) * iA;
      const double P = fma(uq0, fma(t00, ug0, t01 * ug1), fma(uq1, fma(t01, ug0, t11 * ug1), base));
      const bool pc = (m >> 2) == j;  // a pivot column of the tiles (., t)
      double pw[RT];                  // -P M[K][c], and +P in the pivot columns
#pragma unroll
      for (int ct = 0; ct < RT; ++ct) {
        const d4 zero = {0.0, 0.0, 0.0, 0.0};
        pw[ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(-P, W[ct], zero, 0, 0, 0)[0];
      }
      pw[t] = pc ? P : pw[t];
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) acc[rt][t][jj] = pc ? 0.0 : acc[rt][t][jj];
      constexpr int tn = (s + 1) / 4 < RT ? (s + 1) / 4 : 0;  // the next pivots' row tile first
#pragma unroll
      for (int rr = 0; rr < RT; ++rr)
#pragma unroll
        for (int cc = 0; cc < RT; ++cc) {
          const int rt = (rr + tn) % RT, ct = (cc + tn) % RT;
          acc[rt][ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(W[rt], pw[ct], acc[rt][ct], 0, 0, 0);
        }
#pragma unroll
      for (int ct = 0; ct < RT; ++ct) acc[t][ct][j] = -pw[ct];
    });
    // a block that is not finite counts none: the sign bits of its NaN pivots mean nothing, and
    // the determinant stays NaN from there.  Once per block: comparisons in place of the sign
    // bits take 2 to 4 % of the factorisation.
    neg = mant == mant ? neg : before;
  };
  // S_i^-1 for the block solves
  auto keep = [&](int bead) __attribute__((always_inline)) {
    if (!sinv) return;
    double* out = sinv + ((size_t)boff[c] + bead) * D * D;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < RT; ++ct)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int r = 16 * rt + 4 * j + g, k = 16 * ct + m;
          if (r < D && k < D) out[r * D + k] = -acc[rt][ct][j];
        }
  };

#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int ct = 0; ct < RT; ++ct) acc[rt][ct] = d4{0.0, 0.0, 0.0, 0.0};
  const int count = side ? n - 1 - h : h;  // beads of this side, without the middle one
  load(side ? n - 1 : 0);
  for (int k = 0; k < count; ++k) {
    const int i = side ? n - 1 - k : k;
    // beads i - 1 and i are coupled for i >= 2 (side 0), i and i + 1 for i >= 1 (side 1)
    form((side ? k > 0 : i >= 2) ? c2 : 0.0);
    load(side ? i - 1 : i + 1);  // in flight during the sweep; the last one is the middle bead
    sweep();
    keep(i);
  }
  if (side) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < RT; ++ct)
#pragma unroll
        for (int j = 0; j < 4; ++j) other[((rt * RT + ct) * 4 + j) * 64 + lane] = acc[rt][ct][j];
    if (lane == 0) {
      slg = log(fabs(mant)) + (double)ex * 0.69314718055994531;
      sng = neg;
    }
  }
  __syncthreads();
  if (side) return;
  form(h >= 2 ? c2 : 0.0);
  if (h >= 1 && h < n - 1) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < RT; ++ct)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int r = 16 * rt + 4 * j + g, k = 16 * ct + m;
          const double o = other[((rt * RT + ct) * 4 + j) * 64 + lane];
          acc[rt][ct][j] += r < D && k < D ? c2 * o : 0.0;
        }
  }
  sweep();
  keep(h);
  if (lane == 0) {
    logdet[task] = log(fabs(mant)) + (double)ex * 0.69314718055994531 + slg;
    nneg[task] = neg + sng;
  }
}
