// rp_batch.h -- device side of the batched engine.
//
// Every normal mode of the reference's chain has the same frequency 1/tau (beadmass =
// m (lam tau)^2, verletmodule.f90:315, 519).  The exact rotation of mode i by h is then
//   q' = c q + s_q p~ / (m lam_i^2),  p~' = -s_p m lam_i^2 q + c p~
// with (c, s_q, s_p) = (cos(h/tau), sin(h/tau)/tau, tau sin(h/tau)) or the Cayley map's
// counterparts, and the transform T diagonalises K = tridiag(-1, 2, -1) / betan^2 into
// lam_i^2.  So in bead space, with y = x - xeq (xeq the straight line between the fixed ends,
// which is what beadvec transforms to), the rotation needs no transform at all:
//   y' = c y + s_q K^-1 p / m,  p' = -s_p m K y + c p,
// a three-point stencil and a solve with K in closed form, O(N) per dof.  The O-step scales
// every mode by the same c1^2 and adds sqrt(m) kappa lam_i z_i, so A O A is one such linear
// step with T (lam z) as its source: one transform, of the noise alone, where the mode-space
// form has two of x and p.  (c1 = exp(-gamma dt / tau), kappa = tau c2 sqrt((1+c1^2)/betan).)
// Its rounding error against the reference's dense transforms in exact arithmetic is below
// the mode-space form's: x and p are not rounded through two sums of N terms per step.
//
// The state x, p stays in registers (rp_batch_kernel.h) for a block of K steps; LDS holds the
// step's normals, the tiles' edge beads and sums, and the potential's parameters.
#pragma once
#include "rp_dispatch.h"
#include "rp_evb_mfma.h"
#include "rp_nm.h"
#include "rp_philox.h"

namespace rp {

// Per-polymer 64-bit fields (BatchArgs::pi64[poly * kPI64 + field])
enum : int { PI_STATE_OFF = 0, PI_CURSOR, PI_TICNT, PI_NREINIT, PI_KCURSOR, PI_NOISE_OFF,
             PI_KICK_OFF, PI_ACOUNT, PI_RKICK, kPI64 };
// Per-polymer doubles (BatchArgs::pf64[poly * kPF64 + field])
enum : int { PF_TISUM = 0, PF_XI, kPF64 };
// Row tables of a polymer group in LDS (DC doubles each): mass, 1/mass, the O-step's and the
// resample's momentum scales, m db/dxi, harmonic k and centre; PACK: stream positions and ids
// (64-bit integers); the re-initialisation flag
enum : int { RW_M = 0, RW_IM, RW_SK, RW_MDB, RW_SV, RW_FLAG, RW_K, RW_C, kRW,
             RW_CUR = RW_SV /* PACK, and its next row: no resamples, no flag there */ };

// Scalars of a linear step in (y, p) with y = x - xeq:
//   y' = cy y + gx K^-1 (cu p + r) / m,   p' = cp p - ck m K y + cr r,
// K = tridiag(-1, 2, -1) / betan^2 between the fixed ends; gx is stored times betan^2/(N+1)
// and ck over betan^2, the closed forms' factors.  A(h) alone: cy = cp = c, cu = 1,
// gx = s_q, ck = s_p, r = 0.  A(h) O A(h), with r = sqrt(m) kappa T (lambda z):
//   cu = c (1 + c1^2), cy = c^2 - s_q s_p c1^2, cp = c^2 c1^2 - s_p s_q, ck = s_p c (1 + c1^2),
//   cr = c.
struct Linear {
  double cy, gx, cu, cp, ck, cr;
};

struct BatchArgs {
  PesDev pes;
  int N, NPAD, D, ndim, natom;
  int first, count;   // polymers (batch order) of this launch's family
  int groups, pack;   // polymer groups per workgroup, polymers per group (launch_batch_kind)
  int ncu;            // compute units of the device
  int helpers;        // kWide: helper waves
  uint32_t moved;     // EVB: K-chunks of 4 dofs with a dof that the wells' permutation moves
  int nsteps;
  int64_t step0, imin;
  const int64_t* step0p;        // step counter in device memory (graph replays), else nullptr
  double dt, limit, stdev0;
  Linear rot, aoa;              // A(dt/2), and A(dt/2) O A(dt/2)
  double kappa, tau, iG;        // the O-step's scale, and 1/(N+1)
  int64_t noutput;
  uint64_t seed;
  double* state;                // per polymer [x: D*N][p: D*N]
  int64_t* pi64;                // per polymer 64-bit fields
  double* pf64;                 // per polymer doubles
  const uint64_t* stream;       // per polymer Philox stream id
  const double* T;              // NPAD*NPAD, zero padded (init_path)
  const double* Tf;             // T lam in two halves [odd|even modes][HP modes][HP beads]
  const double* lam;            // per mode, zero padded (init_path)
  const double* pdata;          // per polymer [a | b | dbdl], DC each, zero padded
  const double* massd;          // per dof mass, DC, padded with 1
  const double* noise;          // injected draws or nullptr
  int64_t noise_cap;
  const int32_t* kicks;         // injected Poisson draws or nullptr
  int64_t kick_cap;
  int waves;                    // wave budget of a workgroup (2, 4 or 8); 0: by occupancy
  int npath;
  const double* pathd;          // [lampath (npath) | path (D*npath) | y2 (D*npath)]
  int* flags;                   // [0] NaN, [1] injected draws exhausted
};

int launch_batch_simple(const rp_pes* pes, const BatchArgs& a, int thermostat, int npoly,
                        hipStream_t s);
int launch_batch_evb(const rp_pes* pes, const BatchArgs& a, int thermostat, int npoly,
                     hipStream_t s);
int launch_batch_water(const rp_pes* pes, const BatchArgs& a, int thermostat, int npoly,
                       hipStream_t s);

inline int batch_dtiles(const rp_pes* pes) {
  const int D = pes->ndof;
  if (pes->kind == PES_WATER) return pes->natom == 3 ? 1 : pes->natom == 6 ? 2 : 4;
  if (pes->kind == PES_COUPLED2D || D <= 16) return 1;
  return 2;
}

// Doubles per bead of the water cluster's positions in LDS
__host__ __device__ constexpr int water_stride(int D) { return D | 1; }

// Bead tiles of each half of a polymer, 16 beads each
__host__ __device__ inline int batch_tiles(int n) { return (((n + 1) >> 1) + 15) >> 4; }

__host__ __device__ constexpr int wave_lds(int dt_tiles, int water_d) {
  const int ex = 256 * (dt_tiles > 1 ? dt_tiles / 2 : 1);
  const int wx = water_d ? (16 * water_stride(water_d) + 1) & ~1 : 0;
  return ex > wx ? ex : wx;  // at least the carries' 32 dt_tiles
}

// LDS of a workgroup, in doubles: the shared parameters, then `group` per polymer group, at
// these offsets in it: normals Z (0), edge beads e, tile sums tot, the waves' own areas ex, row
// tables.  A wave's own area (wave_lds doubles) holds in turn the water cluster's positions in
// the kick, the noise transform's exchange, read by the other wave of the tile between two
// barriers, and the carries.
struct BatchLds {
  int shared, group, e, tot, ex, row;
  // kWide: the next step's source, after one group: 2 nt tiles x DC rows x 16 beads
  __host__ __device__ int wide() const { return shared + group; }
};
__host__ __device__ inline BatchLds batch_lds(int n, int dt_tiles, int pes_lds, int water_d) {
  const int DC = 16 * dt_tiles, nt = batch_tiles(n), HP = 16 * nt;
  BatchLds B;
  B.shared = (pes_lds + 1) & ~1;
  B.e = 2 * HP * DC;
  B.tot = B.e + (nt + 2) * 4 * DC;
  B.ex = B.tot + nt * DC * 4;
  B.row = B.ex + 2 * nt * wave_lds(dt_tiles, water_d);
  B.group = B.row + kRW * DC;
  return B;
}
constexpr size_t kBatchLds = 160 * 1024;

// Whether the engine takes polymers of n beads: the bound that a workgroup holding the whole
// state in LDS would have (x and p of npad beads, five doubles per mode, the parameters),
// which keeps the accepted sizes independent of the kernel's layout.
inline bool batch_size_ok(const rp_pes* pes, int n) {
  const int npad = (n + 31) / 32 * 32, DC = 16 * batch_dtiles(pes);
  const size_t pl = pes->kind == PES_EVB ? 2 + 4 * DC + 2 * DC * (DC + 1) : 0;
  return ((size_t)npad * (2 * DC + 1 + 5) + pl) * sizeof(double) <= kBatchLds;
}

}  // namespace rp
