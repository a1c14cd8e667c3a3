// rp_ring.h -- internal interface between the ring kernels and the instanton driver.
#pragma once
#include <vector>

#include "rp_internal.h"

namespace rp {
int ring_eval(rp_ring* r, bool want_grad);            // energies (+ adjoint gradients) on device
int ring_upload_x(rp_ring* r, const double* x);
int ring_download(rp_ring* r, double* e, double* g);  // synchronises the ring's stream
int ring_tot(const rp_ring* r);
int ring_nchain(const rp_ring* r);
int ring_D(const rp_ring* r);
const std::vector<int>& ring_n(const rp_ring* r);
const std::vector<int64_t>& ring_off(const rp_ring* r);
int ring_lowest_eigen(rp_ring* r, const std::vector<int>& ng, double* eta);
// device views used by the instanton search: the evaluation point x, its adjoint gradient
// g and energies e (written by ring_eval), chain offsets and bead counts, the stream
struct RingBufs {
  double* x;
  double* g;
  const double* e;
  const int64_t* off;
  const int* n;
  int D;
  hipStream_t s;
};
RingBufs ring_bufs(rp_ring* r);
// the instanton search's preconditioner (rp_ring_set_preconditioner): Thomas coefficients per
// (chain, atom) from tab + off[chain], [1/denominator | alpha], or tab = nullptr (off).  A lane
// of the solve takes `run` consecutive beads; bead lane run + q is entry 64 q + lane, so that
// a wave's loads are contiguous; the entries past the chain's end are {0, 0}.
constexpr int kPcRun = 16;  // beads per lane at most: n <= 64 kPcRun = 1024
inline int pc_run(int n) { return (n + 63) >> 6; }
struct RingPc {
  const double* tab;
  const int64_t* off;
  int ndim;
};
RingPc ring_pc(rp_ring* r);
// the instanton search's vectors, kept by the ring between searches: `words` doubles and `ints`
// ints of device memory at least
int ring_search_ws(rp_ring* r, size_t words, size_t ints, double** w, int** iw);
}  // namespace rp
