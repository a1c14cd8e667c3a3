// rp_batch.hip -- host side of the batched engine (rp_batch_* in rp_hip.h).
//
// Polymers are grouped into families of equal (n, betan): one family shares the tables of its
// modes, and is advanced by one launch of the fused step kernel (rp_batch_kernel.h), whose
// workgroups hold one polymer or several (launch_batch_kind).
#include <algorithm>
#include <chrono>
#include <climits>
#include <cmath>
#include <cstring>
#include <map>

#include "rp_batch.h"

using namespace rp;

namespace {
struct Family {
  int N = 0, NPAD = 0;
  double betan = 0;
  int first = 0, count = 0;  // polymers [first, first+count) in batch order
  int waves = 4;             // wave budget of a workgroup (2, 4 or 8)
  bool waves_set = false;    // by set_launch or autotune, else the launch picks by occupancy
  DevBuf<double> d_T, d_Tf, d_lam;
};
}  // namespace

struct rp_batch {
  rp_pes* pes = nullptr;
  int ndim = 0, natom = 0, D = 0, DT = 0, DC = 0;
  int npoly = 0;
  double tau = 0, dt = 0, gamma = 0, limit = -1;
  int thermostat = RP_THERMO_LANGEVIN, cayley = 0;
  int64_t noutput = 1;
  uint64_t seed = 0;
  std::vector<int> order;     // batch position -> user index
  std::vector<int> pos;       // user index -> batch position
  std::vector<int> N;         // per batch position
  std::vector<int64_t> soff;  // per batch position, state offset (doubles)
  std::vector<Family> fam;
  hipStream_t s = nullptr;
  DevBuf<double> d_state, d_pf64, d_pdata, d_massd, d_noise, d_pathd;
  DevBuf<int64_t> d_pi64;
  DevBuf<uint64_t> d_stream;
  DevBuf<int32_t> d_kicks;
  DevBuf<int> d_flags;
  int npath = 0, ncu = 1;
  int64_t kick_cap = 0;
  int64_t steps_done = 0;
  int steps_per_launch = 64;
  std::vector<hipEvent_t> fev;  // per family: start, end
  std::vector<double> fam_ms;   // per family: summed launch time of the last run
  int64_t last_launches = 0;
  // Where every family's workgroups fit on the device at once, the families' launches run side
  // by side: on s and these streams, between the fork event and the families' end events.  The
  // longest chains take the streams first; family fi runs on lane[fi] (0: s).
  std::vector<hipStream_t> side;
  std::vector<int> lane;
  hipEvent_t fork = nullptr;
  bool in_turn = false;  // launch the families one after another all the same (autotune)
  // rp_batch_set_graphs: each family's launch of a step block (the last family's followed by
  // the step counter update) captured as a HIP graph and replayed between its timing events; a
  // graph is rebuilt when anything it captured changes.  Off by default: a block is one kernel
  // per family, so a replay saves no launch (run of 8 steps, 44 polymers of the 27-dof EVB,
  // N = 32: 96 us by graph, 81 us launched), and the first one pays for the capture.
  int use_graph = 0;
  struct GraphKey {
    int fam = -1;
    int steps = -1;
    int64_t imin = -1, kick_cap = -1;
    const void* kicks = nullptr;
    const void* pathd = nullptr;
    int npath = -1;
    std::vector<int> waves;
    bool operator==(const GraphKey& o) const {
      return fam == o.fam && steps == o.steps && imin == o.imin && kick_cap == o.kick_cap &&
             kicks == o.kicks &&
             pathd == o.pathd && npath == o.npath && waves == o.waves;
    }
  };
  PinBuf own_pin;
  PinBuf* pin = &own_pin;      // read-backs (fetch)
  std::vector<char> unpinned;  // larger ones
  std::vector<std::pair<GraphKey, hipGraphExec_t>> graphs;  // recent family step blocks
  DevBuf<int64_t> d_step0;
};

static void graph_drop(rp_batch* b) {
  for (auto& g : b->graphs) (void)hipGraphExecDestroy(g.second);
  b->graphs.clear();
}

// T lam in two halves, odd and even modes: Tf[half][r][l] = T(2 r + half, l) lam(2 r + half)
// over beads l < ceil(N/2), each half HP x HP and zero-padded.  Because
// sin(i (N+1-l) pi/(N+1)) = (-1)^(i+1) sin(i l pi/(N+1)), the other beads' values are the odd
// modes' sum minus the even modes': half the multiply-adds.  The identity holds to 3.4e-13
// relative at N = 256 with the reference's truncated pi.
static void family_tables(const Family& f, std::vector<double>& T, std::vector<double>& Tf,
                          std::vector<double>& lam) {
  const int N = f.N, NP = f.NPAD, Hc = (N + 1) / 2, HP = 16 * batch_tiles(N);
  T.assign((size_t)NP * NP, 0.0);
  Tf.assign(2 * (size_t)HP * HP, 0.0);
  lam.assign(NP, 0.0);
  for (int i = 1; i <= N; ++i) {
    lam[i - 1] = 2.0 * std::sin((double)i * kPiRef / (double)(2 * N + 2)) / f.betan;
    for (int l = i; l <= N; ++l) {
      double t = std::sin((double)(i * l) * kPiRef / (double)(N + 1)) * std::sqrt(2.0 / (double)(N + 1));
      T[(size_t)(i - 1) * NP + (l - 1)] = t;
      T[(size_t)(l - 1) * NP + (i - 1)] = t;
    }
  }
  for (int i = 0; i < N; ++i)
    for (int l = 0; l < Hc; ++l)
      Tf[((size_t)(i & 1) * HP + (i >> 1)) * HP + l] = T[(size_t)i * NP + l] * lam[i];
}

// Device arrays -> consecutive places in host memory (*out), then the stream is waited for.  The
// memory is b->pin, allocated with the batch at the size of its largest read-back (allocating
// 5.8 MB takes 2 ms, more than a run of 65536 small polymers), and beyond kPinMax pageable.
constexpr size_t kPinMax = (size_t)16 << 20;
static int fetch(rp_batch* b, std::initializer_list<std::pair<const void*, size_t>> parts, const char** out) {
  size_t bytes = 0;
  for (auto& q : parts) bytes += q.second;
  int rc;
  char* dst;
  if (bytes > kPinMax) {
    b->unpinned.resize(bytes);
    dst = b->unpinned.data();
  } else {
    if ((rc = b->pin->ensure(bytes))) return rc;
    dst = b->pin->p;
  }
  *out = dst;
  for (auto& q : parts) {
    RP_HIP(hipMemcpyAsync(dst, q.first, q.second, hipMemcpyDeviceToHost, b->s));
    dst += q.second;
  }
  RP_HIP(hipStreamSynchronize(b->s));
  return RP_OK;
}
// every polymer's 64-bit fields
static int fetch_pi(rp_batch* b, const int64_t** pi) {
  const char* h = nullptr;
  const int rc = fetch(b, {{b->d_pi64.p, b->d_pi64.n * sizeof(int64_t)}}, &h);
  *pi = reinterpret_cast<const int64_t*>(h);
  return rc;
}

static int batch_flags(rp_batch* b) {
  int rc;
  const char* h;
  if ((rc = fetch(b, {{b->d_flags.p, 2 * sizeof(int)}}, &h))) return rc;
  const int f[2] = {reinterpret_cast<const int*>(h)[0], reinterpret_cast<const int*>(h)[1]};
  if (f[0] || f[1]) {
    int z[2] = {0, 0};
    RP_HIP(hipMemcpy(b->d_flags.p, z, sizeof(z), hipMemcpyHostToDevice));
    if (f[0]) return set_error(RP_ERR_NAN, "NaN in the momenta of a batched polymer");
    return set_error(RP_ERR_NOISE, "injected noise or Poisson draws exhausted in the batch");
  }
  return RP_OK;
}

bool rp::batch_supports(const rp_pes* pes, int n) {
  if (!pes || n < 2 || n > 256) return false;
  const int D = pes->ndof;
  bool kind_ok = false;
  switch (pes->kind) {
    case PES_EVB: kind_ok = D <= 32; break;
    case PES_WATER: kind_ok = pes->natom == 3 || pes->natom == 6 || pes->natom == 18; break;
    case PES_QUARTIC: kind_ok = D <= 32; break;
    case PES_HARMONIC: kind_ok = D <= 16; break;
    case PES_COUPLED2D: kind_ok = true; break;
    default: kind_ok = false;  // host potentials and unknown kinds
  }
  return kind_ok && batch_size_ok(pes, n);
}

// A family's wave budget as rp_batch_family_shape reports it and rp_batch_set_launch bounds
// it: 8 from 8 to 16 MFMA units (32 modes x 16 dofs), 2 for at most 2, else 4.  Until a budget
// is asked for, the launch picks its groups per workgroup by occupancy (launch_batch_kind).
static int default_waves(int DT, int NPAD) {
  const int units = (NPAD >> 5) * DT;
  if (units <= 2 && DT <= 2) return 2;
  return (units >= 8 && units <= 16) ? 8 : 4;
}

static BatchArgs base_args(rp_batch* b, const Family& f, double h) {
  BatchArgs a;
  memset(&a, 0, sizeof(a));
  a.pes = b->pes->dev();
  a.waves = f.waves_set ? f.waves : 0;
  a.N = f.N;
  a.NPAD = f.NPAD;
  a.D = b->D;
  a.ndim = b->ndim;
  a.natom = b->natom;
  a.ncu = b->ncu;
  if (b->pes->kind == PES_EVB) a.moved = evb_moved(b->pes);
  a.first = f.first;
  a.dt = b->dt;
  a.limit = b->limit;
  a.stdev0 = std::sqrt(1.0 / f.betan);
  a.tau = b->tau;
  const double tau = b->tau;
  double c, sq, sp;
  if (b->cayley) {
    const double w2 = h * h / (tau * tau);
    c = (4.0 - w2) / (4.0 + w2);
    sq = 4.0 * h / (tau * tau * (4.0 + w2));
    sp = 4.0 * h / (4.0 + w2);
  } else {
    c = std::cos(h / tau);
    sq = std::sin(h / tau) / tau;
    sp = tau * std::sin(h / tau);
  }
  const double c1 = std::exp(-b->gamma * b->dt / tau), c1sq = c1 * c1;
  const double c2 = std::sqrt(1.0 - c1 * c1);
  a.kappa = tau * c2 * std::sqrt((1.0 + c1 * c1) / f.betan);
  const double bn2 = f.betan * f.betan, gx = sq * bn2 / (f.N + 1), ck = sp / bn2;
  a.iG = 1.0 / (f.N + 1);
  a.rot = Linear{c, gx, 1.0, c, ck, 0.0};
  a.aoa = Linear{c * c - sq * sp * c1sq, gx, c * (1.0 + c1sq), c * c * c1sq - sp * sq,
                 ck * c * (1.0 + c1sq), c};
  a.noutput = b->noutput;
  a.seed = b->seed;
  a.state = b->d_state.p;
  a.pi64 = b->d_pi64.p;
  a.pf64 = b->d_pf64.p;
  a.stream = b->d_stream.p;
  a.T = f.d_T.p;
  a.Tf = f.d_Tf.p;
  a.lam = f.d_lam.p;
  a.pdata = b->d_pdata.p;
  a.massd = b->d_massd.p;
  a.npath = b->npath;
  a.pathd = b->d_pathd.p;
  a.flags = b->d_flags.p;
  return a;
}

static int launch_family(rp_batch* b, const BatchArgs& a, int npoly, hipStream_t st) {
  switch (b->pes->kind) {
    case PES_EVB: return launch_batch_evb(b->pes, a, b->thermostat, npoly, st);
    case PES_WATER: return launch_batch_water(b->pes, a, b->thermostat, npoly, st);
    default: return launch_batch_simple(b->pes, a, b->thermostat, npoly, st);
  }
}

// Streams for families side by side.  A polymer takes at most one workgroup and a CU holds at
// least one, so with no more polymers than CUs nothing queues for a CU and each family takes as
// long as it would alone.  Beyond that the families fill the device one at a time, and their
// launches stay in order on one stream.  Up to kLanes at once, the hardware queues a process has
// by default; streams that share one still run in turn.  A run of 24 steps of 11 polymers each
// of 17, 45, 99, 150 and 251 beads (27-dof EVB): 1.59 ms in turn, 1.07 side by side; the longest
// family alone takes 0.65.
constexpr int kLanes = 4;
static int side_streams(rp_batch* b) {
  const int nf = (int)b->fam.size();
  b->lane.assign(nf, 0);
  if (nf < 2 || b->npoly > b->ncu) return RP_OK;
  RP_HIP(hipEventCreateWithFlags(&b->fork, hipEventDisableTiming));
  b->side.assign(std::min(nf, kLanes) - 1, nullptr);
  for (auto& st : b->side) RP_HIP(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
  std::vector<int> ord(nf);
  for (int i = 0; i < nf; ++i) ord[i] = i;
  std::stable_sort(ord.begin(), ord.end(), [&](int u, int v) { return b->fam[u].N > b->fam[v].N; });
  std::vector<int64_t> load(b->side.size() + 1, 0);
  for (int fi : ord) {
    const int l = (int)(std::min_element(load.begin(), load.end()) - load.begin());
    b->lane[fi] = l;
    load[l] += b->fam[fi].N;
  }
  return RP_OK;
}

extern "C" int rp_batch_create(rp_pes* pes, const double* mass, int npoly,
                               const rp_polymer_desc* desc, double tau, double dt, double gamma,
                               int thermostat, int64_t noutput, double dhdrlimit, int cayley,
                               uint64_t seed, rp_batch** out) {
  RP_REQUIRE(out, "rp_batch_create: out is NULL");
  *out = nullptr;
  RP_REQUIRE(pes && mass && desc && npoly > 0, "rp_batch_create: bad arguments");
  RP_REQUIRE(thermostat == RP_THERMO_LANGEVIN || thermostat == RP_THERMO_ANDERSEN,
             "rp_batch_create: thermostat must be 1 (Andersen) or 2 (Langevin)");
  RP_REQUIRE(tau > 0 && dt > 0, "rp_batch_create: tau and dt must be positive");
  RP_REQUIRE(thermostat != RP_THERMO_ANDERSEN || noutput > 0, "rp_batch_create: noutput <= 0");
  RP_REQUIRE(pes->kind != PES_HOST,
             "rp_batch_create: the fused kernel evaluates the potential on the device; a "
             "potential that lives on the host runs through the plain path (rp_nm_setup)");
  int rc = ensure_init();
  if (rc) return rc;
  rp_batch* b = new rp_batch();
  b->pes = pes;
  b->ndim = pes->ndim;
  b->natom = pes->natom;
  b->D = pes->ndof;
  b->DT = batch_dtiles(pes);
  b->DC = 16 * b->DT;
  b->npoly = npoly;
  b->tau = tau;
  b->dt = dt;
  b->gamma = gamma;
  b->limit = dhdrlimit;
  b->thermostat = thermostat;
  b->cayley = cayley;
  b->noutput = noutput;
  b->seed = seed;
  auto fail = [&](int code) {
    rp_batch_destroy(b);
    return code;
  };
  for (int p = 0; p < npoly; ++p) {
    const int n = desc[p].n;
    if (n < 2 || n > 256) return fail(set_error(RP_ERR_ARG, "polymer %d: n=%d outside 2..256", p, n));
    if (!(desc[p].betan > 0) || !desc[p].a || !desc[p].b || !desc[p].dbdl)
      return fail(set_error(RP_ERR_ARG, "polymer %d: bad descriptor", p));
    if (!batch_size_ok(pes, n))
      return fail(set_error(RP_ERR_ARG, "polymer %d: n=%d with %d dof needs more LDS than a CU has",
                            p, n, b->D));
  }
  // families of equal (n, betan), each contiguous in batch order
  std::map<std::pair<int, double>, std::vector<int>> groups;
  for (int p = 0; p < npoly; ++p) groups[{desc[p].n, desc[p].betan}].push_back(p);
  for (auto& kv : groups) {
    Family f;
    f.N = kv.first.first;
    f.NPAD = (f.N + 31) / 32 * 32;
    f.betan = kv.first.second;
    f.first = (int)b->order.size();
    f.count = (int)kv.second.size();
    f.waves = default_waves(b->DT, f.NPAD);
    for (int p : kv.second) b->order.push_back(p);
    b->fam.push_back(std::move(f));
  }
  b->pos.assign(npoly, 0);
  for (int k = 0; k < npoly; ++k) b->pos[b->order[k]] = k;
  const int D = b->D, DC = b->DC;
  std::vector<int64_t> pi64((size_t)npoly * kPI64, 0);
  std::vector<double> pf64((size_t)npoly * kPF64, 0.0), pdata((size_t)npoly * 3 * DC, 0.0);
  std::vector<uint64_t> streams(npoly);
  int64_t off = 0;
  b->N.resize(npoly);
  b->soff.resize(npoly);
  for (int k = 0; k < npoly; ++k) {
    const rp_polymer_desc& d = desc[b->order[k]];
    b->N[k] = d.n;
    b->soff[k] = off;
    pi64[(size_t)k * kPI64 + PI_STATE_OFF] = off;
    pi64[(size_t)k * kPI64 + PI_RKICK] = -1;  // first Poisson interval not drawn yet
    off += 2 * (int64_t)D * d.n;
    pf64[(size_t)k * kPF64 + PF_XI] = d.xi;
    for (int j = 0; j < D; ++j) {
      pdata[(size_t)k * 3 * DC + j] = d.a[j];
      pdata[(size_t)k * 3 * DC + DC + j] = d.b[j];
      pdata[(size_t)k * 3 * DC + 2 * DC + j] = d.dbdl[j];
    }
    streams[k] = d.stream;
  }
  std::vector<double> massd(DC, 1.0);
  for (int a = 0; a < b->natom; ++a)
    for (int j = 0; j < b->ndim; ++j) massd[a * b->ndim + j] = mass[a];
  int zf[2] = {0, 0};
  if ((rc = [&]() -> int {
        RP_HIP(hipStreamCreateWithFlags(&b->s, hipStreamNonBlocking));
        int dev = 0;
        RP_HIP(hipGetDevice(&dev));
        RP_HIP(hipDeviceGetAttribute(&b->ncu, hipDeviceAttributeMultiprocessorCount, dev));
        b->fev.assign(2 * b->fam.size(), nullptr);
        for (auto& e : b->fev) RP_HIP(hipEventCreate(&e));
        int sr;
        if ((sr = side_streams(b))) return sr;
        // a one-polymer batch may be a chain's plan, which brings the chain's buffer
        const size_t nmax = *std::max_element(b->N.begin(), b->N.end());
        const size_t most = std::max(2 * 8 * nmax * D, (size_t)npoly * 8 * (size_t)(int(kPI64) + int(kPF64)));
        if (npoly > 1 && (sr = b->own_pin.ensure(std::min(most, kPinMax)))) return sr;
        int r;
        if ((r = b->d_state.alloc(off))) return r;
        RP_HIP(hipMemsetAsync(b->d_state.p, 0, off * sizeof(double), b->s));
        if ((r = b->d_pi64.alloc(pi64.size())) || (r = b->d_pi64.upload(pi64.data(), pi64.size(), b->s))) return r;
        if ((r = b->d_pf64.alloc(pf64.size())) || (r = b->d_pf64.upload(pf64.data(), pf64.size(), b->s))) return r;
        if ((r = b->d_pdata.alloc(pdata.size())) || (r = b->d_pdata.upload(pdata.data(), pdata.size(), b->s))) return r;
        if ((r = b->d_stream.alloc(npoly)) || (r = b->d_stream.upload(streams.data(), npoly, b->s))) return r;
        if ((r = b->d_massd.alloc(DC)) || (r = b->d_massd.upload(massd.data(), DC, b->s))) return r;
        if ((r = b->d_flags.alloc(2)) || (r = b->d_flags.upload(zf, 2, b->s))) return r;
        for (Family& f : b->fam) {
          std::vector<double> T, Tf, lam;
          family_tables(f, T, Tf, lam);
          if ((r = f.d_T.alloc(T.size())) || (r = f.d_T.upload(T.data(), T.size(), b->s))) return r;
          if ((r = f.d_Tf.alloc(Tf.size())) || (r = f.d_Tf.upload(Tf.data(), Tf.size(), b->s))) return r;
          if ((r = f.d_lam.alloc(lam.size())) || (r = f.d_lam.upload(lam.data(), lam.size(), b->s))) return r;
          RP_HIP(hipStreamSynchronize(b->s));  // the host tables are released here
        }
        RP_HIP(hipStreamSynchronize(b->s));
        return RP_OK;
      }()))
    return fail(rc);
  *out = b;
  return RP_OK;
}

extern "C" int rp_batch_destroy(rp_batch* b) {
  if (!b) return RP_OK;
  if (b->s) (void)hipStreamSynchronize(b->s);
  for (auto& st : b->side)
    if (st) (void)hipStreamSynchronize(st);
  graph_drop(b);
  b->d_step0.free();
  for (Family& f : b->fam) {
    f.d_T.free();
    f.d_Tf.free();
    f.d_lam.free();
  }
  for (DevBuf<double>* d : {&b->d_state, &b->d_pf64, &b->d_pdata, &b->d_massd, &b->d_noise, &b->d_pathd})
    d->free();
  b->d_pi64.free();
  b->d_stream.free();
  b->d_kicks.free();
  b->d_flags.free();
  b->own_pin.free();
  for (auto& e : b->fev)
    if (e) (void)hipEventDestroy(e);
  if (b->fork) (void)hipEventDestroy(b->fork);
  for (auto& st : b->side)
    if (st) (void)hipStreamDestroy(st);
  if (b->s) (void)hipStreamDestroy(b->s);
  delete b;
  return RP_OK;
}

extern "C" int rp_batch_set_path(rp_batch* b, int npath, const double* lampath, const double* path) {
  RP_REQUIRE(b && lampath && path && npath >= 2, "rp_batch_set_path: bad arguments");
  std::vector<double> y2;
  path_spline_host(npath, b->D, lampath, path, y2);
  std::vector<double> pd((size_t)npath * (1 + 2 * b->D));
  memcpy(pd.data(), lampath, npath * sizeof(double));
  memcpy(pd.data() + npath, path, (size_t)npath * b->D * sizeof(double));
  memcpy(pd.data() + (size_t)npath * (1 + b->D), y2.data(), (size_t)npath * b->D * sizeof(double));
  int rc;
  if ((rc = b->d_pathd.alloc(pd.size())) || (rc = b->d_pathd.upload(pd.data(), pd.size(), b->s))) return rc;
  b->npath = npath;
  RP_HIP(hipStreamSynchronize(b->s));
  return RP_OK;
}

// Injected draws: polymer p (user order) owns noise[p*cap, (p+1)*cap), indexed from 0 for
// this call; the Philox cursors are saved before and restored after, so injected calls
// leave the engine's own streams where they were.
static int noise_begin(rp_batch* b, const double* noise, int64_t cap, std::vector<int64_t>& saved) {
  int rc;
  const size_t tot = (size_t)b->npoly * cap;
  if (b->d_noise.n < tot && (rc = b->d_noise.alloc(tot))) return rc;
  if ((rc = b->d_noise.upload(noise, tot, b->s))) return rc;
  saved.resize((size_t)b->npoly * kPI64);
  if ((rc = b->d_pi64.download(saved.data(), saved.size(), b->s))) return rc;
  RP_HIP(hipStreamSynchronize(b->s));
  std::vector<int64_t> pi = saved;
  for (int k = 0; k < b->npoly; ++k) {
    pi[(size_t)k * kPI64 + PI_NOISE_OFF] = (int64_t)b->order[k] * cap;
    pi[(size_t)k * kPI64 + PI_CURSOR] = 0;
  }
  return b->d_pi64.upload(pi.data(), pi.size(), b->s);
}

static int noise_end(rp_batch* b, const std::vector<int64_t>& saved) {
  std::vector<int64_t> pi(saved.size());
  int rc;
  if ((rc = b->d_pi64.download(pi.data(), pi.size(), b->s))) return rc;
  RP_HIP(hipStreamSynchronize(b->s));
  for (int k = 0; k < b->npoly; ++k)
    pi[(size_t)k * kPI64 + PI_CURSOR] = saved[(size_t)k * kPI64 + PI_CURSOR];
  return b->d_pi64.upload(pi.data(), pi.size(), b->s);
}

// init_path (verletmodule.f90:32-119) of every polymer of a family, one workgroup each:
// NM momenta sqrt(m'/betan) z with the draws in (dim outer, atom inner) blocks of N
// (:102-106), p = T v (:107-115), and the beads spread along the path spline,
// x_k = splint(path, (k-1) xi/(N-1)) (:40-48).  It runs once per task, so a plain dense
// product serves; the step kernel's launches then all have the same shape.
__global__ void __launch_bounds__(256) batch_init_kernel(BatchArgs A) {
  extern __shared__ double V[];
  const int poly = A.first + blockIdx.x, tid = threadIdx.x;
  const int N = A.N, NPAD = A.NPAD, D = A.D, ndim = A.ndim, natom = A.natom;
  int64_t* pi = A.pi64 + (size_t)poly * kPI64;
  double* st = A.state + pi[PI_STATE_OFF];
  const int64_t noff = pi[PI_NOISE_OFF], cur = pi[PI_CURSOR], need = (int64_t)N * D;
  const uint64_t strm = A.stream[poly];
  if (A.noise && cur + need > A.noise_cap) {  // the same for every thread of the block
    if (tid == 0) atomicOr(&A.flags[1], 1);
    return;
  }
  for (int e = tid; e < N * D; e += blockDim.x) {
    const int c = e / N, i = e - c * N;
    const int atom = c / ndim, dim = c - atom * ndim;
    const int64_t idx = cur + (int64_t)(dim * natom + atom) * N + i;
    const double z = A.noise ? A.noise[noff + idx] : philox_normal(A.seed, strm, idx);
    V[e] = (A.stdev0 * z) * (sqrt(A.massd[c]) * A.lam[i] * A.tau);
  }
  __syncthreads();
  const double xi = A.pf64[(size_t)poly * kPF64 + PF_XI];
  const double* lampath = A.pathd;
  for (int e = tid; e < N * D; e += blockDim.x) {
    const int c = e / N, i = e - c * N;
    double acc = 0.0;
    for (int k = 0; k < N; ++k) acc += A.T[(size_t)k * NPAD + i] * V[c * N + k];
    st[(size_t)D * N + e] = acc;
    st[e] = splint_dev(lampath, lampath + A.npath + (size_t)c * A.npath,
                       lampath + A.npath * (1 + D) + (size_t)c * A.npath, A.npath,
                       (double)i * xi / (double)(N - 1));
  }
  if (tid == 0) pi[PI_CURSOR] = cur + need;
}

static int run_init(rp_batch* b, const double* dn, int64_t cap) {
  for (size_t fi = 0; fi < b->fam.size(); ++fi) {
    Family& f = b->fam[fi];
    BatchArgs a = base_args(b, f, 0.5 * b->dt);
    a.nsteps = 0;
    a.noise = dn;
    a.noise_cap = cap;
    const size_t lds = (size_t)f.N * b->D * sizeof(double);
    RP_REQUIRE(lds <= 160 * 1024, "rp_batch_init_path: N*ndof = %d is too large",
               f.N * b->D);
    RP_HIP(hipFuncSetAttribute((const void*)batch_init_kernel,
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    batch_init_kernel<<<f.count, 256, lds, b->s>>>(a);
    RP_HIP(hipGetLastError());
  }
  RP_HIP(hipStreamSynchronize(b->s));
  return RP_OK;
}

__global__ void batch_advance_kernel(int64_t* step0, int steps) {
  if (threadIdx.x == 0) *step0 += steps;
}

static rp_batch::GraphKey graph_key(const rp_batch* b, size_t fi, int steps, int64_t imin) {
  rp_batch::GraphKey k;
  k.fam = (int)fi;
  k.steps = steps;
  k.imin = imin;
  k.kick_cap = b->kick_cap;
  k.kicks = b->d_kicks.p;
  k.pathd = b->d_pathd.p;
  k.npath = b->npath;
  for (const Family& f : b->fam) k.waves.push_back(f.waves_set ? f.waves : 0);
  return k;
}

// Capture family fi's launch of one step block (and, for the last family, the device step
// counter advance).  The stream leaves capture mode on every path.
static int graph_build(rp_batch* b, size_t fi, int steps, int64_t imin, hipGraphExec_t* out) {
  int rc;
  if (!b->d_step0.p && (rc = b->d_step0.alloc(1))) return rc;
  Family& f = b->fam[fi];
  BatchArgs a = base_args(b, f, 0.5 * b->dt);
  a.nsteps = steps;
  a.step0 = 0;
  a.step0p = b->d_step0.p;
  a.imin = imin;
  a.kicks = b->d_kicks.p;
  a.kick_cap = b->kick_cap;
  RP_HIP(hipStreamBeginCapture(b->s, hipStreamCaptureModeRelaxed));
  rc = launch_family(b, a, f.count, b->s);
  if (rc == RP_OK && fi + 1 == b->fam.size()) {
    batch_advance_kernel<<<1, 64, 0, b->s>>>(b->d_step0.p, steps);
    if (hipGetLastError() != hipSuccess)
      rc = set_error(RP_ERR_HIP, "batch graph: capture of the step counter failed");
  }
  hipGraph_t g = nullptr;
  const hipError_t e = hipStreamEndCapture(b->s, &g);
  if (rc == RP_OK && e != hipSuccess)
    rc = set_error(RP_ERR_HIP, "batch graph: capture failed (%s)", hipGetErrorString(e));
  hipGraphExec_t exec = nullptr;
  if (rc == RP_OK) {
    const hipError_t ei = hipGraphInstantiate(&exec, g, nullptr, nullptr, 0);
    if (ei != hipSuccess)
      rc = set_error(RP_ERR_HIP, "batch graph: instantiate failed (%s)", hipGetErrorString(ei));
  }
  if (g) (void)hipGraphDestroy(g);
  if (rc != RP_OK) return rc;
  if (b->graphs.size() >= 64) {
    (void)hipGraphExecDestroy(b->graphs.front().second);
    b->graphs.erase(b->graphs.begin());
  }
  b->graphs.emplace_back(graph_key(b, fi, steps, imin), exec);
  *out = exec;
  return RP_OK;
}

// One launch per family of `steps` steps, each bracketed by its own events; per-family
// durations are accumulated into fam_ms.  By graph (use_graph, no injected draws) the block is a
// replay, in order on one stream; else its launches run side by side where side_streams set that
// up.
static int run_block(rp_batch* b, int steps, int64_t imin, const double* dn, int64_t cap,
                     std::vector<double>& fam_ms) {
  int rc;
  if (b->use_graph && !dn) {
    std::vector<hipGraphExec_t> exec(b->fam.size(), nullptr);
    for (size_t fi = 0; fi < b->fam.size(); ++fi) {
      const rp_batch::GraphKey key = graph_key(b, fi, steps, imin);
      for (auto& g : b->graphs)
        if (g.first == key) exec[fi] = g.second;
      if (!exec[fi] && (rc = graph_build(b, fi, steps, imin, &exec[fi]))) return rc;
    }
    RP_HIP(hipMemcpyAsync(b->d_step0.p, &b->steps_done, sizeof(int64_t), hipMemcpyHostToDevice, b->s));
    for (size_t fi = 0; fi < b->fam.size(); ++fi) {
      RP_HIP(hipEventRecord(b->fev[2 * fi], b->s));
      RP_HIP(hipGraphLaunch(exec[fi], b->s));
      RP_HIP(hipEventRecord(b->fev[2 * fi + 1], b->s));
    }
  } else {
    const bool apart = !b->side.empty() && !b->in_turn;
    auto stream = [&](size_t fi) { return apart && b->lane[fi] ? b->side[b->lane[fi] - 1] : b->s; };
    if (apart) {
      RP_HIP(hipEventRecord(b->fork, b->s));
      for (hipStream_t st : b->side) RP_HIP(hipStreamWaitEvent(st, b->fork, 0));
    }
    auto launch = [&](size_t fi) -> int {
      Family& f = b->fam[fi];
      BatchArgs a = base_args(b, f, 0.5 * b->dt);
      a.nsteps = steps;
      a.step0 = b->steps_done;
      a.imin = imin;
      a.noise = dn;
      a.noise_cap = cap;
      a.kicks = b->d_kicks.p;
      a.kick_cap = b->kick_cap;
      int q;
      RP_HIP(hipEventRecord(b->fev[2 * fi], stream(fi)));
      if ((q = launch_family(b, a, f.count, stream(fi)))) return q;
      RP_HIP(hipEventRecord(b->fev[2 * fi + 1], stream(fi)));
      return RP_OK;
    };
    // the longest first; families come in the order of their bead counts
    rc = RP_OK;
    size_t fi = b->fam.size();
    while (fi > 0 && !rc) rc = launch(--fi);
    // s waits for what the other streams got, once it has its own; after a failure too
    if (apart)
      for (hipStream_t st : b->side) {
        RP_HIP(hipEventRecord(b->fork, st));
        RP_HIP(hipStreamWaitEvent(b->s, b->fork, 0));
      }
    if (rc) return rc;
  }
  RP_HIP(hipStreamSynchronize(b->s));  // which waits for every family
  fam_ms.resize(b->fam.size(), 0.0);
  for (size_t fi = 0; fi < b->fam.size(); ++fi) {
    float ms = 0.f;
    RP_HIP(hipEventElapsedTime(&ms, b->fev[2 * fi], b->fev[2 * fi + 1]));
    fam_ms[fi] += ms;
  }
  return RP_OK;
}

extern "C" int rp_batch_init_path(rp_batch* b, const double* noise) {
  RP_REQUIRE(b, "rp_batch_init_path: NULL batch");
  RP_REQUIRE(b->npath >= 2, "rp_batch_init_path: no path set (rp_batch_set_path)");
  int rc;
  std::vector<int64_t> saved;
  int64_t cap = 0;
  if (noise) {
    // polymer p's n*ndof draws follow each other in user order; repack at a uniform stride
    for (int k = 0; k < b->npoly; ++k) cap = std::max<int64_t>(cap, (int64_t)b->N[k] * b->D);
    std::vector<double> packed((size_t)b->npoly * cap, 0.0);
    int64_t src = 0;
    for (int p = 0; p < b->npoly; ++p) {
      const int64_t cnt = (int64_t)b->N[b->pos[p]] * b->D;
      memcpy(packed.data() + (size_t)p * cap, noise + src, cnt * sizeof(double));
      src += cnt;
    }
    if ((rc = noise_begin(b, packed.data(), cap, saved))) return rc;
  }
  if ((rc = run_init(b, noise ? b->d_noise.p : nullptr, cap))) return rc;
  if (noise && (rc = noise_end(b, saved))) return rc;
  return batch_flags(b);
}

extern "C" int rp_batch_set_state(rp_batch* b, int poly, const double* x, const double* p) {
  RP_REQUIRE(b && x && p && poly >= 0 && poly < b->npoly, "rp_batch_set_state: bad arguments");
  const int k = b->pos[poly];
  const size_t nd = (size_t)b->N[k] * b->D;
  RP_HIP(hipMemcpyAsync(b->d_state.p + b->soff[k], x, nd * sizeof(double), hipMemcpyHostToDevice, b->s));
  RP_HIP(hipMemcpyAsync(b->d_state.p + b->soff[k] + nd, p, nd * sizeof(double), hipMemcpyHostToDevice, b->s));
  RP_HIP(hipStreamSynchronize(b->s));
  return RP_OK;
}

extern "C" int rp_batch_get_state(rp_batch* b, int poly, double* x, double* p) {
  RP_REQUIRE(b && poly >= 0 && poly < b->npoly, "rp_batch_get_state: bad arguments");
  const int k = b->pos[poly];
  const size_t nd = (size_t)b->N[k] * b->D, bytes = nd * sizeof(double);
  if (!x && !p) return RP_OK;
  int rc;
  const char* h;
  if ((rc = fetch(b, {{b->d_state.p + b->soff[k] + (x ? 0 : nd), x && p ? 2 * bytes : bytes}},
                  &h)))
    return rc;
  if (x) memcpy(x, h, bytes);
  if (p) memcpy(p, h + (x ? bytes : 0), bytes);
  return RP_OK;
}

namespace rp {
int batch_restart(rp_batch* b, const double* d_state, int64_t cursor, int64_t kcursor, PinBuf* pin) {
  RP_REQUIRE(b->npoly == 1, "batch_restart: one polymer");
  RP_REQUIRE(cursor >= 0 && kcursor >= 0, "rp_batch_set_cursor: negative cursor");
  b->pin = pin;
  int rc;
  if ((rc = pin->ensure(8 * kPI64 + 8 * kPF64))) return rc;
  int64_t* pi = reinterpret_cast<int64_t*>(pin->p);
  std::fill(pi, pi + kPI64, 0);  // and the state's offset
  pi[PI_CURSOR] = cursor;
  pi[PI_KCURSOR] = kcursor;
  pi[PI_RKICK] = -1;
  double* sum = reinterpret_cast<double*>(pi + kPI64);
  *sum = 0.0;
  RP_HIP(hipMemcpyAsync(b->d_pi64.p, pi, kPI64 * 8, hipMemcpyHostToDevice, b->s));
  RP_HIP(hipMemcpyAsync(b->d_pf64.p + PF_TISUM, sum, 8, hipMemcpyHostToDevice, b->s));
  RP_HIP(hipMemcpyAsync(b->d_state.p, d_state, 2 * (size_t)b->N[0] * b->D * sizeof(double),
                        hipMemcpyDeviceToDevice, b->s));
  RP_HIP(hipStreamSynchronize(b->s));  // pin is free again
  b->steps_done = 0;
  return RP_OK;
}

int batch_result(rp_batch* b, double* d_state, double* sum, int64_t* count, int64_t* nreinit,
                 int64_t* cursor, int64_t* kcursor) {
  RP_HIP(hipMemcpyAsync(d_state, b->d_state.p, 2 * (size_t)b->N[0] * b->D * sizeof(double),
                        hipMemcpyDeviceToDevice, b->s));
  int rc;
  const char* h;
  if ((rc = fetch(b, {{b->d_pi64.p, kPI64 * 8}, {b->d_pf64.p, kPF64 * 8}}, &h))) return rc;
  const int64_t* pi = reinterpret_cast<const int64_t*>(h);
  *sum = reinterpret_cast<const double*>(pi + kPI64)[PF_TISUM];
  *count = pi[PI_TICNT];
  *nreinit = pi[PI_NREINIT];
  *cursor = pi[PI_CURSOR];
  *kcursor = pi[PI_KCURSOR];
  return RP_OK;
}
}  // namespace rp

extern "C" int rp_batch_set_kicks(rp_batch* b, const int32_t* kicks, int64_t nkicks_per_poly) {
  RP_REQUIRE(b && (kicks == nullptr || nkicks_per_poly > 0), "rp_batch_set_kicks: bad arguments");
  int rc;
  if (!kicks) {
    b->d_kicks.free();
    b->kick_cap = 0;
    return RP_OK;
  }
  const size_t tot = (size_t)b->npoly * nkicks_per_poly;
  if ((rc = b->d_kicks.alloc(tot)) || (rc = b->d_kicks.upload(kicks, tot, b->s))) return rc;
  std::vector<int64_t> pi((size_t)b->npoly * kPI64);
  if ((rc = b->d_pi64.download(pi.data(), pi.size(), b->s))) return rc;
  RP_HIP(hipStreamSynchronize(b->s));
  for (int k = 0; k < b->npoly; ++k) {
    pi[(size_t)k * kPI64 + PI_KICK_OFF] = (int64_t)b->order[k] * nkicks_per_poly;
    pi[(size_t)k * kPI64 + PI_KCURSOR] = 0;
    pi[(size_t)k * kPI64 + PI_RKICK] = -1;
    pi[(size_t)k * kPI64 + PI_ACOUNT] = 0;
  }
  b->kick_cap = nkicks_per_poly;
  if ((rc = b->d_pi64.upload(pi.data(), pi.size(), b->s))) return rc;
  RP_HIP(hipStreamSynchronize(b->s));
  return RP_OK;
}

extern "C" int rp_batch_run(rp_batch* b, int64_t nsteps, int64_t imin, const double* noise,
                            int64_t nnoise_per_poly) {
  RP_REQUIRE(b && nsteps >= 0 && imin >= 0, "rp_batch_run: bad arguments");
  RP_REQUIRE(!noise || nnoise_per_poly > 0, "rp_batch_run: injected noise needs nnoise_per_poly > 0");
  RP_REQUIRE(!(b->thermostat == RP_THERMO_LANGEVIN && b->limit >= 0.0) || b->npath >= 2,
             "rp_batch_run: dHdrlimit >= 0 re-initialises from the path: call rp_batch_set_path");
  int rc;
  std::vector<int64_t> saved;
  if (noise && (rc = noise_begin(b, noise, nnoise_per_poly, saved))) return rc;
  std::vector<double> fam_ms(b->fam.size(), 0.0);
  int64_t launches = 0, left = nsteps;
  while (left > 0) {
    const int steps = (int)std::min<int64_t>(left, b->steps_per_launch);
    if ((rc = run_block(b, steps, imin, noise ? b->d_noise.p : nullptr, nnoise_per_poly,
                        fam_ms)))
      return rc;
    ++launches;
    b->steps_done += steps;
    left -= steps;
  }
  b->fam_ms = fam_ms;
  b->last_launches = launches;
  if (noise && (rc = noise_end(b, saved))) return rc;
  return batch_flags(b);
}

extern "C" int rp_batch_ti_readout(rp_batch* b, double* dhdr_sum, int64_t* count,
                                   int64_t* nreinit) {
  RP_REQUIRE(b, "rp_batch_ti_readout: NULL batch");
  int rc;
  const char* h;
  if ((rc = fetch(b, {{b->d_pi64.p, b->d_pi64.n * 8}, {b->d_pf64.p, b->d_pf64.n * 8}}, &h))) return rc;
  const int64_t* pi = reinterpret_cast<const int64_t*>(h);
  const double* pf = reinterpret_cast<const double*>(pi + b->d_pi64.n);
  for (int p = 0; p < b->npoly; ++p) {
    const int k = b->pos[p];
    if (dhdr_sum) dhdr_sum[p] = pf[(size_t)k * kPF64 + PF_TISUM];
    if (count) count[p] = pi[(size_t)k * kPI64 + PI_TICNT];
    if (nreinit) nreinit[p] = pi[(size_t)k * kPI64 + PI_NREINIT];
  }
  return RP_OK;
}

extern "C" int rp_batch_get_cursor(rp_batch* b, int64_t* cursor) {
  RP_REQUIRE(b && cursor, "rp_batch_get_cursor: bad arguments");
  const int64_t* pi;
  int rc;
  if ((rc = fetch_pi(b, &pi))) return rc;
  for (int p = 0; p < b->npoly; ++p) cursor[p] = pi[(size_t)b->pos[p] * kPI64 + PI_CURSOR];
  return RP_OK;
}

extern "C" int rp_batch_get_kick_cursor(rp_batch* b, int64_t* kick_cursor) {
  RP_REQUIRE(b && kick_cursor, "rp_batch_get_kick_cursor: bad arguments");
  const int64_t* pi;
  int rc;
  if ((rc = fetch_pi(b, &pi))) return rc;
  for (int p = 0; p < b->npoly; ++p)
    kick_cursor[p] = pi[(size_t)b->pos[p] * kPI64 + PI_KCURSOR];
  return RP_OK;
}

// Resume: place every polymer's normal and Poisson draws at saved stream positions.  A new
// Poisson cursor also discards the interval in progress, so the next step draws a fresh one,
// as propagate_pimd_nm does on entry.
extern "C" int rp_batch_set_cursor(rp_batch* b, const int64_t* cursor, const int64_t* kick_cursor) {
  RP_REQUIRE(b, "rp_batch_set_cursor: NULL batch");
  for (int p = 0; p < b->npoly; ++p)
    RP_REQUIRE((!cursor || cursor[p] >= 0) && (!kick_cursor || kick_cursor[p] >= 0),
               "rp_batch_set_cursor: negative cursor");
  std::vector<int64_t> pi((size_t)b->npoly * kPI64);
  int rc;
  if ((rc = b->d_pi64.download(pi.data(), pi.size(), b->s))) return rc;
  RP_HIP(hipStreamSynchronize(b->s));
  for (int p = 0; p < b->npoly; ++p) {
    int64_t* q = pi.data() + (size_t)b->pos[p] * kPI64;
    if (cursor) q[PI_CURSOR] = cursor[p];
    if (kick_cursor) {
      q[PI_KCURSOR] = kick_cursor[p];
      q[PI_RKICK] = -1;
      q[PI_ACOUNT] = 0;
    }
  }
  if ((rc = b->d_pi64.upload(pi.data(), pi.size(), b->s))) return rc;
  RP_HIP(hipStreamSynchronize(b->s));
  return RP_OK;
}

extern "C" int rp_batch_set_graphs(rp_batch* b, int enable) {
  RP_REQUIRE(b, "rp_batch_set_graphs: NULL batch");
  b->use_graph = enable ? 1 : 0;
  if (!enable) graph_drop(b);
  return RP_OK;
}

// 8 waves per workgroup needs at most 16 MFMA units (2 per wave)
static bool eight_waves_fit(const rp_batch* b, const Family& f) {
  return (f.NPAD >> 5) * b->DT <= 16;
}

// 2 waves run a family only when each wave holds one of at most two units (W is a multiple
// of DT); otherwise such a request falls back to 4
static bool two_waves_fit(const rp_batch* b, const Family& f) {
  return b->DT <= 2 && (f.NPAD >> 5) * b->DT <= 2;
}

static int fitted_waves(const rp_batch* b, const Family& f, int w) {
  if (w == 8) return eight_waves_fit(b, f) ? 8 : 4;
  if (w == 2) return two_waves_fit(b, f) ? 2 : 4;
  return 4;
}

extern "C" int rp_batch_set_launch(rp_batch* b, int steps_per_launch, int waves) {
  RP_REQUIRE(b && steps_per_launch >= 0, "rp_batch_set_launch: bad arguments");
  RP_REQUIRE(waves == 0 || waves == 2 || waves == 4 || waves == 8,
             "rp_batch_set_launch: waves per workgroup must be 2, 4 or 8");
  if (steps_per_launch > 0) b->steps_per_launch = steps_per_launch;
  if (waves)
    for (Family& f : b->fam) {
      f.waves = fitted_waves(b, f, waves);
      f.waves_set = true;
    }
  return RP_OK;
}

extern "C" int rp_batch_autotune(rp_batch* b, int trial_steps, int* best_steps, int* best_waves) {
  RP_REQUIRE(b && trial_steps > 0, "rp_batch_autotune: bad arguments");
  int rc;
  // save the whole mutable state, time each candidate, restore
  const size_t ns = b->d_state.n;
  std::vector<double> st(ns), pf((size_t)b->npoly * kPF64);
  std::vector<int64_t> pi((size_t)b->npoly * kPI64);
  if ((rc = b->d_state.download(st.data(), ns, b->s)) || (rc = b->d_pf64.download(pf.data(), pf.size(), b->s)) ||
      (rc = b->d_pi64.download(pi.data(), pi.size(), b->s)))
    return rc;
  RP_HIP(hipStreamSynchronize(b->s));
  auto restore = [&]() -> int {
    int r;
    if ((r = b->d_state.upload(st.data(), ns, b->s)) || (r = b->d_pf64.upload(pf.data(), pf.size(), b->s)) ||
        (r = b->d_pi64.upload(pi.data(), pi.size(), b->s)))
      return r;
    RP_HIP(hipStreamSynchronize(b->s));
    return RP_OK;
  };
  auto trial = [&](int cs, std::vector<double>& fam_ms, double& sec) -> int {
    fam_ms.assign(b->fam.size(), 0.0);
    auto t0 = std::chrono::steady_clock::now();
    int64_t left = trial_steps;
    while (left > 0) {
      const int steps = (int)std::min<int64_t>(left, cs);
      int r;
      if ((r = run_block(b, steps, INT64_MAX / 2, nullptr, 0, fam_ms))) return r;
      left -= steps;
    }
    sec = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    return restore();
  };
  const int64_t steps0 = b->steps_done;
  // 1. waves per family, from each family's own hipEvent-timed launches, one family at a time:
  // no budget set (0: groups by occupancy, helper waves for small batches; launch_batch_kind),
  // and the budgets that fit.  A budget takes over only where it is faster by more than two runs
  // of one kernel differ.  Each is run once before it is timed: its first launch loads its code.
  const size_t nf = b->fam.size();
  std::vector<double> best_ms(nf, 1e300), fam_ms;
  std::vector<int> best_w(nf, 0);
  auto set_waves = [&](Family& f, int w) {
    f.waves = w ? fitted_waves(b, f, w) : default_waves(b->DT, f.NPAD);
    f.waves_set = w != 0;
  };
  double sec = 0.0;
  b->in_turn = true;
  for (int w : {0, 2, 4, 8}) {
    for (Family& f : b->fam) set_waves(f, w);
    for (int k = 0; k < 2; ++k)
      if ((rc = trial(std::min(b->steps_per_launch, trial_steps), fam_ms, sec))) {
        b->in_turn = false;
        return rc;
      }
    for (size_t fi = 0; fi < nf; ++fi)
      if (w == 0 || (b->fam[fi].waves == w && fam_ms[fi] < (best_w[fi] ? 1.0 : 0.97) * best_ms[fi])) {
        best_ms[fi] = fam_ms[fi];
        best_w[fi] = w;
      }
  }
  b->in_turn = false;
  int nw[9] = {0};
  for (size_t fi = 0; fi < nf; ++fi) {
    set_waves(b->fam[fi], best_w[fi]);
    ++nw[b->fam[fi].waves];
  }
  // 2. steps per launch
  const int cands[] = {8, 32, 128};
  double best = 1e300;
  int bs = b->steps_per_launch;
  for (int cs : cands) {
    if (cs > trial_steps) continue;
    if ((rc = trial(cs, fam_ms, sec))) return rc;
    if (sec < best) {
      best = sec;
      bs = cs;
    }
  }
  b->steps_done = steps0;
  b->steps_per_launch = bs;
  if (best_steps) *best_steps = bs;
  if (best_waves)  // the most frequent choice (ties to the wider workgroup)
    *best_waves = (nw[8] >= nw[4] && nw[8] >= nw[2]) ? 8 : (nw[4] >= nw[2] ? 4 : 2);
  return batch_flags(b);
}

extern "C" int rp_batch_last_kernel_ms(rp_batch* b, double* avg_ms, int64_t* launches) {
  RP_REQUIRE(b && avg_ms, "rp_batch_last_kernel_ms: bad arguments");
  // per family: average duration of one launch of the fused kernel in the last run
  for (size_t fi = 0; fi < b->fam.size(); ++fi)
    avg_ms[fi] = b->last_launches ? b->fam_ms[fi] / b->last_launches : 0.0;
  if (launches) *launches = b->last_launches;
  return RP_OK;
}

extern "C" int rp_batch_family_shape(rp_batch* b, int fam, int* waves, int* units_per_wave,
                                     int* folded) {
  RP_REQUIRE(b && fam >= 0 && fam < (int)b->fam.size(), "rp_batch_family_shape: bad arguments");
  const Family& f = b->fam[fam];
  // units of 32 modes x 16 dofs over the wave budget
  const int units = (f.NPAD >> 5) * b->DT;
  if (waves) *waves = f.waves;
  if (units_per_wave) *units_per_wave = (units + f.waves - 1) / f.waves;
  if (folded) *folded = (f.N % 2 == 0) && b->pes->kind != PES_WATER;
  return RP_OK;
}

extern "C" int rp_batch_families(rp_batch* b, int* nfam, int* n, int* count) {
  RP_REQUIRE(b && nfam, "rp_batch_families: bad arguments");
  *nfam = (int)b->fam.size();
  for (size_t fi = 0; fi < b->fam.size(); ++fi) {
    if (n) n[fi] = b->fam[fi].N;
    if (count) count[fi] = b->fam[fi].count;
  }
  return RP_OK;
}
