// MI355X (gfx950) trial-move energy engine: host side of the C ABI declared
// in include/plum_gpu.h.  Kernels live in kernels_move.h / kernels_full.h.
//
// Data layout in HBM (one system per context):
//   beads (index order):  x,y,z current unwrapped FP64, q FP64, type, molecule
//   cell list:            per cell a high-water count and `cap` slots with
//                         slot-major copies of (wrapped x,y,z,q) as double4,
//                         a float4 copy relative to the cell origin for the
//                         FP32 path, the bead index (-1 = tombstone) and type
//   k space:              half-space k list (lx,ly,lz) int4, c_k FP64,
//                         running S(k) double2, pending dS(k) double2
//   pending move:         moved list (index, old/new position+charge) and the
//                         per-bead phase tables e^{i l theta_d}, |l| <= n_d
//   control block:        dipole moment, dipole lag state, running totals,
//                         the last dE per term, status flags, move counters
#include "kernels_batch.h"
#include "kernels_cbmc.h"
#include "kernels_grow.h"
#include "kernels_full.h"
#include "kernels_move.h"
#include "kernels_pressure.h"
#include "plum_gpu.h"
#include "surrogate.h"

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <mutex>
#include <random>
#include <string>
#include <vector>

using namespace plum;

struct plum_batch;
struct SurHost;
struct CbmcHost;
struct VpHost;
void cbmc_free(CbmcHost* h);
void vp_free(VpHost* h);
extern "C" int plum_batch_destroy(plum_batch* batch);
void sur_free(SurHost* s);

struct plum_ctx {
  plum_params p{};
  Geo g{};
  plum_info info{};
  Dev d{};
  hipStream_t st = nullptr;
  int device = 0;        // HIP device the context lives on
  int maxm = 1;          // capacity of the moved list (largest molecule)
  int nkb = 0;           // blocks of the k-space delta kernel (64 k each)
  int nkb_full = 0;      // blocks of the full S(k) kernels (256 k each)
  int nmmb = 1;          // blocks of the moved-moved pair work
  int nchunk = 1;        // bead chunks of the S(k) build
  int chunk = 512;
  int full_cells = 1, full_groups = 1, full_parts = 1;   // grid of the full real-space kernel
  size_t fpart_cap = 0;  // its partials allocated
  int *cell_list = nullptr, *cell_cnt = nullptr;   // its cells, where a block takes several (k_cell_scan)
  int cell_per = 0;      // list entries of a block (0: a block per cell)
  size_t list_cap = 0;
  int nsplit = 1;        // blocks per real-space query
  double cand = 0;       // expected candidate pair-images per query
  int cell_div = 2;      // cells per search radius and dimension
  int grid_gen = 0;      // bumped by every re-grid (batches re-upload their copies)
  int nkb_s = 0;         // k-space tiles of the speculative loop
  plum_batch* self = nullptr;  // this system as a batch of one (device loop)
  SurHost* sur = nullptr;      // delayed-acceptance surrogate (null when off)
  CbmcHost* cbmc = nullptr;    // configurational-bias trial buffers
  VpHost* vp = nullptr;        // volume-perturbation pressure buffers
  int screen_cap = kMaxProp;   // proposal slots allocated
  double self_img = 0;   // real-space energy of a unit charge and its own images
  double *epart_k = nullptr, *opart = nullptr;   // from-scratch k-space / springs, walls, self, dipole partials
  int *d_max = nullptr, *h_max = nullptr;        // largest cell count (device, pinned host)
  std::vector<int> mol_start;
  char* h_in = nullptr;  // pinned: trial coordinates, then bead indices of the caller's move
  HostRes* h_res = nullptr;  // pinned: results of the host path
  int seq = 0;               // its calls so far
  Ctl* h_ctl = nullptr;  // pinned copy of the control block
  size_t off_idx = 0;
  char* d_in = nullptr;
  int drec_cap = 0;      // decision-record capacity allocated (plum_mc_record)
  hipEvent_t ev_idle = nullptr;  // marks the end of the work queued on st
  bool pending = false;
  bool profiling = false;
  std::vector<void*> dev_allocs;
  // kernel timing (profiling mode of plum_mc_run)
  std::vector<std::string> kname;
  std::vector<double> ksum_us;
  std::vector<long long> kcount;
};

namespace {

thread_local std::string g_err;

int fail(int code, const std::string& msg) {
  g_err = msg;
  return code;
}

#define HIPCHK(x)                                                               \
  do {                                                                          \
    hipError_t e_ = (x);                                                        \
    if (e_ != hipSuccess)                                                       \
      return fail(PLUM_E_HIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
  } while (0)

#define CHK(x)                      \
  do {                              \
    int rc_ = (x);                  \
    if (rc_ != PLUM_OK) return rc_; \
  } while (0)

template <typename T>
int dalloc(plum_ctx* c, T** ptr, size_t count) {
  if (count == 0) count = 1;
  void* p = nullptr;
  hipError_t e = hipMalloc(&p, sizeof(T) * count);
  if (e != hipSuccess) return fail(PLUM_E_NOMEM, std::string("hipMalloc: ") + hipGetErrorString(e));
  c->dev_allocs.push_back(p);
  *ptr = static_cast<T*>(p);
  return PLUM_OK;
}

// Gives back a buffer of dalloc's before the context is destroyed.
template <typename T>
void dfree(plum_ctx* c, T** ptr) {
  auto& v = c->dev_allocs;
  const auto it = std::find(v.begin(), v.end(), (void*)*ptr);
  if (it != v.end()) {
    (void)hipFree(*it);
    v.erase(it);
  }
  *ptr = nullptr;
}

// potential_ewald_coul.cc:43-75: slab padding and the derived cutoffs.
void derive_cutoffs(const plum_params& p, plum_info& info) {
  double box[3] = {p.box[0], p.box[1], p.box[2]};
  if (p.dipole_correction) {
    const double min_padding = 150;
    if (box[2] * kDiCorrection > min_padding) box[2] = box[2] * kDiCorrection;
    else box[2] += min_padding;
  }
  for (int i = 0; i < 3; i++) info.box_e[i] = box[i];
  info.vol_e = box[0] * box[1] * box[2];
  if (!p.use_ewald) return;
  const double lB = p.lB, alpha = p.alpha;
  double real_cutoff = 1;
  while (0.5 * lB * 1 * 1 * erfc(sqrt(alpha) * real_cutoff) / real_cutoff > kEwaldCutoff)
    real_cutoff += 1;
  info.real_cutoff = real_cutoff;
  for (int i = 0; i < 3; i++) info.real_cell[i] = (int)ceil(real_cutoff / box[i]);
  double repl_cutoff = alpha;
  const double min_box_vol = pow(box[0], 3);
  while (lB * 1 * 1 / (2 * kPi * min_box_vol) * (4 * kPi * kPi) * exp(-repl_cutoff / (4 * alpha)) /
             repl_cutoff >
         kEwaldCutoff)
    repl_cutoff += alpha;
  info.repl_cutoff = repl_cutoff;
  for (int i = 0; i < 3; i++) info.repl_cell[i] = (int)ceil(sqrt(repl_cutoff) * box[i] / (2 * kPi));
}

// Real-space energy of a unit charge with its own images (half of each pair;
// potential_ewald_coul.cc:134-164 at separation 0) where the period along z is
// Lz: whole edges, exactly, since an edge may equal the cutoff (both are often
// whole numbers).
long double self_images(const plum_ctx* c, double Lz) {
  const Geo& g = c->g;
  if (!g.use_ewald) return 0;
  const long double sa = g.sqrt_alpha;
  long double e = 0;
  for (int i = -g.real_cell[0]; i <= g.real_cell[0]; i++)
    for (int j = -g.real_cell[1]; j <= g.real_cell[1]; j++)
      for (int k = -g.real_cell[2]; k <= g.real_cell[2]; k++) {
        const double x = i * g.L[0], y = j * g.L[1], z = k * Lz;
        const double r = sqrt(x * x + y * y + z * z);
        if (r > 0 && r <= g.rc) e += erfcl(sa * r) / r;
      }
  return 0.5L * g.lB * e;
}

// Most blocks of the full real-space kernel with a block per cell, and blocks
// where each takes several.
constexpr int kFullBlocks = 65536, kListBlocks = 8192;

// The cells of each block of the full real-space kernel (listed by scan_cells).
CellList full_cells(const plum_ctx* c) { return CellList{c->cell_list, c->cell_cnt, c->cell_per, c->full_cells}; }

// Partials of the full real-space kernel.
size_t full_partials(const plum_ctx* c) {
  return (size_t)c->full_cells * c->full_groups * c->full_parts * kQWaves;
}

// Builds the cell list from the current device positions, each cell's beads in
// index order (k_cell_*).  The largest count comes back to the host, which
// sizes the slots.
int build_cells(plum_ctx* c, int min_cap) {
  const Geo& g = c->g;
  const int nb = (g.n + kBlock - 1) / kBlock;
  HIPCHK(hipMemsetAsync(c->d.ccount, 0, sizeof(int) * g.ncell, c->st));
  HIPCHK(hipMemsetAsync(c->d_max, 0, sizeof(int), c->st));
  hipLaunchKernelGGL(k_cell_count, dim3(nb), dim3(kBlock), 0, c->st, g, c->d);
  hipLaunchKernelGGL(k_cell_max, dim3(std::min(64, (g.ncell + kBlock - 1) / kBlock)), dim3(kBlock), 0, c->st, g,
                     c->d, c->d_max);
  HIPCHK(hipGetLastError());
  HIPCHK(hipMemcpyAsync(c->h_max, c->d_max, sizeof(int), hipMemcpyDeviceToHost, c->st));
  HIPCHK(hipStreamSynchronize(c->st));
  const int maxc = *c->h_max;
  const int cap = std::max(std::max(16, min_cap), ((maxc * 2 + 8 + 7) / 8) * 8);
  const size_t slots = (size_t)g.ncell * cap;
  if (cap != c->g.cap || c->d.cbead == nullptr) {
    CHK(dalloc(c, &c->d.cbead, slots));
    CHK(dalloc(c, &c->d.cpos, slots));
    CHK(dalloc(c, &c->d.cpos32, slots));
    CHK(dalloc(c, &c->d.ctype, slots));
    c->g.cap = cap;
  }
  // from-scratch real space: block (residue of the cells, group of kCluster
  // slots, share of the query's cells).  Groups for the counts the list holds
  // now (a fuller cell's blocks take several), shares where few cells hold many
  // beads.  A block takes one cell while that needs no more than kFullBlocks
  // blocks and, past 1,024, two blocks a bead; else the cells are listed without
  // the empty ones and dealt to fewer blocks: a block for each of 2.1 million
  // cells, and its partials in the final sum, took 2.1 ms for 800 beads, 63 us now.
  c->full_groups = std::max(1, std::min((maxc + kCluster - 1) / kCluster, 65535));
  const long long most = std::max(1024LL, 2LL * g.n);
  c->full_cells = g.ncell;
  if (g.ncell > most || (long long)g.ncell * c->full_groups > kFullBlocks)
    c->full_cells = (int)std::min({(long long)g.ncell, most, std::max(1024LL, (long long)kListBlocks / c->full_groups)});
  const long long blocks = (long long)c->full_cells * c->full_groups;
  c->full_parts = (int)std::max(1LL, std::min<long long>(kMaxQBlock, std::min<long long>(
                      4096 / blocks, (long long)(c->cand / kQShare))));
  c->cell_per = c->full_cells < g.ncell ? (g.ncell + c->full_cells - 1) / c->full_cells : 0;
  const size_t nl = (size_t)c->full_cells * (c->cell_per + 1);
  if (c->cell_per && nl > c->list_cap) {
    c->list_cap = 0;
    dfree(c, &c->cell_list);
    CHK(dalloc(c, &c->cell_list, nl));
    c->list_cap = nl;
  }
  c->cell_cnt = c->cell_per ? c->cell_list + (size_t)c->full_cells * c->cell_per : nullptr;
  const size_t fp = full_partials(c);
  if (fp > c->fpart_cap) {
    CHK(dalloc(c, &c->d.fpart, fp));
    c->fpart_cap = fp;
  }
  HIPCHK(hipMemsetAsync(c->d.ccount, 0, sizeof(int) * g.ncell, c->st));
  hipLaunchKernelGGL(k_cell_fill, dim3(nb), dim3(kBlock), 0, c->st, g, c->d);
  hipLaunchKernelGGL(k_cell_order, dim3(g.ncell), dim3(kBlock), 0, c->st, g, c->d);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(c->st));
  c->info.cell_cap = cap;
  return PLUM_OK;
}

int split_for(double cand, int split_div) {
  return std::max(1, std::min(kMaxSplit, (int)std::lround(cand / split_div)));
}

// Cell grid of edge ~ rs / div in every dimension (at most 256 cells each).
void set_cell_grid(plum_ctx* c, int div) {
  Geo& g = c->g;
  for (int k = 0; k < 3; k++) {
    int nc = (int)floor(g.L[k] / (g.rs / div));
    nc = std::max(1, std::min(nc, 256));
    g.nc[k] = nc;
    g.h[k] = g.L[k] / nc;
    g.inv_h[k] = 1.0 / g.h[k];
    c->info.n_cells[k] = nc;
  }
  g.ncell = g.nc[0] * g.nc[1] * g.nc[2];
  c->cell_div = div;
}

// Expected candidate slots of a real-space query (the cells within the search
// radius of a point) and the query split it gives.  With two periodic
// dimensions the beads fill the simulation box only, not the padding of the
// Ewald box (a brush 40 high in a box of 190: 16,600 candidates, not 3,500).
void set_cand(plum_ctx* c) {
  const Geo& g = c->g;
  double cand = g.n;
  for (int k = 0; k < 3; k++) {
    const double w = 2 * g.rs + g.h[k];
    cand *= k < g.npbc ? w / g.L[k] : std::min(1.0, w / g.Lsim[k]);
  }
  c->cand = cand;
  c->nsplit = split_for(cand, kDefaultSplitDiv);
}

// A new cell grid for the current positions: the cell list rebuilt from
// scratch (the old arrays stay allocated until the context is destroyed).
int regrid_cells(plum_ctx* c, int div) {
  if (div == c->cell_div) return PLUM_OK;
  HIPCHK(hipStreamSynchronize(c->st));
  const int old_ncell = c->g.ncell;
  set_cell_grid(c, div);
  if (c->g.ncell != old_ncell) CHK(dalloc(c, &c->d.ccount, c->g.ncell));
  c->d.cbead = nullptr;   // slot arrays sized for the new grid
  set_cand(c);
  CHK(build_cells(c, 0));
  c->grid_gen++;
  return PLUM_OK;
}

constexpr int kFullSmall = 128;   // blocks of k_full_small

// From-scratch energy on the device; with set_running the running totals,
// dipole state and the per-molecule spring cache are reset to it.
int run_full(plum_ctx* c, int set_running, double out[8]) {
  const Geo& g = c->g;
  const CellList cl = full_cells(c);
  if (cl.per) hipLaunchKernelGGL(k_cell_scan, dim3(c->full_cells), dim3(kBlock), 0, c->st, g, c->d, cl);
  hipLaunchKernelGGL(k_full_real, dim3(c->full_cells, c->full_groups, c->full_parts), dim3(kBlock), 0, c->st, g, c->d,
                     cl, c->full_parts);
  const bool ksp = g.use_ewald && g.n_kh > 0;
  if (ksp) {
    // by tiles where a step of four beads' tables fits the LDS stage
    if (sk_sub(g.tab_w) >= 4)
      hipLaunchKernelGGL(k_full_sk_tile, dim3((c->nkb_s + kQWaves - 1) / kQWaves, c->nchunk), dim3(kBlock), 0, c->st,
                         g, c->d, c->chunk, c->nkb_s);
    else
      hipLaunchKernelGGL(k_full_sk_part, dim3(c->nkb_full, c->nchunk), dim3(kBlock), 0, c->st, g, c->d, c->chunk);
    hipLaunchKernelGGL(k_full_sk_reduce, dim3(c->nkb_full), dim3(kBlock), 0, c->st, g, c->d, c->nchunk,
                       c->epart_k);
  }
  hipLaunchKernelGGL(k_full_small, dim3(kFullSmall), dim3(kBlock), 0, c->st, g, c->d, (int)full_partials(c),
                     c->self_img, c->opart);
  hipLaunchKernelGGL(k_full_final, dim3(1), dim3(kFinalThreads), 0, c->st, g, c->d, ksp ? c->nkb_full : 0,
                     kFullSmall, c->epart_k, c->opart, set_running);
  HIPCHK(hipGetLastError());
  HIPCHK(hipMemcpyAsync(c->h_ctl, c->d.ctl, sizeof(Ctl), hipMemcpyDeviceToHost, c->st));
  HIPCHK(hipStreamSynchronize(c->st));
  for (int k = 0; k < 8; k++) out[k] = c->h_ctl->full[k];
  return PLUM_OK;
}

void to_terms(const double t[8], plum_terms* o) {
  o->lj = t[T_LJ]; o->real = t[T_REAL]; o->kspace = t[T_KSPACE]; o->self = t[T_SELF];
  o->dipole = t[T_DIPOLE]; o->bond = t[T_BOND]; o->wall = t[T_WALL];
}

int validate(const plum_params* p, int n, const double* xyz, const double* q, const int* type,
             int n_mols, const int* ms) {
  if (!p || !xyz || !q || !type || !ms) return fail(PLUM_E_ARG, "null argument");
  if (n <= 0 || n_mols <= 0) return fail(PLUM_E_ARG, "empty system");
  if (p->npbc != 2 && p->npbc != 3)
    return fail(PLUM_E_ARG, "npbc must be 2 or 3 (simulation.cc:152-156)");
  if (p->npbc == 3 && p->dipole_correction)
    return fail(PLUM_E_UNSUPPORTED, "dipole correction with 3 periodic dimensions");
  if (!(p->beta > 0)) return fail(PLUM_E_ARG, "beta must be > 0 (simulation.cc:142-146)");
  for (int k = 0; k < 3; k++)
    if (!(p->box[k] > 0) || !std::isfinite(p->box[k])) return fail(PLUM_E_ARG, "box lengths must be > 0");
  if (p->n_types <= 0 || p->n_types > PLUM_MAX_TYPES) return fail(PLUM_E_ARG, "n_types out of range");
  if (p->use_ewald && !(p->alpha > 0 && p->lB >= 0)) return fail(PLUM_E_ARG, "Ewald alpha must be > 0");
  if (p->precision != PLUM_FP64 && p->precision != PLUM_FP32_PAIR)
    return fail(PLUM_E_ARG, "unknown precision");
  if (ms[0] != 0 || ms[n_mols] != n) return fail(PLUM_E_ARG, "mol_start must span 0..n_beads");
  for (int m = 0; m < n_mols; m++) {
    if (ms[m + 1] <= ms[m]) return fail(PLUM_E_ARG, "empty or unordered molecule");
    if (ms[m + 1] - ms[m] > kMaxChainDev)
      return fail(PLUM_E_UNSUPPORTED, "molecule longer than 2048 beads");
  }
  for (int i = 0; i < n; i++) {
    if (type[i] < 0 || type[i] >= p->n_types) return fail(PLUM_E_ARG, "bead type out of range");
    for (int k = 0; k < 3; k++)
      if (!std::isfinite(xyz[3 * (size_t)i + k])) return fail(PLUM_E_ARG, "non-finite coordinate");
    if (!std::isfinite(q[i])) return fail(PLUM_E_ARG, "non-finite charge");
  }
  return PLUM_OK;
}

int nmm_for(const plum_ctx*, int nm) { return nmm_blocks(nm); }

// Waits until the kernel of host-path call `seq` has written its results to
// c->h_res: polled for a while (a call takes tens of microseconds), then by
// the stream, which also reports a kernel that failed.
int host_wait(plum_ctx* c, int seq) {
  const auto t0 = std::chrono::steady_clock::now();
  for (int i = 1;; i++) {
    if (__atomic_load_n(&c->h_res->seq, __ATOMIC_ACQUIRE) == seq) return PLUM_OK;
    if (i % 64 == 0 && std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(2)) break;
  }
  HIPCHK(hipStreamSynchronize(c->st));
  if (__atomic_load_n(&c->h_res->seq, __ATOMIC_ACQUIRE) != seq) return fail(PLUM_E_HIP, "trial-move kernel did not finish");
  return PLUM_OK;
}

// k-space and real-space work of one trial move in one launch, once the
// moved list (and, for the k space, the phase tables) exists on the device.
// nm is the exact count (host path) or the capacity (device loop; the
// kernels read the real count on the device).
void launch_compute(plum_ctx* c, int nm) {
  const Geo& g = c->g;
  const int nkb = (g.use_ewald && g.n_kh > 0) ? c->nkb : 0;
  const int nmm = nmm_for(c, nm);
  const int nreal = 2 * nm * c->nsplit;
  const int grid = nkb + nreal + nmm;
  if (c->p.precision == PLUM_FP32_PAIR)
    hipLaunchKernelGGL(k_compute<1>, dim3(grid), dim3(kBlock), 0, c->st, g, c->d, nkb, nreal, nmm, c->nsplit);
  else
    hipLaunchKernelGGL(k_compute<0>, dim3(grid), dim3(kBlock), 0, c->st, g, c->d, nkb, nreal, nmm, c->nsplit);
}

}  // namespace

extern "C" {

const char* plum_last_error(void) { return g_err.c_str(); }

int plum_create(const plum_params* params, int n, const double* xyz, const double* q, const int* type,
                int n_mols, const int* ms, plum_ctx** out) {
  if (!out) return fail(PLUM_E_ARG, "null output");
  *out = nullptr;
  CHK(validate(params, n, xyz, q, type, n_mols, ms));
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return fail(PLUM_E_HIP, "no HIP device available");
  plum_ctx* c = new plum_ctx();
  c->p = *params;
  const plum_params& p = c->p;
  int rc = PLUM_OK;
  auto bail = [&](int code) {
    plum_destroy(c);
    return code;
  };
  plum_info& info = c->info;
  derive_cutoffs(p, info);
  Geo& g = c->g;
  for (int k = 0; k < 3; k++) {
    g.L[k] = info.box_e[k];
    g.Lsim[k] = p.box[k];
    g.inv_L[k] = 1.0 / g.L[k];
  }
  g.npbc = p.npbc;
  g.n = n;
  g.n_mols = n_mols;
  g.beta = p.beta;
  g.use_pair = p.use_pair;
  g.use_ewald = p.use_ewald;
  g.use_bond = p.use_bond;
  g.use_ext = p.use_ext;
  g.n_types = p.n_types;
  g.rc = p.use_ewald ? info.real_cutoff : 0;
  g.sqrt_alpha = p.use_ewald ? sqrt(p.alpha) : 0;
  g.lB = p.lB;
  g.self_coef = p.use_ewald ? -p.lB * sqrt(p.alpha / kPi) : 0;
  g.dip_coef = p.lB * 2 * kPi / (info.vol_e / 1.0);
  for (int k = 0; k < 3; k++) g.real_cell[k] = info.real_cell[k];
  g.k_bond = p.k_bond;
  g.r0 = p.r0;
  g.wall_cut = p.wall_cut;
  g.wall_r3_k213 = pow((1.0 / k213), 3);
  g.wall_r3_cut = pow((1.0 / p.wall_cut), 3);
  g.dipole = p.use_ewald && p.dipole_correction;
  g.dipole_exact = p.dipole_exact;

  // LJ pair table with the reference's expressions (potential_truncated_lj.cc:49-85)
  std::vector<LJPair> lj((size_t)p.n_types * p.n_types);
  std::vector<LJPair32> lj32(lj.size());
  double lj_max = 0;
  for (int a = 0; a < p.n_types; a++)
    for (int b = 0; b < p.n_types; b++) {
      LJPair& e = lj[(size_t)a * p.n_types + b];
      e.sigma = (p.lj_sigma[a] + p.lj_sigma[b]) / 2;
      e.eps = sqrt((p.lj_eps[a] * p.lj_eps[b]));
      if (p.lj_cutoff < 0) {
        const double r6_ref = pow((1.0 / k216), 6);
        e.shift = 4 * e.eps * (r6_ref * r6_ref - r6_ref);
        e.cut = k216 * e.sigma;
      } else {
        const double r6_ref = pow((e.sigma / p.lj_cutoff), 6);
        e.shift = 4 * e.eps * (r6_ref * r6_ref - r6_ref);
        e.cut = p.lj_cutoff;
      }
      LJPair32& f = lj32[(size_t)a * p.n_types + b];
      f.sigma2 = (float)(e.sigma * e.sigma);
      f.eps4 = (float)(4 * e.eps);
      f.cut = e.cut;
      f.shift = (float)e.shift;
      if (p.use_pair) lj_max = std::max(lj_max, e.cut);
    }
  for (int k = 0; k < p.npbc; k++)
    if (p.use_pair && !(p.box[k] > 2 * lj_max)) {
      delete c;
      return fail(PLUM_E_UNSUPPORTED, "periodic box shorter than twice the LJ cutoff");
    }
  std::vector<WallType> wall(p.n_types);
  for (int t = 0; t < p.n_types; t++) {
    wall[t].sigma = p.wall_sigma[t];
    wall[t].eps = p.wall_eps[t];
    wall[t].kind = p.type_kind[t];
    wall[t].pad = 0;
  }
  // FP32 path: pairs closer than 1.3 x the largest LJ sigma (the steep,
  // large close-contact terms), and pairs whose real-space term for unit
  // charges exceeds 3e-3 kT, are evaluated in FP64.  FP32 pair math carries
  // ~1e-7 of relative error per pair; summed over the ~10^5 pair images of a
  // long chain's move (old and new) the large near terms would leave ~1e-5 kT
  // of error in dE, the small far ones leave < 1e-6 kT.
  double sig_max = 0;
  for (int t = 0; t < p.n_types; t++) sig_max = std::max(sig_max, p.lj_sigma[t]);
  double r_u = 0;
  if (p.use_ewald && p.lB > 0) {
    const double sa = sqrt(p.alpha);
    r_u = 0.05;
    while (r_u < info.real_cutoff && p.lB * erfc(sa * r_u) / r_u > 3e-3) r_u += 0.05;
  }
  g.fp64_below = std::max(1.3 * std::max(sig_max, 0.0), r_u);
  // explicit pair sums need only the minimum image when no other image can
  // reach rc along a periodic edge (edges longer than 2 rc); a non-periodic z
  // is checked per pair (real_pair)
  g.single_image = p.use_ewald ? 1 : 0;
  for (int k = 0; k < p.npbc && p.use_ewald; k++)
    if (!(2 * g.rc * (1 + 1e-9) < g.L[k])) g.single_image = 0;
  g.rs = std::max(g.rc, lj_max);
  if (g.rs <= 0) g.rs = 1.0;
  g.rs2 = g.rs * g.rs;
  g.lj2_max = lj_max * lj_max * (1 + 1e-12);
  c->self_img = (double)self_images(c, g.L[2]);

  // cell grid: edge ~ rs / div
  set_cell_grid(c, p.cell_div > 0 ? p.cell_div : 2);

  // half-space k list (potential_ewald_coul.cc:78-115; k and -k paired)
  std::vector<int4> kl;
  std::vector<double> ck;
  info.n_k_full = 0;
  if (p.use_ewald) {
    const int* n3 = info.repl_cell;
    g.nkx = n3[0]; g.nky = n3[1]; g.nkz = n3[2];
    const double pref0 = p.lB / (kPi * info.vol_e) * (4 * kPi * kPi);
    for (int lx = -n3[0]; lx <= n3[0]; lx++)
      for (int ly = -n3[1]; ly <= n3[1]; ly++)
        for (int lz = -n3[2]; lz <= n3[2]; lz++) {
          const double kx = (double)(lx * 2) * kPi / g.L[0];
          const double ky = (double)(ly * 2) * kPi / g.L[1];
          const double kz = (double)(lz * 2) * kPi / g.L[2];
          const double k2 = kx * kx + ky * ky + kz * kz;
          if (!(k2 > 0 && k2 <= info.repl_cutoff)) continue;
          info.n_k_full++;
          const bool half = lx > 0 || (lx == 0 && (ly > 0 || (ly == 0 && lz > 0)));
          if (!half) continue;
          kl.push_back(make_int4(lx, ly, lz, 0));
          ck.push_back(pref0 * (exp(-k2 / (4 * p.alpha)) / k2));
        }
    g.tab_w = (g.nkx + 1) + (g.nky + 1) + (g.nkz + 1);
  }
  g.n_kh = (int)kl.size();
  info.n_k_half = g.n_kh;
  // rows of one (l_x, l_y) with their l_z from -m to m (the l_x = l_y = 0 row:
  // 1 to m; the list has l_z fastest and the cutoff takes both signs), longest
  // first so that the 16 rows of a tile need about the same l_z, and the tiles
  // of the speculative k-space
  std::vector<int4> krow;
  for (int k = 0; k < g.n_kh;) {
    int e = k;
    while (e < g.n_kh && kl[e].x == kl[k].x && kl[e].y == kl[k].y) e++;
    krow.push_back(make_int4(kl[k].x, kl[k].y, k, kl[e - 1].z));
    k = e;
  }
  std::stable_sort(krow.begin(), krow.end(), [](const int4& a, const int4& b) { return a.w > b.w; });
  while (krow.size() % kKTile) krow.push_back(make_int4(0, 0, 0, -1));
  std::vector<int2> ktile;
  for (size_t r = 0; r < krow.size(); r += kKTile)
    for (int z = 0; z <= krow[r].w; z += kKTile) ktile.push_back(make_int2((int)r, z));
  c->nkb_s = p.use_ewald ? (int)ktile.size() : 0;
  c->nkb = std::max(1, (g.n_kh + kKPerBlock - 1) / kKPerBlock);
  c->nkb_full = std::max(1, (g.n_kh + kBlock - 1) / kBlock);

  c->mol_start.assign(ms, ms + n_mols + 1);
  int maxm = 1;
  for (int m = 0; m < n_mols; m++) maxm = std::max(maxm, ms[m + 1] - ms[m]);
  c->maxm = maxm;
  info.n_beads = n;
  info.n_mols = n_mols;
  info.max_mol_len = maxm;
  c->nmmb = nmm_blocks(maxm);
  // bead chunks of the S(k) build: about 512 blocks over the groups of four
  // tiles, 64 to 512 beads each
  {
    const int groups = std::max(1, (c->nkb_s + kQWaves - 1) / kQWaves), want = std::max(1, 512 / groups);
    c->chunk = std::max(64, std::min(512, ((n + want - 1) / want + 63) / 64 * 64));
  }
  c->nchunk = (n + c->chunk - 1) / c->chunk;

  if (hipGetDevice(&c->device) != hipSuccess || hipStreamCreate(&c->st) != hipSuccess) {
    delete c;
    return fail(PLUM_E_HIP, "hipStreamCreate failed");
  }
  if (hipEventCreateWithFlags(&c->ev_idle, hipEventDisableTiming) != hipSuccess) {
    (void)hipStreamDestroy(c->st);
    delete c;
    return fail(PLUM_E_HIP, "hipEventCreate failed");
  }
  Dev& d = c->d;
  std::vector<double> hx(n), hy(n), hz(n);
  std::vector<int> mol_of(n);
  for (int i = 0; i < n; i++) {
    hx[i] = xyz[3 * (size_t)i]; hy[i] = xyz[3 * (size_t)i + 1]; hz[i] = xyz[3 * (size_t)i + 2];
  }
  for (int m = 0; m < n_mols; m++)
    for (int i = ms[m]; i < ms[m + 1]; i++) mol_of[i] = m;
#define ALLOC(ptr, cnt) if ((rc = dalloc(c, &ptr, cnt)) != PLUM_OK) return bail(rc)
  ALLOC(d.x, n); ALLOC(d.y, n); ALLOC(d.z, n); ALLOC(d.q, n);
  ALLOC(d.type, n); ALLOC(d.mol_of, n); ALLOC(d.mol_start, n_mols + 1);
  ALLOC(d.bcell, n); ALLOC(d.bslot, n); ALLOC(d.moved, n); ALLOC(d.mv_slot, n);
  ALLOC(d.ccount, g.ncell);
  // per-proposal slots (kMaxProp) for the speculative device loop; the host
  // path uses slot 0
  ALLOC(d.kl, g.n_kh); ALLOC(d.ck, g.n_kh); ALLOC(d.Sk, g.n_kh); ALLOC(d.dS, (size_t)kMaxProp * g.n_kh);
  ALLOC(d.tab, (size_t)kMaxProp * maxm * 2 * std::max(1, g.tab_w));
  ALLOC(d.lj, lj.size()); ALLOC(d.lj32, lj32.size()); ALLOC(d.wall, wall.size());
  ALLOC(d.bond_cur, n_mols);
  ALLOC(d.mv_old, (size_t)kMaxProp * maxm); ALLOC(d.mv_new, (size_t)kMaxProp * maxm);
  ALLOC(d.mv_type, (size_t)kMaxProp * maxm);
  ALLOC(d.recs, kMaxScreen); ALLOC(d.smv_idx, (size_t)kMaxProp * maxm);
  ALLOC(d.prop, kMaxScreen); ALLOC(d.plan, 1);
  ALLOC(d.krow, krow.size()); ALLOC(d.ktile, ktile.size());
  // erfc nodes {erfc(x_i), (2 / sqrt(pi)) exp(-x_i^2)}, x_i = i / kErfcPerUnit,
  // each rounded once from long double (erfc_nodes)
  std::vector<double2> erfc_h(kErfcNodes);
  for (int i = 0; i < kErfcNodes; i++) {
    const long double x = (long double)i / kErfcPerUnit;
    erfc_h[i] = make_double2((double)erfcl(x), (double)(2.0L / sqrtl(3.141592653589793238462643383279502884L) *
                                                        expl(-x * x)));
  }
  double2* erfc_d = nullptr;
  ALLOC(erfc_d, kErfcNodes);
  g.erfc_tab = erfc_d;
  std::vector<float2> erfc32_h(kErfcNodes);
  for (int i = 0; i < kErfcNodes; i++) erfc32_h[i] = make_float2((float)erfc_h[i].x, (float)erfc_h[i].y);
  float2* erfc32_d = nullptr;
  ALLOC(erfc32_d, kErfcNodes);
  g.erfc_tab32 = erfc32_d;
  ALLOC(d.part_ks, (size_t)kMaxProp * std::max(1, c->nkb_s) * kQWaves);
  ALLOC(d.part_x, kMaxPairs * cross_blocks(maxm, maxm));
  ALLOC(d.ctl, 1);
  set_cand(c);
  // room for any split (the batch autotuner may change it)
  ALLOC(d.part_k, c->nkb); ALLOC(d.part_r, (size_t)kMaxProp * std::max(query_blocks(maxm, kMaxQBlock) * kQWaves, 2 * maxm * kMaxSplit));
  ALLOC(d.part_mm, (size_t)kMaxProp * c->nmmb);
  ALLOC(d.sk_part, (size_t)c->nchunk * std::max(1, g.n_kh));
  ALLOC(c->epart_k, c->nkb_full); ALLOC(c->opart, kSmallSums * kFullSmall); ALLOC(c->d_max, 1);
  ALLOC(d.chain_ids, n_mols); ALLOC(d.ion_ids, n_mols);
  {
    // move record of the host path: header, then the bead indices
    char* din = nullptr;
    ALLOC(din, sizeof(MoveRec) + sizeof(int) * maxm);
    c->d_in = din;
    d.rec = reinterpret_cast<MoveRec*>(din);
    d.mv_idx = reinterpret_cast<int*>(din + sizeof(MoveRec));
  }
  c->off_idx = sizeof(double) * 3 * maxm;
#undef ALLOC
  if (hipHostMalloc((void**)&c->h_in, c->off_idx + sizeof(int) * maxm, hipHostMallocCoherent) != hipSuccess ||
      hipHostMalloc((void**)&c->h_res, sizeof(HostRes), hipHostMallocCoherent) != hipSuccess ||
      hipHostMalloc((void**)&c->h_max, sizeof(int), hipHostMallocDefault) != hipSuccess ||
      hipHostMalloc((void**)&c->h_ctl, sizeof(Ctl), hipHostMallocDefault) != hipSuccess)
    return bail(fail(PLUM_E_NOMEM, "hipHostMalloc failed"));
  std::memset(c->h_res, 0, sizeof(HostRes));
  auto up = [&](void* dst, const void* src, size_t bytes) -> int {
    if (bytes == 0) return PLUM_OK;
    HIPCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, c->st));
    return PLUM_OK;
  };
  if ((rc = up(d.x, hx.data(), sizeof(double) * n)) || (rc = up(d.y, hy.data(), sizeof(double) * n)) ||
      (rc = up(d.z, hz.data(), sizeof(double) * n)) || (rc = up(d.q, q, sizeof(double) * n)) ||
      (rc = up(d.type, type, sizeof(int) * n)) || (rc = up(d.mol_of, mol_of.data(), sizeof(int) * n)) ||
      (rc = up(d.mol_start, ms, sizeof(int) * (n_mols + 1))) ||
      (rc = up(d.kl, kl.data(), sizeof(int4) * kl.size())) ||
      (rc = up(d.krow, krow.data(), sizeof(int4) * krow.size())) ||
      (rc = up(d.ktile, ktile.data(), sizeof(int2) * ktile.size())) ||
      (rc = up(d.ck, ck.data(), sizeof(double) * ck.size())) ||
      (rc = up(d.lj, lj.data(), sizeof(LJPair) * lj.size())) ||
      (rc = up(d.lj32, lj32.data(), sizeof(LJPair32) * lj32.size())) ||
      (rc = up(d.wall, wall.data(), sizeof(WallType) * wall.size())) ||
      (rc = up(erfc_d, erfc_h.data(), sizeof(double2) * kErfcNodes)) ||
      (rc = up(erfc32_d, erfc32_h.data(), sizeof(float2) * kErfcNodes)))
    return bail(rc);
  if (hipMemsetAsync(d.moved, 0, n, c->st) != hipSuccess ||
      hipMemsetAsync(d.mv_slot, 0xff, sizeof(int) * n, c->st) != hipSuccess ||
      hipMemsetAsync(d.ctl, 0, sizeof(Ctl), c->st) != hipSuccess ||
      hipMemsetAsync(d.plan, 0, sizeof(SpecPlan), c->st) != hipSuccess ||
      hipMemsetAsync(d.recs, 0, sizeof(MoveRec) * kMaxScreen, c->st) != hipSuccess ||
      hipMemsetAsync(c->d_in, 0, sizeof(MoveRec) + sizeof(int) * maxm, c->st) != hipSuccess)
    return bail(fail(PLUM_E_HIP, "hipMemsetAsync failed"));
  if ((rc = build_cells(c, 0)) != PLUM_OK) return bail(rc);
  double f[8];
  if ((rc = run_full(c, 1, f)) != PLUM_OK) return bail(rc);
  *out = c;
  return PLUM_OK;
}

int plum_destroy(plum_ctx* c) {
  if (!c) return PLUM_OK;
  // Teardown order: drain the context stream first (a rollback's commit
  // kernel may still be queued on it), then the device-loop batch (it drains
  // its own stream before destroying its graph), then the growth graph and
  // the surrogate, and only then the buffers those graphs and kernels read.
  if (c->st) (void)hipStreamSynchronize(c->st);
  if (c->self) plum_batch_destroy(c->self);
  c->self = nullptr;
  if (c->cbmc) cbmc_free(c->cbmc);
  c->cbmc = nullptr;
  if (c->sur) sur_free(c->sur);
  c->sur = nullptr;
  if (c->vp) vp_free(c->vp);
  c->vp = nullptr;
  for (void* p : c->dev_allocs) (void)hipFree(p);
  if (c->h_in) (void)hipHostFree(c->h_in);
  if (c->h_res) (void)hipHostFree(c->h_res);
  if (c->h_ctl) (void)hipHostFree(c->h_ctl);
  if (c->h_max) (void)hipHostFree(c->h_max);
  if (c->ev_idle) (void)hipEventDestroy(c->ev_idle);
  if (c->st) (void)hipStreamDestroy(c->st);
  delete c;
  return PLUM_OK;
}

int plum_get_info(const plum_ctx* c, plum_info* out) {
  if (!c || !out) return fail(PLUM_E_ARG, "null argument");
  *out = c->info;
  return PLUM_OK;
}

int plum_energy_full(plum_ctx* c, plum_terms* out) {
  if (!c || !out) return fail(PLUM_E_ARG, "null argument");
  if (c->pending) return fail(PLUM_E_STATE, "a trial move is pending finalize");
  double f[8];
  CHK(run_full(c, 0, f));
  to_terms(f, out);
  return PLUM_OK;
}

int plum_energy_difference(plum_ctx* c, int mol, int n_moved, const int* idx, const double* trial_xyz,
                           plum_terms* dE, double* total) {
  if (!c) return fail(PLUM_E_ARG, "null context");
  if (c->pending) return fail(PLUM_E_STATE, "previous trial move not finalized");
  if (mol < 0 || mol >= c->g.n_mols) return fail(PLUM_E_ARG, "molecule index out of range");
  const int a = c->mol_start[mol], b = c->mol_start[mol + 1];
  if (n_moved < 0 || n_moved > b - a) return fail(PLUM_E_ARG, "n_moved out of range");
  if (n_moved > 0 && (!idx || !trial_xyz)) return fail(PLUM_E_ARG, "null moved list");
  std::vector<char> seen(b - a, 0);
  for (int k = 0; k < n_moved; k++) {
    if (idx[k] < a || idx[k] >= b) return fail(PLUM_E_ARG, "moved bead not in the molecule");
    if (seen[idx[k] - a]++) return fail(PLUM_E_ARG, "moved bead listed twice");
    for (int e = 0; e < 3; e++)
      if (!std::isfinite(trial_xyz[3 * k + e])) return fail(PLUM_E_ARG, "non-finite trial coordinate");
  }
  MoveRec r{};
  r.n_moved = n_moved;
  r.mol = mol;
  r.move_type = -1;
  r.valid = 1;
  int lo = b, hi = a - 1;
  for (int k = 0; k < n_moved; k++) {
    lo = std::min(lo, idx[k]);
    hi = std::max(hi, idx[k]);
  }
  r.contig = (n_moved > 0 && hi - lo + 1 == n_moved) ? 1 : 0;
  r.lo = lo;
  r.hi = hi;
  int* h_idx = reinterpret_cast<int*>(c->h_in + c->off_idx);
  double* h_xyz = reinterpret_cast<double*>(c->h_in);
  if (n_moved > 0) {
    std::memcpy(h_idx, idx, sizeof(int) * n_moved);
    std::memcpy(h_xyz, trial_xyz, sizeof(double) * 3 * n_moved);
  }
  const Geo& g = c->g;
  hipLaunchKernelGGL(k_host_move, dim3(std::max(1, (n_moved + kHostBeads - 1) / kHostBeads)), dim3(kBlock), 0, c->st,
                     g, c->d, r, h_idx, h_xyz);
  launch_compute(c, n_moved);
  const int seq = ++c->seq;
  hipLaunchKernelGGL(k_epilogue, dim3(1), dim3(kBlock), 0, c->st, g, c->d,
                     (g.use_ewald && g.n_kh > 0) ? c->nkb : 0, 2 * n_moved * c->nsplit, nmm_for(c, n_moved),
                     c->h_res, seq);
  HIPCHK(hipGetLastError());
  CHK(host_wait(c, seq));
  c->pending = true;
  if (dE) to_terms(c->h_res->terms, dE);
  if (total) *total = c->h_res->total;
  return PLUM_OK;
}

int plum_finalize(plum_ctx* c, int accept) {
  if (!c) return fail(PLUM_E_ARG, "null context");
  if (!c->pending) return fail(PLUM_E_STATE, "no pending trial move");
  const Geo& g = c->g;
  const int seq = accept ? ++c->seq : c->seq;
  hipLaunchKernelGGL(k_commit, dim3(g.use_ewald && g.n_kh > 0 && accept ? 1 + c->nkb_full : 1), dim3(kBlock), 0, c->st,
                     g, c->d, accept ? 1 : 0, c->h_res, seq);
  HIPCHK(hipGetLastError());
  c->pending = false;
  if (accept) {
    CHK(host_wait(c, seq));
    if (c->h_res->overflow) {
      // a cell ran out of slots: rebuild with twice the capacity
      HIPCHK(hipStreamSynchronize(c->st));
      int zero = 0;
      HIPCHK(hipMemcpyAsync(&c->d.ctl->overflow, &zero, sizeof(int), hipMemcpyHostToDevice, c->st));
      CHK(build_cells(c, 2 * c->g.cap));
    }
  }
  return PLUM_OK;
}

int plum_totals(plum_ctx* c, plum_terms* out) {
  if (!c || !out) return fail(PLUM_E_ARG, "null argument");
  HIPCHK(hipMemcpyAsync(c->h_ctl, c->d.ctl, sizeof(Ctl), hipMemcpyDeviceToHost, c->st));
  HIPCHK(hipStreamSynchronize(c->st));
  to_terms(c->h_ctl->running, out);
  return PLUM_OK;
}

int plum_resync(plum_ctx* c, plum_terms* drift) {
  if (!c) return fail(PLUM_E_ARG, "null context");
  if (c->pending) return fail(PLUM_E_STATE, "a trial move is pending finalize");
  HIPCHK(hipMemcpyAsync(c->h_ctl, c->d.ctl, sizeof(Ctl), hipMemcpyDeviceToHost, c->st));
  HIPCHK(hipStreamSynchronize(c->st));
  double before[8];
  for (int k = 0; k < 8; k++) before[k] = c->h_ctl->running[k];
  int zero = 0;
  HIPCHK(hipMemcpyAsync(&c->d.ctl->overflow, &zero, sizeof(int), hipMemcpyHostToDevice, c->st));
  CHK(build_cells(c, c->g.cap));
  double f[8];
  CHK(run_full(c, 1, f));
  if (drift) {
    double dd[8];
    for (int k = 0; k < 8; k++) dd[k] = before[k] - f[k];
    to_terms(dd, drift);
  }
  return PLUM_OK;
}

int plum_get_positions(plum_ctx* c, double* xyz) {
  if (!c || !xyz) return fail(PLUM_E_ARG, "null argument");
  const int n = c->g.n;
  std::vector<double> x(n), y(n), z(n);
  HIPCHK(hipMemcpyAsync(x.data(), c->d.x, sizeof(double) * n, hipMemcpyDeviceToHost, c->st));
  HIPCHK(hipMemcpyAsync(y.data(), c->d.y, sizeof(double) * n, hipMemcpyDeviceToHost, c->st));
  HIPCHK(hipMemcpyAsync(z.data(), c->d.z, sizeof(double) * n, hipMemcpyDeviceToHost, c->st));
  HIPCHK(hipStreamSynchronize(c->st));
  for (int i = 0; i < n; i++) {
    xyz[3 * (size_t)i] = x[i]; xyz[3 * (size_t)i + 1] = y[i]; xyz[3 * (size_t)i + 2] = z[i];
  }
  return PLUM_OK;
}

int plum_set_profiling(plum_ctx* c, int on) {
  if (!c) return fail(PLUM_E_ARG, "null context");
  c->profiling = on != 0;
  return PLUM_OK;
}

int plum_kernel_times(plum_ctx* c, int cap, const char** names, double* avg_us, long long* count) {
  if (!c) return fail(PLUM_E_ARG, "null context");
  int n = 0;
  for (size_t i = 0; i < c->kname.size() && n < cap; i++) {
    if (!c->kcount[i]) continue;   // kernels that did not run
    if (names) names[n] = c->kname[i].c_str();
    if (avg_us) avg_us[n] = c->ksum_us[i] / c->kcount[i];
    if (count) count[n] = c->kcount[i];
    n++;
  }
  return n;
}

}  // extern "C"

#include "batch_api.h"
#include "surrogate_api.h"
#include "cbmc_api.h"
#include "noalloc_api.h"
#include "pressure_api.h"
