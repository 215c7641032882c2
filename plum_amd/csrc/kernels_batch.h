// Device-resident Monte Carlo over R independent systems (R = 1 for a single
// system), in speculative batches.
//
// A batch makes up to `pmax` proposals (screen slots) per system; the ones to
// be evaluated exactly get one of kMaxProp exact slots.  Without delayed
// acceptance every proposal is evaluated exactly (pmax <= kMaxProp).  With
// it, a surrogate screens up to kMaxScreen proposals and only those passing
// the first stage (plus, as training data, a few that did not) are evaluated.
//
// One batch = five launches (kernel boundaries order them; no grid-wide
// fences, which on a multi-XCD part would write back and invalidate L2),
// plus the surrogate's two between proposal and plan:
//   k_propose_spec   grid (pmax, R): proposal s of system r (move number
//                    counter + s), its spring / wall / dipole parts and
//                    bounding sphere (a molecule proposed twice is proposed
//                    from its current coordinates the second time).
//   k_plan_spec      grid (R, 1 + pmax chunks + fold chunks): first-stage
//                    decisions, exact slots, block counts; pairs of exact
//                    slots within interaction range get cross-term blocks;
//                    beside it, the proposals' phase tables in chunks of rows
//                    and the fold of the previous batch's accepted dS(k) into
//                    S(k).
//   k_compute_spec   all systems' k-space blocks (dS_e(k) of every exact slot
//                    and its dE_k per k tile), real-space query blocks
//                    (cluster queries by blocks) and moved-moved blocks per
//                    slot, and cross blocks (LJ + real pairs between two
//                    slots' moved beads, old/new combinations), spread over
//                    one grid.
//   k_reduce_spec    the sums of every system, fixed order; the k-space cross
//                    sums 2 c_k Re(dS_p* dS_q) as a Gram matrix of the dS rows.
//   k_resolve_spec   grid R: the reference's sequential Metropolis chain over
//                    the batch (simulation.cc:241-355), decided by one wave,
//                    each dE corrected by the cross terms of the proposals
//                    accepted before it, then the commits.
// Every proposal is evaluated against the state before the batch; accepting
// p changes q's dE by exactly the cross terms, so the chain is the sequential
// one (the random numbers depend only on the move number).  A second
// proposal of one molecule assumes the first is rejected; if it was
// accepted, the batch ends before the second.  A surrogate value
// has no such correction: the batch ends before the first proposal whose
// descriptors could see a bead accepted earlier in the batch, and that
// proposal is made again, from the same move number, in the next batch.
#pragma once
#include "kernels_move.h"

namespace plum {

constexpr int kMaxReplicas = 1024;
constexpr int kMaxSplit = 8;           // most blocks per real-space query
constexpr int kDefaultSplitDiv = 384;   // candidate slots per query share
constexpr int kKTile = 16;             // rows and l_z of a speculative k-space tile

// Per-system launch shape.
struct RepCfg {
  int nkb_s;    // k-space tiles (0 without Ewald)
  int qmax, qfine;   // blocks of a real-space query, ordinary and on an idle chip (query_split)
  int pmax;     // proposals per batch (<= kMaxProp, <= kMaxScreen with the surrogate)
  int maxm;     // moved-list capacity per proposal (longest molecule)
  int nmmb;     // moved-moved block capacity per exact slot
  int rstride;  // real-space partials per exact slot
  int da;       // delayed acceptance on
  int fill;     // exact slots given to first-stage rejections (training data)
  float r_d;    // descriptor radius of the surrogate
  int train;    // this system feeds the surrogate's training ring
  int qfill;    // waves of k_compute_spec resident on the chip at once
};

// Real-space query blocks of a move of nm beads: one query per cluster of up
// to kCluster consecutive moved beads at their old and one at their new
// positions, qb blocks per query (each takes a share of the query's cells),
// kQWaves waves per block.
constexpr int kQWaves = kBlock / kWave;
constexpr int kMaxQBlock = 8;
constexpr int kQShare = 800;   // candidate slots per block of a query at the default split_div
constexpr int kQFine = 480;    // the same where the queries leave the chip idle
// Most blocks of a query of `cand` expected candidate slots, `share` slots
// each at the default split_div.
__host__ __device__ __forceinline__ int query_split(double cand, int share, int split_div) {
  const double s = share * (double)split_div / kDefaultSplitDiv;
  return max(1, min(kMaxQBlock, (int)(cand / s + 0.5)));
}
// Blocks per query of a system with `clusters` queries in the batch (its own
// only: a system's sums do not depend on the systems beside it).  A query wave
// is a serial chain (cell list, candidate loads, pair drains) that ends the
// launch when it is long, but each more block of a query repeats its set-up:
// shares of about kQShare candidates (qmax blocks) are the shortest launches
// where a batch has its 16 proposals (k_compute_spec of the 40,000-bead system
// at 330, 650 and 1,000 a block: 45, 32 and 36 us; 1,000 beads at 1,000 and
// 1,600: 28 and 33), kQFine (qfine blocks) where few proposals leave most of the chip idle
// (delayed acceptance on the brush: 50 and 35 us).  More query waves than 5/8
// of what the chip holds at once (fill; the other blocks take the rest) start
// a second round: a query is spread no further (the brush at 16 and 32 waves a
// query: 71 and 110 us).
__host__ __device__ __forceinline__ int query_spread(int qmax, int qfine, int clusters, int fill) {
  if (clusters < 1) clusters = 1;
  const int want = 5 * fill / 8 / kQWaves / clusters, idle = fill / 4 / kQWaves / clusters;
  return max(max(1, min(want, qmax)), min(idle, qfine));
}
constexpr int kCluster = 8;   // moved beads per real-space query (cluster)
__host__ __device__ __forceinline__ int query_clusters(int nm) { return (nm + kCluster - 1) / kCluster; }
__host__ __device__ __forceinline__ int query_blocks(int nm, int qb) { return 2 * query_clusters(nm) * qb; }

// Moved-moved pair blocks: 256 pairs each, independent of the launch size.
__host__ __device__ __forceinline__ int nmm_blocks(int nm) {
  const int npair = nm * (nm - 1) / 2;
  return npair > 0 ? (npair + kBlock - 1) / kBlock : 1;
}

__host__ __device__ __forceinline__ int cross_blocks(int np, int nq) { return (np * nq + kBlock - 1) / kBlock; }

template <typename T>
__device__ __forceinline__ T load_const(const T* p, int i) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef __attribute__((address_space(4))) const T CT;
  return ((CT*)p)[i];
#else
  return p[i];
#endif
}

__device__ __forceinline__ int uload(const int* p) { return __builtin_amdgcn_readfirstlane(*p); }

// A value every lane of the wave holds, kept in scalar registers.
__device__ __forceinline__ double uniform_double(double v) {
  const unsigned long long b = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)b);
  const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(b >> 32));
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Lane `lane`'s value, in every lane.
__device__ __forceinline__ double lane_double(double v, int lane) {
  const unsigned long long b = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readlane((unsigned)b, lane);
  const unsigned hi = __builtin_amdgcn_readlane((unsigned)(b >> 32), lane);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// System r owning virtual block v: first r with pre[r] > v (inclusive prefix).
__device__ __forceinline__ int find_replica(const int* pre, int R, int v) {
  int lo = 0, hi = R - 1;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (pre[mid] > v) hi = mid;
    else lo = mid + 1;
  }
  return lo;
}

// View of proposal s (move record, moved list, phase tables) with the dS(k)
// and partial sums of exact slot e.
__device__ __forceinline__ Dev prop_view(const Geo& g, const Dev& d, const RepCfg& rc, int s, int e) {
  Dev v = d;
  v.rec = d.recs + s;
  v.mv_idx = d.smv_idx + s * rc.maxm;
  v.mv_old = d.mv_old + s * rc.maxm;
  v.mv_new = d.mv_new + s * rc.maxm;
  v.mv_type = d.mv_type + s * rc.maxm;
  v.tab = d.tab + (size_t)s * rc.maxm * 2 * g.tab_w;
  v.dS = d.dS + (size_t)e * g.n_kh;
  v.part_r = d.part_r + (size_t)e * rc.rstride;
  v.part_mm = d.part_mm + (size_t)e * rc.nmmb;
  return v;
}

// Minimum-image distance of two points in the Ewald box (x, y periodic; z
// periodic in the padded box as the real-space image sum is).
__device__ __forceinline__ double center_dist(const double* a, const double* b, const Geo& g) {
  double s = 0;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    double dk = a[k] - b[k];
    dk -= g.L[k] * rint(dk * g.inv_L[k]);
    s += dk * dk;
  }
  return sqrt(s);
}

// ------------------------------------------------------------ proposals
struct PropSmem {
  double s_b[kMaxChainDev][3];       // new positions of the moved beads
  double sbuf[7 * (kBlock / kWave)];
  double sh[kBlock / kWave];
  int s_forbid, s_prev;
  MoveSel s_sel;
};

// One proposal per block: a chain of dependent round trips (move number,
// molecule, its beads, the reductions), so the system's descriptors come in
// one read each, nothing that a thread computed is read back from memory, and
// the six sums share one reduction (13.7 -> 12.7 us at 100 beads a chain, 40,000
// beads; with the resolve's loads in one pass, below, 18.6 -> 17.9 ms for
// 4,000 moves).
__global__ __launch_bounds__(kBlock) void k_propose_spec(const Geo* __restrict__ G, const Dev* __restrict__ D,
                                                         const McDev* __restrict__ MC,
                                                         const RepCfg* __restrict__ RC, int R) {
  __shared__ PropSmem sm;
  const int p = blockIdx.x, r = blockIdx.y;
  if (r >= R) return;
  const Geo g = load_const(G, r);
  const Dev d = load_const(D, r);
  const McDev mc = load_const(MC, r);
  const RepCfg rc = load_const(RC, r);
  Ctl* C = d.ctl;
  const unsigned long long ctr0 = C->move_counter;
  const int overflow = C->overflow;
  int cut = rc.pmax;
  if (mc.ctr_limit <= ctr0) cut = 0;
  else if ((long long)(mc.ctr_limit - ctr0) < cut) cut = (int)(mc.ctr_limit - ctr0);
  if (p == 0 && threadIdx.x == 0) d.plan->n_prop = cut;
  if (p >= cut) return;
  const int lane = threadIdx.x % kWave, wv = threadIdx.x / kWave;
  if (threadIdx.x == 0) sm.s_forbid = 0;
  if (wv == 0) {
    // a molecule proposed again in the batch is proposed from its current
    // coordinates, i.e. on the assumption that its earlier proposal is
    // rejected; the resolve ends the batch there if it was accepted
    MoveSel sel = {-1, 0, 0};
    if (lane <= p) sel = select_move(d, mc, ctr0 + lane);
    const int mol_p = __shfl(sel.mol, p, kWave);   // read by all lanes, lane p among them
    const unsigned long long same = __ballot(lane < p && sel.mol == mol_p);
    if (lane == p) {
      sm.s_sel = sel;
      sm.s_prev = same ? 63 - __builtin_clzll(same) : -1;
    }
  }
  __syncthreads();
  const MoveSel sel = sm.s_sel;
  const int mol = __builtin_amdgcn_readfirstlane(sel.mol), mt = __builtin_amdgcn_readfirstlane(sel.mt);
  const int a = uload(&d.mol_start[mol]), bend = uload(&d.mol_start[mol + 1]);
  const double bcur = d.bond_cur[mol];
  const int len = bend - a;
  // an overflowed cell list is incomplete: skip, redo later
  const int valid = __builtin_amdgcn_readfirstlane(sel.valid && !overflow && len <= kMaxChainDev);
  PropRange mv = {0, 0};
  if (valid) mv = propose_positions(d, mc, ctr0 + p, mt, a, len, sm.s_b);
  const int lo = __builtin_amdgcn_readfirstlane(mv.lo), nm = __builtin_amdgcn_readfirstlane(mv.n), hi = lo + nm - 1;
  __syncthreads();
  // everything of the dE that involves this proposal alone: spring energy of
  // the trial molecule (molecule_spring's terms and order), wall and dipole
  // parts, bounding sphere; and the moved list.  (A valid move that moves no
  // bead keeps the molecule's current energy.)
  const bool spring = valid && g.use_bond && len > 1;
  auto bond = [&](int i) {
    const bool in0 = i >= lo && i <= hi, in1 = i + 1 >= lo && i + 1 <= hi;
    const int k0 = in0 ? i - lo : 0, k1 = in1 ? i + 1 - lo : 0;
    const double x0 = in0 ? sm.s_b[k0][0] : d.x[i], y0 = in0 ? sm.s_b[k0][1] : d.y[i];
    const double z0 = in0 ? sm.s_b[k0][2] : d.z[i];
    const double x1 = in1 ? sm.s_b[k1][0] : d.x[i + 1], y1 = in1 ? sm.s_b[k1][1] : d.y[i + 1];
    const double z1 = in1 ? sm.s_b[k1][2] : d.z[i + 1];
    return spring_energy(g, x0 - x1, y0 - y1, z0 - z1);
  };
  double v6[6] = {0, 0, 0, 0, 0, 0};   // spring (first block of bonds), wall, q dz, centre
  if (spring && a + (int)threadIdx.x < bend - 1) v6[0] = bond(a + threadIdx.x);
  double4* mv_old = d.mv_old + (size_t)p * rc.maxm;
  double4* mv_new = d.mv_new + (size_t)p * rc.maxm;
  int* mv_type = d.mv_type + (size_t)p * rc.maxm;
  int* mv_idx = d.smv_idx + (size_t)p * rc.maxm;
  // bead threadIdx.x kept in registers for the radius pass when every bead
  // has its own thread
  double4 pn0 = make_double4(0, 0, 0, 0), po0 = pn0;
  for (int k = threadIdx.x; k < nm; k += kBlock) {
    const int i = lo + k;
    const double q = d.q[i];
    const int ty = d.type[i];
    const double4 po = make_double4(d.x[i], d.y[i], d.z[i], q);
    const double4 pn = make_double4(sm.s_b[k][0], sm.s_b[k][1], sm.s_b[k][2], q);
    mv_old[k] = po;
    mv_new[k] = pn;
    mv_type[k] = ty;
    mv_idx[k] = i;
    if (k == (int)threadIdx.x) {
      pn0 = pn;
      po0 = po;
    }
    if (g.use_ext) {
      const WallType w = d.wall[ty];
      const double en = wall_energy(pn.z, w, g);
      if (en >= kVeryLargeEnergy) atomicOr(&sm.s_forbid, 1);
      v6[1] += en - wall_energy(po.z, w, g);
    }
    v6[2] += pn.w * (pn.z - po.z);
    v6[3] += pn.x + po.x;
    v6[4] += pn.y + po.y;
    v6[5] += pn.z + po.z;
  }
  // the six sums in one pass (waves, then the wave partials in order, as
  // block_sum does), then the bounding radius (max)
#pragma unroll
  for (int i = 0; i < 6; i++) {
    v6[i] = wave_sum(v6[i]);
    if (lane == 0) sm.sbuf[6 * wv + i] = v6[i];
  }
  __syncthreads();
  double t6[6] = {0, 0, 0, 0, 0, 0};
  for (int w = 0; w < kBlock / kWave; w++)
#pragma unroll
    for (int i = 0; i < 6; i++) t6[i] += sm.sbuf[6 * w + i];
  double ebt = t6[0];
  if (spring)
    for (int base = a + kBlock; base < bend - 1; base += kBlock) {
      const int i = base + threadIdx.x;
      ebt += block_sum<kBlock>(i < bend - 1 ? bond(i) : 0.0, sm.sh);   // valid in thread 0
    }
  const double inv = nm > 0 ? 1.0 / (2.0 * nm) : 0.0;
  const double c0 = t6[3] * inv, c1 = t6[4] * inv, c2 = t6[5] * inv;
  double rad = 0;
  for (int k = threadIdx.x; k < nm; k += kBlock) {
    const double4 pn = nm <= kBlock ? pn0 : mv_new[k], po = nm <= kBlock ? po0 : mv_old[k];
    const double dn = (pn.x - c0) * (pn.x - c0) + (pn.y - c1) * (pn.y - c1) + (pn.z - c2) * (pn.z - c2);
    const double dd = (po.x - c0) * (po.x - c0) + (po.y - c1) * (po.y - c1) + (po.z - c2) * (po.z - c2);
    rad = fmax(rad, fmax(dn, dd));
  }
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) rad = fmax(rad, __shfl_down(rad, off, kWave));
  if (lane == 0) sm.sbuf[6 * (kBlock / kWave) + wv] = rad;
  __syncthreads();
  if (threadIdx.x != 0) return;
  rad = 0;
  for (int w = 0; w < kBlock / kWave; w++) rad = fmax(rad, sm.sbuf[6 * (kBlock / kWave) + w]);
  MoveRec rec = {};
  rec.n_moved = nm;
  rec.mol = mol;
  rec.move_type = mt;
  rec.valid = valid;
  rec.contig = 1;   // every generator moves a contiguous index range
  rec.lo = valid ? lo : 0;
  rec.hi = valid ? hi : -1;
  d.recs[p] = rec;
  PropInfo pi;
  pi.bond_trial = ebt;
  pi.ew = t6[1];
  pi.dmz = t6[2];
  pi.c[0] = c0;
  pi.c[1] = c1;
  pi.c[2] = c2;
  pi.rad = sqrt(rad);
  pi.forbid = sm.s_forbid;
  pi.n = nm;
  pi.mol = mol;
  pi.type = mt;
  pi.valid = valid;
  pi.skipped = (overflow && sel.valid) ? 1 : 0;
  pi.prev = sm.s_prev;
  pi.len = len;
  pi.bcur = bcur;
  d.prop[p] = pi;
}

// Plan of a batch, one block per system: first-stage decisions (delayed
// acceptance), exact slots, real-space + moved-moved blocks per exact slot,
// the exact-slot pairs within interaction range (bounding spheres closer than
// the search radius) and their cross-term blocks, the virtual-block count.
constexpr int kPlanThreads = 512;

struct PlanSmem {
  PropInfo s_prop[kMaxScreen];
  double s_nn[kMaxScreen];
  double s_bcur[kMaxScreen];
  double s_u1[kMaxScreen];
  int s_len[kMaxScreen];
  int s_screen[kMaxProp];
  int s_xblk[kMaxPairs];   // cross blocks of a slot pair within range, -1 if not
  int s_pq[kMaxPairs];     // slots (p, q) of pair j: p | q << 8
  int s_ne, s_off;
};
static_assert(kMaxPairs <= 2 * kWave, "near-pair compaction: two pairs per lane of one wave");

// Phase tables of the proposals, in chunks of rows beside the plan (the plan
// is one block per system; the chunks fill the rest of the chip meanwhile).
constexpr int kTabStage = 3072;   // LDS stage of a table chunk, entries

__host__ __device__ __forceinline__ int tab_chunk_rows(int tab_w) {
  const int ws = tab_w | 1;
  return ws <= kTabStage ? min(kTabStage / ws, kPlanThreads / 3) : kPlanThreads / 3;
}

__device__ void plan_tables(const Geo* __restrict__ G, const Dev* __restrict__ D, const RepCfg* __restrict__ RC,
                            int r, int c, int nch, double2* stage) {
  const Geo& g = G[r];
  const Dev& d = D[r];
  const RepCfg& rc = RC[r];
  if (!g.use_ewald || g.n_kh == 0) return;
  const int p = c / nch, ch = c - p * nch;
  if (p >= d.plan->n_prop) return;
  const Dev v = prop_view(g, d, rc, p, 0);
  const int nrow = 2 * v.rec->n_moved, cr = tab_chunk_rows(g.tab_w);
  const int r0 = ch * cr;
  if (r0 >= nrow) return;
  const int ws = (g.tab_w | 1) <= kTabStage ? (g.tab_w | 1) : 0;
  tables_chunk(g, v, r0, min(cr, nrow - r0), stage, ws);
}

// The S(k) of the slots the previous batch accepted, folded in by chunks of
// k vectors beside the plan (before this batch's k-space overwrites their dS
// rows), in slot order.  A batch with no proposal leaves them pending (its
// resolve keeps the mask).
__device__ void plan_fold(const Geo* __restrict__ G, const Dev* __restrict__ D, int r, int f) {
  const Geo& g = G[r];
  const Dev& d = D[r];
  if (d.plan->n_prop == 0) return;
  const unsigned mask = d.plan->acc_mask;
  const int k = f * kPlanThreads + threadIdx.x;
  if (!mask || k >= g.n_kh) return;
  double2 S = d.Sk[k];
  for (int e = 0; e < kMaxProp; e++)
    if (mask & (1u << e)) {
      const double2 ds = d.dS[(size_t)e * g.n_kh + k];
      S.x += ds.x;
      S.y += ds.y;
    }
  d.Sk[k] = S;
}

__global__ __launch_bounds__(kPlanThreads) void k_plan_spec(const Geo* __restrict__ G, const Dev* __restrict__ D,
                                                            const McDev* __restrict__ MC,
                            const RepCfg* __restrict__ RC, int* vb_count, int R, int nch, int ntab) {
  __shared__ union {
    PlanSmem p;
    double2 stage[kTabStage];
  } smu;
  PlanSmem& sm = smu.p;
  const int r = blockIdx.x;
  if (r >= R) return;
  if (blockIdx.y > 0) {
    const int c = blockIdx.y - 1;
    if (c < ntab) plan_tables(G, D, RC, r, c, nch, smu.stage);
    else plan_fold(G, D, r, c - ntab);
    return;
  }
  // by-value copies through the constant address space: the per-system
  // structs stay in scalar registers instead of being re-read after stores
  const Geo g = load_const(G, r);
  const Dev d = load_const(D, r);
  const McDev mc = load_const(MC, r);
  const RepCfg rc = load_const(RC, r);
  SpecPlan* plan = d.plan;
  const int np = plan->n_prop;
  const int t = threadIdx.x;
  const unsigned long long ctr0 = d.ctl->move_counter;
  if (t < np) {
    const PropInfo P = d.prop[t];
    sm.s_prop[t] = P;
    sm.s_bcur[t] = P.bcur;
    sm.s_len[t] = P.len;
    const unsigned long long ctr = ctr0 + t;
    const uint4 u = Philox::gen(make_uint4((uint32_t)ctr, (uint32_t)(ctr >> 32), 0xDA1u, 0u),
                                make_uint2((uint32_t)mc.seed, (uint32_t)(mc.seed >> 32)));
    sm.s_u1[t] = u01_32(u.x);
  }
  __syncthreads();
  if (rc.da) {
    // network part of the surrogate, one wave per proposal: sum over moved
    // beads of f(new) - f(old), fixed order
    const int w = t / kWave, lane = t % kWave;
    for (int s = w; s < np; s += kPlanThreads / kWave) {
      const PropInfo& P = sm.s_prop[s];
      const float* f = d.sur_f + (size_t)(2 * s) * rc.maxm;
      double nn = 0;
      if (P.valid)
        for (int m = lane; m < P.n; m += kWave) nn += (double)f[rc.maxm + m] - (double)f[m];
#pragma unroll
      for (int off = kWave / 2; off > 0; off >>= 1) nn += __shfl_down(nn, off, kWave);
      if (lane == 0) sm.s_nn[s] = nn;
    }
    __syncthreads();
  }
  if (t < kWave) {
    // one lane per proposal: the first stage, then exact slots in proposal
    // order (a proposal past the last slot is decided next batch), then spare
    // slots for first-stage rejections (training data), by ballots
    const bool have = t < np;
    PropInfo P = {};
    if (have) P = sm.s_prop[t];
    int pass = 1;
    double des = 0;
    if (have && rc.da && P.valid) {
      // surrogate dE: exact spring and wall parts plus the network's estimate
      // of the pair and k-space parts; first stage min(1, exp(-beta dE_s))
      if (g.use_bond && sm.s_len[t] > 1) des += P.bond_trial - sm.s_bcur[t];
      if (g.use_ext) des += P.forbid ? kVeryLargeEnergy : P.ew;
      des += sm.s_nn[t];
      pass = des < kVeryLargeEnergy && sm.s_u1[t] < exp(-g.beta * des);
    }
    const unsigned long long ex = __ballot(have && pass && P.valid);
    const int nex = __popcll(ex);
    int ndec = np;
    if (nex > kMaxProp) {
      // no exact slot left for the (kMaxProp + 1)-th: decided next batch
      unsigned long long m = ex;
      for (int i = 0; i < kMaxProp; i++) m &= m - 1;
      ndec = __builtin_ctzll(m);
    }
    const int ne0 = min(nex, kMaxProp);
    int exact = (have && pass && P.valid && t < ndec) ? lanes_below(ex) : -1;
    const unsigned long long fl = __ballot(have && t < ndec && !pass && P.valid && P.n > 0);
    const int nfill = max(0, min(__popcll(fl), rc.fill - ne0));
    if (((fl >> t) & 1ull) && lanes_below(fl) < nfill) exact = ne0 + lanes_below(fl);
    const int ne = ne0 + nfill;
    if (have) {
      plan->exact_of[t] = exact;
      plan->pass1[t] = pass;
      plan->de_s[t] = des;
      if (exact >= 0) sm.s_screen[exact] = t;
    }
    wave_sync_lds();
    // blocks per query for this batch's exact slots, then query and
    // moved-moved blocks per exact slot, prefixes over the slots
    int ncl = t < ne ? 2 * query_clusters(sm.s_prop[sm.s_screen[t]].n) : 0;
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) ncl += __shfl_xor(ncl, o, kWave);
    const int qb = query_spread(rc.qmax, rc.qfine, ncl, rc.qfill);
    int nq = 0, nmb = 0;
    if (t < ne) {
      const int n = sm.s_prop[sm.s_screen[t]].n;
      nq = n > 0 ? query_blocks(n, qb) : 0;
      nmb = n > 0 ? nmm_blocks(n) : 0;
      plan->screen_of[t] = sm.s_screen[t];
    }
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const int u = __shfl_up(nq, o, kWave), v = __shfl_up(nmb, o, kWave);
      if (t >= o) {
        nq += u;
        nmb += v;
      }
    }
    if (t < ne) {
      plan->q_off[t + 1] = nq;
      plan->mm_off[t + 1] = nmb;
    }
    const int off = ne > 0 ? __shfl(nq, ne - 1, kWave) + __shfl(nmb, ne - 1, kWave) : 0;
    if (t == 0) {
      plan->qblk = qb;
      plan->q_off[0] = 0;
      plan->mm_off[0] = 0;
      plan->n_decide = ndec;
      plan->n_exact = ne;
      sm.s_ne = ne;
      sm.s_off = off;
    }
  }
  __syncthreads();
  // slot pairs whose moved beads can interact (bounding spheres within the
  // search radius), one thread per pair
  const int ne = sm.s_ne, npair = ne * (ne - 1) / 2;
  for (int j = t; j < npair; j += kPlanThreads) {
    int e = (int)((1.0 + sqrt(1.0 + 8.0 * j)) * 0.5);
    while (e * (e - 1) / 2 > j) e--;
    while ((e + 1) * e / 2 <= j) e++;
    const int e0 = j - e * (e - 1) / 2;
    const PropInfo& pq = sm.s_prop[sm.s_screen[e]];
    const PropInfo& pp = sm.s_prop[sm.s_screen[e0]];
    int xb = -1;
    if (pq.n > 0 && pp.n > 0 && pp.mol != pq.mol &&
        center_dist(pp.c, pq.c, g) <= pp.rad + pq.rad + g.rs + 1e-9)
      xb = cross_blocks(pp.n, pq.n);
    sm.s_xblk[j] = xb;
    sm.s_pq[j] = e0 | (e << 8);
  }
  __syncthreads();
  if (t >= kWave) return;
  // near pairs in (e, e0) order, e0 < e, compacted by one wave: lane l holds
  // pairs 2l and 2l + 1; a prefix scan gives each its place and block offset
  const int j0 = 2 * t, j1 = j0 + 1;
  const int x0 = j0 < npair ? sm.s_xblk[j0] : -1, x1 = j1 < npair ? sm.s_xblk[j1] : -1;
  const int c0 = x0 >= 0, c1 = x1 >= 0;
  const int own_c = c0 + c1, own_b = (c0 ? x0 : 0) + (c1 ? x1 : 0);
  int cs = own_c, bs = own_b;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const int a = __shfl_up(cs, o, kWave), b = __shfl_up(bs, o, kWave);
    if (t >= o) {
      cs += a;
      bs += b;
    }
  }
  int nn = cs - own_c, xo = bs - own_b;
  if (t == 0) plan->pair_off[0] = 0;
  if (c0) {
    plan->pair_p[nn] = sm.s_pq[j0] & 0xff;
    plan->pair_q[nn] = sm.s_pq[j0] >> 8;
    xo += x0;
    nn++;
    plan->pair_off[nn] = xo;
  }
  if (c1) {
    plan->pair_p[nn] = sm.s_pq[j1] & 0xff;
    plan->pair_q[nn] = sm.s_pq[j1] >> 8;
    xo += x1;
    nn++;
    plan->pair_off[nn] = xo;
  }
  if (t == kWave - 1) {
    plan->n_near = cs;
    // k-space blocks: one per exact slot and k tile
    vb_count[r] = (np > 0 && ne > 0) ? rc.nkb_s * ne + sm.s_off + bs : 0;
  }
}

// ------------------------------------------------------------ k space
// One block per (k tile, exact slot).  A tile is 16 rows (l_x, l_y) of the
// half-space list by 16 consecutive l_z >= 0, and both signs of l_z: with
// a = q e^{i (l_x theta_x + l_y theta_y)} and z = e^{i l_z theta_z} of a moved
// bead at its new (+) or old (-) position,
//   dS(+-l_z) = sum (Re a Re z -+ Im a Im z) + i (Im a Re z +- Re a Im z),
// four real products of a 16 x 2n by a 2n x 16 matrix on
// v_mfma_f64_16x16x4f64: lane l supplies row l % 16 (column l % 16) of the
// left (right) operand at inner index l / 16 and receives rows 4 v + l / 16 of
// column l % 16 in its value v.  Inner index 2 m + on is row 2 m + on of the
// slot's phase tables, so a step of four takes two beads; the block's waves
// take the steps in turn and meet in LDS, where wave w sums value v = w.  The
// waves then write dS_e(k) and sum the slot's dE_e = sum_k c_k (2 Re(S* dS_e)
// + |dS_e|^2) over their k vectors (S(k) with the previous batch's acceptances
// folded in by the plan).  The cross sums 2 sum_k c_k Re(dS_p* dS_q) are
// formed from the dS rows by k_reduce_spec.
// Bound by the latency of the table loads, hence four waves a tile (one wave
// per tile: 30 us for 100 beads).  The vector form (one lane per run of four
// k vectors, the z phase advanced by multiplication) spent 110 vector
// instructions a bead on 32 runs, 6.6 million wave instructions per batch of
// the 40,000-bead system, half of the launch; here a step is 4 matrix
// instructions for 512 k vectors' terms and some 12 vector instructions, and
// the z phase comes from the table without the multiplications' rounding.
static_assert(kMaxProp <= 32, "exact slots are bits of one mask");
typedef double f64x4 __attribute__((ext_vector_type(4)));

struct KTileSmem {
  double s_acc[kQWaves][4][4][kWave];   // [wave][value][product][lane]
};
static_assert(kQWaves == 4, "wave w of a k tile sums value w");

__device__ void kspace_spec_block(const Geo& g, const Dev& d, const RepCfg& rc, int s, int tile, int e,
                                  KTileSmem& sm) {
  const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
  const int n = uload(&d.recs[s].n_moved);
  const int2 tl = load_const(d.ktile, tile);   // first row, first l_z
  const int col = lane % kKTile, sub = lane / kKTile;
  const int4 row = d.krow[tl.x + col];         // l_x, l_y, first k of the row, largest l_z (-1: no row)
  const int lz = tl.y + col;
  // the rows this lane finishes (value w): row 4 w + sub of the tile
  const int4 mine = d.krow[tl.x + 4 * w + sub];
  f64x4 rr = {0, 0, 0, 0}, ii = rr, ri = rr, ir = rr;
  if (n > 0) {
    const double4* mo = d.mv_old + s * rc.maxm;
    const double2* tab = d.tab + (size_t)s * rc.maxm * 2 * g.tab_w;
    const int ox = row.x, oy = g.nkx + 1 + abs(row.y), oz = g.nkx + 1 + g.nky + 1 + min(lz, g.nkz);
    const double sy = row.y < 0 ? -1.0 : 1.0, sq = (sub & 1) ? 1.0 : -1.0;
    const int last = 2 * n - 1;
#pragma unroll 2
    for (int i0 = 4 * w; i0 <= last; i0 += 4 * kQWaves) {
      const int i = min(i0 + sub, last);   // past the end: the last row again, with no charge
      const double2* t = tab + (size_t)i * g.tab_w;
      const double2 X = t[ox], Y = t[oy], Z = t[oz];
      const double q = i0 + sub <= last ? sq * mo[i >> 1].w : 0.0;
      const double yr = q * Y.x, yi = q * sy * Y.y;
      const double ar = X.x * yr - X.y * yi, ai = X.x * yi + X.y * yr;
      rr = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, Z.x, rr, 0, 0, 0);
      ii = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, Z.y, ii, 0, 0, 0);
      ri = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, Z.y, ri, 0, 0, 0);
      ir = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, Z.x, ir, 0, 0, 0);
    }
  }
#pragma unroll
  for (int v = 0; v < 4; v++) {
    sm.s_acc[w][v][0][lane] = rr[v];
    sm.s_acc[w][v][1][lane] = ii[v];
    sm.s_acc[w][v][2][lane] = ri[v];
    sm.s_acc[w][v][3][lane] = ir[v];
  }
  __syncthreads();
  double t4[4] = {0, 0, 0, 0};
#pragma unroll
  for (int u = 0; u < kQWaves; u++)
#pragma unroll
    for (int p = 0; p < 4; p++) t4[p] += sm.s_acc[u][w][p][lane];
  double part = 0;
  double2* dS = d.dS + (size_t)e * g.n_kh;
  auto put = [&](int k, double x, double y) {
    const double2 S = d.Sk[k];
    dS[k] = make_double2(x, y);
    part += d.ck[k] * (2.0 * (S.x * x + S.y * y) + x * x + y * y);
  };
  if (lz <= mine.w) {
    // the l_x = l_y = 0 row holds l_z > 0 only
    const bool xy = (mine.x | mine.y) != 0;
    const int k0 = xy ? mine.z + mine.w : mine.z - 1;
    if (xy || lz > 0) put(k0 + lz, t4[0] - t4[1], t4[2] + t4[3]);
    if (xy && lz > 0) put(k0 - lz, t4[0] + t4[1], t4[3] - t4[2]);
  }
  part = wave_sum(part);
  if (lane == 0) d.part_ks[((size_t)e * rc.nkb_s + tile) * kQWaves + w] = part;
}

// ------------------------------------------------------------ real space
// Cluster queries: a block takes up to kCluster consecutive moved beads of one
// proposal, all at their old or all at their new positions (the query
// points), and one share of the cells within the search radius of the points'
// bounding box.  Its threads list the share's cells together, one each, with a
// block prefix over their counts, and its waves take 64 candidates in turn, so
// the four of them end together and a cell is listed once.  Each lane takes a
// candidate slot (bead index, position and type loaded together, one
// candidate ahead) and tests it against every point, so a candidate's load,
// cell lookup and image decode serve all the points.  The charged pairs within
// the real-space cutoff go into a per-wave queue in LDS (ballot + lane
// prefix), last in first out; each time it holds 64 pairs every lane takes one
// and evaluates its erfc term, so the lanes never diverge on the pair
// arithmetic.  Pairs within the largest LJ cutoff, one in a hundred at r_c =
// 12, have a queue of their own: in the common one they cost nearly every
// drain the LJ table load and arithmetic.  A wave reduction sums the lanes in
// fixed order.  Bound by VALU issue: about 150 instructions per 64 pairs
// (distance tests of three candidates for each pair in range, queue, erfc).
constexpr int kQueue = 2 * kWave;   // < 64 left after a drain, one push of up to 64
static_assert(kCluster <= kWave, "one lane per query point");

// What a cluster query sums: the moved beads of a proposal against the rest;
// every bead of the list against all (from scratch); the same as the change
// under the stretch of a volume perturbation.
enum QueryMode { Q_MOVED = 0, Q_ALL = 1, Q_STRETCH = 2 };

// Stretched configuration of a volume perturbation: per bead the displacement
// of the image that the cell list holds, the displacement of one period, the
// number of surface-site molecules.
struct StretchArgs {
  const double* dw;
  const int* mol_of;
  double dz;
  int phantom;
};

// Class of a molecule in the pair rule of a volume perturbation: mobile 0,
// first / second half of the surface sites 1 / 2; pairs 0-0, 0-1 and 1-2 count
// (pressure.cc:271-272: a site pairs only from the first half of the list).
__device__ __forceinline__ int stretch_class(int mol, int phantom) {
  return mol >= phantom ? 0 : (mol < phantom / 2 ? 1 : 2);
}
__device__ __forceinline__ bool stretch_pair(int a, int b) { return a + b <= 1 || (a != b && a > 0 && b > 0); }

template <int P, int MODE>
struct QWaveSmem {
  double2 s_q[kQueue];     // squared distance and charge product of a queued pair
  double s_lr[kQueue];     // squared distance of a queued LJ pair
  int s_lt[kQueue];        // its LJ pair index
  // P = 1: the queue of charged pairs at or beyond fp64_below, evaluated in FP32
  float2 s_f[P ? kQueue : 1];
  // Q_STRETCH: the stretched squared distances of the queued pairs
  double s_qn[MODE == Q_STRETCH ? kQueue : 1], s_ln[MODE == Q_STRETCH ? kQueue : 1];
};

template <int P, int MODE>
struct QueryShare {
  int s_cell[kBlock];      // cells of this share, their images and count prefix
  int s_img[kBlock];
  int s_end[kBlock];
  int s_wsum[kQWaves];
  double4 s_pt[kCluster];  // query points (the image nearest the first point) and charges
  int s_ptt[kCluster];     // their types
  int s_own[kCluster];     // their bead indices (not Q_MOVED)
  double s_ptd[kCluster];  // their displacements and classes (Q_STRETCH)
  int s_cls[kCluster];
  QWaveSmem<P, MODE> q[kQWaves];
};

// LJ + real-space energy of up to kCluster points (lane l holds point
// l % kCluster: position and charge, type, whether it counts; at least one
// does) against every bead image in the cell list within the search radius,
// skipping the index range [mlo, mhi] (the device loop's moves are
// contiguous), over share `part` of `nparts` of the query's cells.  Not
// Q_MOVED: the points are beads of the list themselves, own their indices, and
// each pair counts once; a bead's own images are left to the caller (theirs are
// whole edges away, and an edge may be the cutoff itself, where the rounding of
// a position would decide).
// Q_STRETCH: each pair's stretched minus current energy, over the pairs within
// the cutoff in either (the search reaches kStretchMargin further, more than
// a separation changes).  Each wave's part of the result valid in its lane 0.
constexpr double kStretchMargin = 1e-3;

template <int P, int MODE>
__device__ double2 real_query_cluster(const Geo& g, const Dev& d, const double4& p, int type, bool valid, int own,
                                      int mlo, int mhi, int part, int nparts, QueryShare<P, MODE>& sh,
                                      const StretchArgs& st = StretchArgs{nullptr, nullptr, 0, 0}) {
  constexpr bool ALL = MODE != Q_MOVED;
  constexpr bool STR = MODE == Q_STRETCH;
  const int lane = threadIdx.x % kWave, wv = threadIdx.x / kWave;
  const double rs = STR ? g.rs + kStretchMargin : g.rs, rs2 = STR ? rs * rs : g.rs2;
  QWaveSmem<P, MODE>& sm = sh.q[wv];
  // each point as the image nearest the first point (an image of a point has
  // the same pair images within the radius), and the points' bounding box.  The
  // image is the point's own wrapped position plus a whole edge or none, as a
  // candidate's is, so that a bead at the same coordinates is at distance 0 to
  // the bit.  Along a z that is not periodic all points move with the first one,
  // by the edges that wrap it (none inside the slab): LJ counts the candidates of
  // image 0 only, and a chain may span more than half of the height.  (Each
  // wrapped on its own, a trial bead behind a wall would stretch the box over
  // the height: 90 us for the brush's launch instead of 66.)
  const unsigned vm = (unsigned)__ballot(valid) & ((1u << kCluster) - 1u);
  const int np = ALL ? kCluster : __popc(vm);
  const int ref = __builtin_ctz(vm);
  double bl[3], bh[3];
  {
    const double pw[3] = {wrap_coord(p.x, g.L[0], g.inv_L[0]), wrap_coord(p.y, g.L[1], g.inv_L[1]),
                          wrap_coord(p.z, g.L[2], g.inv_L[2])};
    double qv[3], nv[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const double rk = lane_double(pw[k], ref);
      double from = pw[k];
      nv[k] = -rint((pw[k] - rk) * g.inv_L[k]);
      if (k == 2 && g.npbc < 3) {
        from = p.z;
        nv[k] = rint((rk - lane_double(p.z, ref)) * g.inv_L[k]);
      }
      qv[k] = valid ? from + nv[k] * g.L[k] : rk;
    }
    if (threadIdx.x < kCluster) {
      // (a point that does not count is out of every candidate's reach)
      sh.s_pt[lane] = make_double4(valid ? qv[0] : -1e30, qv[1], qv[2], p.w);
      sh.s_ptt[lane] = type;
      sh.s_own[lane] = own;
      if constexpr (STR) {
        // (p is a slot of the list: its own image is the wrapped one)
        const int jo = valid ? own : 0;
        sh.s_ptd[lane] = valid ? st.dw[jo] + nv[2] * st.dz : 0.0;
        sh.s_cls[lane] = stretch_class(st.mol_of[jo], st.phantom);
      }
    }
#pragma unroll
    for (int k = 0; k < 3; k++) {
      bl[k] = qv[k];
      bh[k] = qv[k];
    }
#pragma unroll
    for (int o = kCluster / 2; o > 0; o >>= 1)
#pragma unroll
      for (int k = 0; k < 3; k++) {
        bl[k] = fmin(bl[k], __shfl_xor(bl[k], o, kWave));
        bh[k] = fmax(bh[k], __shfl_xor(bh[k], o, kWave));
      }
    // the butterfly leaves the box in every lane: scalar registers from here
#pragma unroll
    for (int k = 0; k < 3; k++) {
      bl[k] = uniform_double(bl[k]);
      bh[k] = uniform_double(bh[k]);
    }
  }
  int lo[3], nd[3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    lo[k] = (int)floor((bl[k] - rs) * g.inv_h[k]);
    const int hi = (int)floor((bh[k] + rs) * g.inv_h[k]);
    nd[k] = hi - lo[k] + 1;
  }
  const int ncq = nd[0] * nd[1] * nd[2];
  const int mine = (ncq + nparts - 1) / nparts;   // cells of this share, at most
  const int nt = g.n_types;
  const double rcs = STR ? g.rc + kStretchMargin : g.rc;
  const double rc2 = g.use_ewald ? rcs * rcs : -1.0;
  double lj2 = g.use_pair ? g.lj2_max : -1.0;
  if (STR && g.use_pair) {
    const double c = sqrt(g.lj2_max) + kStretchMargin;
    lj2 = c * c;
  }
  const double fp64_b2 = P ? g.fp64_below * g.fp64_below : 0.0;
  double elj = 0, ere = 0;
  int qn = 0, ln = 0, fn = 0;   // queue fills (wave-uniform)
  // real-space terms of the pairs at the queue's end, one per lane
  auto drain = [&](int count) {
    wave_sync_lds();
    qn -= count;
    if (lane < count) {
      const double2 e = sm.s_q[qn + lane];
      double r, rinv;
      sqrt_rsqrt(e.x, r, rinv);
      const double x = g.sqrt_alpha * r;
      const int ni = erfc_node_index(x);
      const double u = erfc_from_node(x, ni, g.erfc_tab[ni]) * rinv;
      if constexpr (!STR) {
        if (e.x > 0) ere = fma(e.y, u, ere);
      } else {
        const double n2 = sm.s_qn[qn + lane];
        double rn, rninv;
        sqrt_rsqrt(n2, rn, rninv);
        const double xn = g.sqrt_alpha * rn;
        const int nn = erfc_node_index(xn);
        const double un = erfc_from_node(xn, nn, g.erfc_tab[nn]) * rninv;
        ere += e.y * ((n2 > 0 && rn <= g.rc ? un : 0.0) - (e.x > 0 && r <= g.rc ? u : 0.0));
      }
    }
    wave_sync_lds();
  };
  // the same in FP32 (pairs at or beyond fp64_below), added to the FP64 sum
  auto drain32 = [&](int count) {
    wave_sync_lds();
    fn -= count;
    if (lane < count) {
      const float2 e = sm.s_f[fn + lane];
      const float rf = sqrtf(e.x);
      const float x = (float)g.sqrt_alpha * rf;
      const int ni = erfc_node_index32(x);
      ere += (double)(e.y * erfc_from_node32(x, ni, g.erfc_tab32[ni]) / rf);
    }
    wave_sync_lds();
  };
  auto drain_lj = [&](int count) {
    wave_sync_lds();
    ln -= count;
    if (lane < count) {
      const LJPair lp = d.lj[sm.s_lt[ln + lane]];
      const double u = lj_energy(sqrt(sm.s_lr[ln + lane]), lp);
      elj += STR ? lj_energy(sqrt(sm.s_ln[ln + lane]), lp) - u : u;
    }
    wave_sync_lds();
  };
  for (int base = 0; base < mine; base += kBlock) {
    const int nloc = min(kBlock, mine - base);
    int end = 0;
    if (threadIdx.x < nloc) {
      // cell of this share in group `grp` of nparts cells: the shares change
      // places from group to group (with a fixed place and nparts a multiple
      // of a grid edge, one share would hold a whole layer of a slab and
      // another the empty padding)
      const int grp = base + threadIdx.x;
      const int c = nparts * grp + (int)((part + (unsigned)grp * 40503u % 8191u) % (unsigned)nparts);
      const int cyx = c / nd[2], cz = c - cyx * nd[2], cx = cyx / nd[1], cy = cyx - cx * nd[1];
      const int u[3] = {lo[0] + cx, lo[1] + cy, lo[2] + cz};
      int cell = 0, img = 0;
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const int qk = floordiv(u[k], g.nc[k]);
        const int w = u[k] - qk * g.nc[k];
        cell = cell * g.nc[k] + w;
        img |= ((qk + 128) & 0xff) << (8 * k);
      }
      sh.s_cell[threadIdx.x] = cell;
      sh.s_img[threadIdx.x] = img;
      // cells whose box (widened by a rounding margin) lies beyond the search
      // radius of the bounding box hold no candidate
      double dmin2 = c < ncq ? 0 : 2 * rs2 + 1;
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const double b0 = (double)u[k] * g.h[k] - 1e-9 * g.L[k], b1 = b0 + g.h[k] + 2e-9 * g.L[k];
        const double dd = fmax(0.0, fmax(b0 - bh[k], bl[k] - b1));
        dmin2 += dd * dd;
      }
      end = dmin2 > rs2 ? 0 : d.ccount[cell];
    }
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const int v = __shfl_up(end, o, kWave);
      if (lane >= o) end += v;
    }
    if (lane == kWave - 1) sh.s_wsum[wv] = end;
    __syncthreads();
    int total = 0;
#pragma unroll
    for (int w = 0; w < kQWaves; w++) {
      const int v = sh.s_wsum[w];
      if (w < wv) end += v;
      total += v;
    }
    total = __builtin_amdgcn_readfirstlane(total);
    sh.s_end[threadIdx.x] = end;
    __syncthreads();
    // candidate it: its cell slot and image (binary search over the share's
    // cell prefix in LDS)
    auto locate = [&](int it, size_t& si, int& img) {
      int lo_i = 0, hi_i = nloc - 1;
      while (lo_i < hi_i) {
        const int mid = (lo_i + hi_i) >> 1;
        if (sh.s_end[mid] > it) hi_i = mid;
        else lo_i = mid + 1;
      }
      si = (size_t)sh.s_cell[lo_i] * g.cap + (it - (lo_i ? sh.s_end[lo_i - 1] : 0));
      img = sh.s_img[lo_i];
    };
    int it = threadIdx.x;
    int j = -1, tj = 0, img = 0;
    double4 pj = make_double4(0, 0, 0, 0);
    if (it < total) {
      size_t si;
      locate(it, si, img);
      j = d.cbead[si];
      pj = d.cpos[si];
      tj = d.ctype[si];
    }
    // wave-uniform trip count: the lanes past `total` ride along
    const int first = wv * kWave;
    const int rounds = total > first ? (total - first + kBlock - 1) / kBlock : 0;
    for (int rd = 0; rd < rounds; rd++) {
      const int it2 = it + kBlock;
      int j2 = -1, tj2 = 0, img2 = 0;
      double4 pj2 = make_double4(0, 0, 0, 0);
      if (it2 < total) {
        size_t si2;
        locate(it2, si2, img2);
        j2 = d.cbead[si2];
        pj2 = d.cpos[si2];
        tj2 = d.ctype[si2];
      }
      // candidate it (its image position) against every point; a candidate
      // that does not count is put where every test fails
      const bool ok = it < total && j >= 0 && !(j >= mlo && j <= mhi);
      const int iz = ((img >> 16) & 0xff) - 128, ix = (img & 0xff) - 128, iy = ((img >> 8) & 0xff) - 128;
      const double cx = ok ? pj.x + ix * g.L[0] : 1e30, cy = pj.y + iy * g.L[1], cz = pj.z + iz * g.L[2];
      const double qj = g.lB * pj.w;
      const double rcj2 = pj.w != 0 ? rc2 : -1.0;
      double ljj2 = (g.npbc == 3 || iz == 0) ? lj2 : -1.0;
      double cd = 0;   // displacement of the candidate's image, its class
      int cj = 0;
      if constexpr (STR) {
        cd = (ok ? st.dw[j] : 0.0) + iz * st.dz;
        cj = ok ? stretch_class(st.mol_of[j], st.phantom) : 0;
        if (cj) ljj2 = -1.0;   // LJ between mobile beads only
      }
#pragma unroll 1
      for (int i = 0; i < np; i++) {
        const double4 qp = sh.s_pt[i];
        const double dx = cx - qp.x, dy = cy - qp.y, dz = cz - qp.z;
        const double r2 = dx * dx + dy * dy + dz * dz;
        double n2 = 0;
        if constexpr (STR) {
          // the same rounding of dz in both separations
          const double dn = dz + (cd - sh.s_ptd[i]);
          n2 = dx * dx + dy * dy + dn * dn;
        }
        // FP64 queue: every charged pair (P = 0), the close ones (P = 1)
        // ALL: a pair counts from its lower index
        const int own = ALL ? sh.s_own[i] : -1;
        const bool in = r2 <= rcj2 && (!ALL || j > own) && (!STR || stretch_pair(sh.s_cls[i], cj));
        const bool near = in && (P == 0 || r2 < fp64_b2);
        const unsigned long long m = __ballot(near);
        if (m) {
          if (near) {
            sm.s_q[qn + lanes_below(m)] = make_double2(r2, qp.w * qj);
            if constexpr (STR) sm.s_qn[qn + lanes_below(m)] = n2;
          }
          qn += __popcll(m);
          if (qn >= kWave) drain(kWave);
        }
        if (P == 1) {
          // each queue drains pairs of one precision at a time, so the lanes
          // of a drain never split between the two
          const bool far = in && !near;
          const unsigned long long mf = __ballot(far);
          if (mf) {
            if (far) sm.s_f[fn + lanes_below(mf)] = make_float2((float)r2, (float)(qp.w * qj));
            fn += __popcll(mf);
            if (fn >= kWave) drain32(kWave);
          }
        }
        const bool lj = r2 < ljj2 && (!ALL || j > own) && (!STR || sh.s_cls[i] == 0);
        const unsigned long long ml = __ballot(lj);
        if (ml) {
          if (lj) {
            const int k = ln + lanes_below(ml);
            sm.s_lr[k] = r2;
            if constexpr (STR) sm.s_ln[k] = n2;
            sm.s_lt[k] = sh.s_ptt[i] * nt + tj;
          }
          ln += __popcll(ml);
          if (ln >= kWave) drain_lj(kWave);
        }
      }
      it = it2;
      j = j2;
      tj = tj2;
      img = img2;
      pj = pj2;
    }
    __syncthreads();   // the next chunk rewrites the cell arrays
  }
  if (qn > 0) drain(qn);
  if (P == 1 && fn > 0) drain32(fn);
  if (ln > 0) drain_lj(ln);
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
    elj += __shfl_down(elj, off, kWave);
    ere += __shfl_down(ere, off, kWave);
  }
  return make_double2(elj, ere);
}

// Cross block: LJ + real pairs between slot q's and slot p's moved beads,
// u(i',j') - u(i,j') - u(i',j) + u(i,j): the change of either one's dE when
// the other has been accepted (same pair functions as the moved-moved pairs).
__device__ void cross_block(const Geo& g, const Dev& d, const RepCfg& rc, int sp, int sq, int np_, int nq,
                            int local, double* sh, double2* out) {
  const int t = local * kBlock + threadIdx.x;
  double elj = 0, ere = 0;
  if (t < np_ * nq) {
    const int i = t / np_, j = t - (t / np_) * np_;
    const int si = sq * rc.maxm + i, sj = sp * rc.maxm + j;
    const double4 a0 = d.mv_old[si], a1 = d.mv_new[si], b0 = d.mv_old[sj], b1 = d.mv_new[sj];
    const LJPair lp = d.lj[d.mv_type[si] * g.n_types + d.mv_type[sj]];
    pair_both(a1, b1, lp, g, 1.0, elj, ere);
    pair_both(a0, b1, lp, g, -1.0, elj, ere);
    pair_both(a1, b0, lp, g, -1.0, elj, ere);
    pair_both(a0, b0, lp, g, 1.0, elj, ere);
  }
  const double a = block_sum<kBlock>(elj, sh);
  const double c = block_sum<kBlock>(ere, sh);
  if (threadIdx.x == 0) *out = make_double2(a, c);
}

struct CSpecSmem {
  double sh[kBlock / kWave];
};

// What a block of k_compute_spec reads of the plan, one array element per
// lane, every load issued before the first is used: a block finds its slot or
// pair by one ballot over the prefix it holds instead of walking the prefix
// with one dependent global read per step (up to 15 steps for a slot and 119
// for a pair, about half a microsecond each).
struct PlanLanes {
  int ne, qb, nn;      // exact slots, blocks per query, near pairs (scalar)
  int q, mm, scr;      // lane l: q_off[l], mm_off[l] (l <= ne), screen_of[l] (l < ne)
  int off0, off1;      // pair_off[l], pair_off[l + 64]
  int pq0, pq1;        // slots of pairs l and l + 64, p | q << 8
};

__device__ __forceinline__ PlanLanes plan_lanes(const SpecPlan* plan) {
  const int lane = threadIdx.x % kWave, l16 = min(lane, kMaxProp), l1 = min(lane + kWave, kMaxPairs);
  PlanLanes L;
  const int ne = plan->n_exact, qb = plan->qblk, nn = plan->n_near;
  L.q = plan->q_off[l16];
  L.mm = plan->mm_off[l16];
  L.scr = plan->screen_of[min(lane, kMaxProp - 1)];
  L.off0 = plan->pair_off[lane];
  L.off1 = plan->pair_off[l1];
  const int p0 = plan->pair_p[lane], q0 = plan->pair_q[lane];
  const int l1p = min(l1, kMaxPairs - 1);
  const int p1 = plan->pair_p[l1p], q1 = plan->pair_q[l1p];
  L.pq0 = p0 | (q0 << 8);
  L.pq1 = p1 | (q1 << 8);
  L.ne = __builtin_amdgcn_readfirstlane(ne);
  L.qb = __builtin_amdgcn_readfirstlane(qb);
  L.nn = __builtin_amdgcn_readfirstlane(nn);
  return L;
}

// Slot e of prefix value `pre` (lane l: the blocks before slot l) that holds
// block b, for b below lane ne's value.
__device__ __forceinline__ int plan_slot(int pre, int ne, int b) {
  const int lane = threadIdx.x % kWave;
  return __popcll(__ballot(lane >= 1 && lane < ne && pre <= b));
}

template <int P>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4))) void k_compute_spec(
    const Geo* __restrict__ G, const Dev* __restrict__ D, const RepCfg* __restrict__ RC,
    const int* __restrict__ vb_count, int R) {
  __shared__ int s_pre[kMaxReplicas];
  __shared__ union {
    QueryShare<P, Q_MOVED> q;
    KTileSmem k;
  } sm;
  __shared__ CSpecSmem cs;
  int total;
  if (R == 1) {
    total = uload(vb_count);
  } else {
    for (int r = threadIdx.x; r < R; r += kBlock) s_pre[r] = vb_count[r];
    __syncthreads();
    lds_scan(s_pre, R);
    total = s_pre[R - 1];
  }
  const int lane = threadIdx.x % kWave;
  for (int vb = blockIdx.x; vb < total; vb += gridDim.x) {
    const int r = R == 1 ? 0 : __builtin_amdgcn_readfirstlane(find_replica(s_pre, R, vb));
    int b = __builtin_amdgcn_readfirstlane(vb - (r ? s_pre[r - 1] : 0));
    const Geo g = load_const(G, r);
    const Dev d = load_const(D, r);
    const RepCfg rc = load_const(RC, r);
    const PlanLanes L = plan_lanes(d.plan);
    const int ne = L.ne;
    // longest work first: queries, k space, moved-moved pairs, cross terms
    const int nqt = __builtin_amdgcn_readlane(L.q, ne), nmt = __builtin_amdgcn_readlane(L.mm, ne);
    if (b < nqt) {
      const int e = plan_slot(L.q, ne, b);
      const int local = b - __builtin_amdgcn_readlane(L.q, e);
      const Dev v = prop_view(g, d, rc, __builtin_amdgcn_readlane(L.scr, e), e);
      const int nm = uload(&v.rec->n_moved), lo = uload(&v.rec->lo), hi = uload(&v.rec->hi);
      // share local % qb of query q2 = local / qb = 2 c + on, cluster c (moved
      // beads c kCluster ..) at their old (on = 0) or new positions
      const int q2 = local / L.qb, part = local - q2 * L.qb;
      const int m0 = (q2 >> 1) * kCluster, on = q2 & 1;
      const int li = lane % kCluster, np = min(kCluster, nm - m0), pi = m0 + min(li, np - 1);
      const double4 pt = (on ? v.mv_new : v.mv_old)[pi];
      const double2 eq = real_query_cluster<P, Q_MOVED>(g, v, pt, v.mv_type[pi], li < np, 0, lo, hi, part, L.qb, sm.q);
      const double sgn = on ? 1.0 : -1.0;
      if (lane == 0) v.part_r[local * kQWaves + threadIdx.x / kWave] = make_double2(sgn * eq.x, sgn * eq.y);
    } else if ((b -= nqt) < rc.nkb_s * ne) {
      // k tile b / ne, exact slot b % ne
      const int kt = b / ne, e = b - kt * ne;
      kspace_spec_block(g, d, rc, __builtin_amdgcn_readlane(L.scr, e), kt, e, sm.k);
    } else if ((b -= rc.nkb_s * ne) < nmt) {
      const int e = plan_slot(L.mm, ne, b);
      const Dev v = prop_view(g, d, rc, __builtin_amdgcn_readlane(L.scr, e), e);
      const int nm = uload(&v.rec->n_moved);
      mm_block(g, v, b - __builtin_amdgcn_readlane(L.mm, e), nmm_blocks(nm), cs.sh);
    } else {
      b -= nmt;
      // pair j of the near list: pair_off is increasing, entry 0 is 0
      const int j = __popcll(__ballot(lane >= 1 && lane < L.nn && L.off0 <= b)) +
                    __popcll(__ballot(lane + kWave < L.nn && L.off1 <= b));
      const int off = j < kWave ? __builtin_amdgcn_readlane(L.off0, j) : __builtin_amdgcn_readlane(L.off1, j - kWave);
      const int pq = j < kWave ? __builtin_amdgcn_readlane(L.pq0, j) : __builtin_amdgcn_readlane(L.pq1, j - kWave);
      const int sp = __builtin_amdgcn_readlane(L.scr, pq & 0xff), sq = __builtin_amdgcn_readlane(L.scr, pq >> 8);
      const int np_ = uload(&d.recs[sp].n_moved), nq = uload(&d.recs[sq].n_moved);
      cross_block(g, d, rc, sp, sq, np_, nq, b - off, cs.sh, d.part_x + b);
    }
    __syncthreads();  // the LDS is reused by the next virtual block
  }
}

constexpr int kReduceThreads = 1024;
constexpr int kReduceWaves = kReduceThreads / kWave;
constexpr int kPairBlocks = (kMaxPairs + kReduceWaves - 1) / kReduceWaves;
constexpr int kReduceBlocks = 2 * kMaxProp + kGramParts + kPairBlocks;

// Blocks of a system's k-space cross sums: 384 k vectors are 96 KB of dS rows
// a block, which a compute unit takes in about 2 us (10,170 k vectors, a launch:
// 17 us by 4 blocks, 7.0 by 20, 5.9 by 27).
__device__ __forceinline__ int gram_parts(int n_kh) { return max(1, min(kGramParts, (n_kh + 383) / 384)); }

// Sums of a batch, fixed order, blocks of one system (blockIdx.y):
//   [0, kMaxProp)   k-space dE per exact slot (the k tiles' partials)
//   gram_parts      k-space cross sums 2 sum_k c_k Re(dS_p* dS_q) of all slot
//                   pairs p < q, a part of the k vectors each (the resolve adds
//                   the parts): a Gram matrix of the sixteen dS rows, so the
//                   FP64 matrix cores read each row once (lane l holds row
//                   l % 16 at k vector l / 16 of four, times c_k as A and
//                   plain as B)
//   kMaxProp        (LJ, real) sums per exact slot (query and moved-moved
//                   blocks)
//   kPairBlocks     real-space cross sums of the near pairs, a wave each
// Launch and latency bound: a block per sum (272 a system, most of them with
// nothing to do, each pair reading its two rows again) took 7.4 us for 16 slots of 10,170 k
// vectors, now 5.9, and 38 us for 24 systems.
__global__ __launch_bounds__(kReduceThreads) void k_reduce_spec(const Geo* __restrict__ G, const Dev* __restrict__ D,
                                                        const RepCfg* __restrict__ RC, int R) {
  __shared__ double sh[kReduceWaves];
  __shared__ double s_g[kReduceWaves][kMaxProp * kMaxProp];
  const int r = blockIdx.y, t = threadIdx.x, lane = t % kWave, wv = t / kWave;
  int j = blockIdx.x;
  if (r >= R) return;
  const Geo g = load_const(G, r);
  const Dev d = load_const(D, r);
  const RepCfg rc = load_const(RC, r);
  SpecPlan* plan = d.plan;
  const int np0 = plan->n_prop, ne = plan->n_exact;
  if (np0 == 0) return;
  if (j < kMaxProp) {
    if (j >= ne) return;
    double s = 0;
    const int np = rc.nkb_s * kQWaves;
    for (int i = t; i < np; i += kReduceThreads) s += d.part_ks[(size_t)j * np + i];
    s = block_sum<kReduceThreads>(s, sh);
    if (t == 0) plan->ksum[j] = s;
  } else if ((j -= kMaxProp) < kGramParts) {
    if (ne < 2) return;
    const int parts = gram_parts(g.n_kh);
    if (j >= parts) return;
    const int waves = parts * kReduceWaves, row = lane % 16, in = lane / 16;
    const int ch = ((g.n_kh + waves - 1) / waves + 3) & ~3;
    const int k0 = (j * kReduceWaves + wv) * ch, k1 = min(k0 + ch, g.n_kh);
    f64x4 acc = {0, 0, 0, 0};
    if (rc.nkb_s > 0) {
      const double2* a = d.dS + (size_t)min(row, ne - 1) * g.n_kh;
#pragma unroll 4
      for (int k = k0; k < k1; k += 4) {
        const int kk = k + in, kc = min(kk, g.n_kh - 1);
        const double2 u = a[kc];
        const double c = kk < k1 ? d.ck[kc] : 0.0;
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(c * u.x, u.x, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(c * u.y, u.y, acc, 0, 0, 0);
      }
    }
#pragma unroll
    for (int v = 0; v < 4; v++) s_g[wv][(4 * v + in) * kMaxProp + row] = acc[v];
    __syncthreads();
    const int p = t / kMaxProp, q = t % kMaxProp;
    if (p < q && q < ne) {
      double s = 0;
#pragma unroll
      for (int w = 0; w < kReduceWaves; w++) s += s_g[w][t];
      plan->kx[j][pair_index(p, q)] = 2.0 * s;
    }
  } else if ((j -= kGramParts) < kMaxProp) {
    if (j >= ne) return;
    const int nm = d.recs[plan->screen_of[j]].n_moved;
    if (nm == 0) return;
    const int nreal = query_blocks(nm, plan->qblk) * kQWaves, nmm = nmm_blocks(nm);
    const double2* pr = d.part_r + (size_t)j * rc.rstride;
    const double2* pm = d.part_mm + (size_t)j * rc.nmmb;
    double lj = 0, re = 0;
    for (int i = t; i < nreal; i += kReduceThreads) {
      lj += pr[i].x;
      re += pr[i].y;
    }
    for (int i = t; i < nmm; i += kReduceThreads) {
      lj += pm[i].x;
      re += pm[i].y;
    }
    lj = block_sum<kReduceThreads>(lj, sh);
    re = block_sum<kReduceThreads>(re, sh);
    if (t == 0) plan->rsum[j] = make_double2(lj, re);
  } else {
    const int jj = (j - kMaxProp) * kReduceWaves + wv;
    if (jj >= plan->n_near) return;
    const int off = plan->pair_off[jj], nblk = plan->pair_off[jj + 1] - off;
    double lj = 0, re = 0;
    for (int i = lane; i < nblk; i += kWave) {
      const double2 x = d.part_x[off + i];
      lj += x.x;
      re += x.y;
    }
    lj = wave_sum(lj);
    re = wave_sum(re);
    if (lane == 0) plan->xsum[jj] = make_double2(lj, re);
  }
}

// ------------------------------------------------------------ resolve
// The items of consecutive accepted exact slots committed together:
// group slot j holds items [goff[j], goff[j + 1]) of proposal gscr[j].
struct SlotItems {
  const double4* mv_new;
  const int* mv_idx;
  int maxm;
  const int* goff;
  const int* gscr;
  int ns, n;
  __device__ __forceinline__ void get(int k, double4& p, int& i) const {
    int j = 0;
    while (j + 1 < ns && goff[j + 1] <= k) j++;
    const size_t o = (size_t)gscr[j] * maxm + (k - goff[j]);
    p = mv_new[o];
    i = mv_idx[o];
  }
};

struct ResSmem {
  CommitSmem cm;
  PropInfo s_prop[kMaxScreen];
  double s_bcur[kMaxScreen];
  int s_len[kMaxScreen];
  double s_u[kMaxScreen];
  double s_des[kMaxScreen];
  int s_pass[kMaxScreen];
  int s_exact[kMaxScreen];
  int s_screen[kMaxProp];
  double2 s_rsum[kMaxProp];
  double s_ksum[kKVals];
  double2 s_xsum[kMaxPairs];
  int s_near[kMaxPairs];
  int s_train[kMaxProp];         // ring slot of a training sample per exact slot, -1 none
  int s_drec[kMaxScreen];        // decision-record index of a proposal, -1 none
  int s_goff[kMaxProp + 1], s_gscr[kMaxProp];
  int s_mask, s_ndone;
  double s_Mz, s_dipl, s_total, s_run[8];   // control block: dipole moment, dipole lag, last total, running totals
};

static_assert(kMaxScreen <= kWave, "one lane per proposal in the decision wave");

// The reference's sequential Metropolis chain over the batch
// (simulation.cc:241-355), one wave, one lane per proposal.  A pass
// evaluates every undecided proposal against the acceptances so far; the
// proposals before the first acceptance (or stop) of the pass are decided
// as they would be one after the other, since nothing they read changes
// until then.  The accepted one updates the cross terms, the dipole moment
// and the stop conditions of the proposals after it, and the next pass
// starts behind it: one pass per acceptance instead of one step per
// proposal.  Each dE adds the cross terms in acceptance order, which is the
// order of increasing exact slot, as the one-at-a-time chain does.
__device__ void resolve_decide(const Geo& g, const Dev& d, const RepCfg& rc, Ctl* C, SpecPlan* plan, int np,
                               int ndec, unsigned long long ctr0, ResSmem& sm) {
  const int lane = threadIdx.x;
  const bool mine = lane < np;
  PropInfo P = {};
  P.prev = -1;
  P.type = -1;
  if (mine) P = sm.s_prop[lane];
  const int e = mine ? sm.s_exact[lane] : -1;
  const int pass = mine ? sm.s_pass[lane] : 0;
  const double des = mine ? sm.s_des[lane] : 0.0, u = mine ? sm.s_u[lane] : 1.0;
  const int len = mine ? sm.s_len[lane] : 0;
  const double bcur = mine ? sm.s_bcur[lane] : 0.0;
  const int use_pair = g.use_pair, use_ext = g.use_ext, use_ewald = g.use_ewald, use_bond = g.use_bond;
  const int dipole = g.dipole, dipole_exact = g.dipole_exact, da_on = rc.da, train = rc.train;
  const double dip_coef = g.dip_coef, beta = g.beta;
  // pair and k-space dE against the state before the batch (a proposal that
  // moves no bead has no real-space blocks: its pair terms are zero), plus
  // the cross terms of the acceptances so far
  double lj = 0, re = 0, kk = 0;
  if (e >= 0) {
    lj = P.n > 0 ? sm.s_rsum[e].x : 0.0;
    re = P.n > 0 ? sm.s_rsum[e].y : 0.0;
    kk = sm.s_ksum[e];
  }
  const bool evaluated = P.valid && (pass || e >= 0);
  bool stop_prev = false, stale = false;
  unsigned mask = 0;
  double Mz = sm.s_Mz, cur_dipl = sm.s_dipl;
  double run[8];
  for (int k = 0; k < 8; k++) run[k] = sm.s_run[k];
  // what each proposal was decided with
  double f_tt[8] = {0, 0, 0, 0, 0, 0, 0, 0}, f_dE = 0, f_target = 0;
  bool f_acc = false, f_early = false;
  int done = ndec, cut = 0, s = 0;
  while (s < ndec) {
    // ForceField::EnergyDifference with its early exits (force_field.cc:407-434)
    double tt[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    double dE = 0;
    bool early = false;
    if (use_pair) {
      tt[T_LJ] = lj;
      dE += lj;
      if (dE >= kVeryLargeEnergy) early = true;
    }
    if (!early && use_ext) {
      tt[T_WALL] = P.forbid ? kVeryLargeEnergy : P.ew;
      dE += tt[T_WALL];
      if (dE >= kVeryLargeEnergy) early = true;
    }
    double trial_dipl = cur_dipl;
    if (!early && use_ewald) {
      tt[T_REAL] = re;
      tt[T_KSPACE] = kk;
      double dd = 0;
      if (dipole) {
        if (dipole_exact) {
          const double mz1 = Mz + P.dmz;
          trial_dipl = dipole_energy(dip_coef, mz1);
          dd = dipole_change(trial_dipl, dipole_energy(dip_coef, Mz));
        } else {
          // potential_ewald.cc:528-531: dipole of the CURRENT coordinates
          trial_dipl = dipole_energy(dip_coef, Mz);
          dd = dipole_change(trial_dipl, cur_dipl);
        }
      }
      tt[T_DIPOLE] = dd;
      dE += re + kk + dd;
    }
    if (!early && use_bond && len > 1) {
      tt[T_BOND] = P.bond_trial - bcur;
      dE += tt[T_BOND];
    }
    // Metropolis (simulation.cc:327-332), no draw for a forbidden move; with
    // the surrogate, the second stage min(1, exp(-beta (dE - dE_s)))
    const bool acc = evaluated && pass && (dE < kVeryLargeEnergy) && (u < exp(-beta * (dE - des)));
    const bool stop = stop_prev || stale;
    const bool open = lane >= s && lane < ndec;
    const unsigned long long ev = __ballot(open && (stop || acc));
    const int f = ev ? __builtin_ctzll(ev) : ndec;
    if (open && (lane < f || (lane == f && !stop))) {
      for (int k = 0; k < 8; k++) f_tt[k] = tt[k];
      f_dE = dE;
      f_early = early;
      f_acc = lane == f;
      f_target = lj + re + kk;
    }
    if (f >= ndec) break;
    if (__builtin_amdgcn_readlane((int)stop, f)) {
      // a proposal made on the assumption that its molecule's earlier
      // proposal in the batch is rejected, or whose surrogate value could see
      // an acceptance of this batch: it is made again next batch
      done = f;
      cut = __builtin_amdgcn_readlane((int)(stale && !stop_prev), f);
      break;
    }
    // proposal f is accepted
    const int ef = __builtin_amdgcn_readlane(e, f);
    mask |= 1u << ef;
    Mz += lane_double(P.dmz, f);
    if (dipole) cur_dipl = lane_double(trial_dipl, f);
    for (int k = 0; k < 8; k++) run[k] += lane_double(tt[k], f);
    if (lane == f && use_bond && len > 1) d.bond_cur[P.mol] = P.bond_trial;
    const double fc0 = lane_double(P.c[0], f), fc1 = lane_double(P.c[1], f), fc2 = lane_double(P.c[2], f);
    const double frad = lane_double(P.rad, f);
    if (lane > f && lane < ndec) {
      if (e >= 0) {
        const int pi = pair_index(ef, e);
        kk += sm.s_ksum[kMaxProp + pi];
        const int j = sm.s_near[pi];
        if (j >= 0) {
          lj += sm.s_xsum[j].x;
          re += sm.s_xsum[j].y;
        }
      }
      if (P.prev == f) stop_prev = true;
      if (da_on) {
        const double fc[3] = {fc0, fc1, fc2};
        stale = stale || center_dist(fc, P.c, g) <= frad + P.rad + (double)rc.r_d + 1e-9;
      }
    }
    s = f + 1;
  }
  // counters of the decided proposals
  const bool decided = lane < done;
  const bool valid = decided && P.valid;
  long long att[5], acc5[5];
  for (int k = 0; k < 5; k++) {
    att[k] = __popcll(__ballot(valid && P.type == k));
    acc5[k] = __popcll(__ballot(valid && f_acc && P.type == k));
  }
  const long long n_valid = __popcll(__ballot(valid));
  const long long skipped = __popcll(__ballot(decided && !P.valid && P.skipped));
  const long long s1r = __popcll(__ballot(valid && !pass));
  const long long tev = __popcll(__ballot(valid && !pass && e >= 0));
  const long long s1p = da_on ? __popcll(__ballot(valid && pass)) : 0;
  if (d.drec) {
    // bounded record of the decided proposals, in decision order: the terms
    // and total the Metropolis test was given (trial positions copied by
    // the block afterwards)
    const unsigned long long rm = __ballot(valid);
    const int rhead = d.drec_ctl[0], rcap = d.drec_ctl[1];
    int slot = -1;
    if (valid) {
      const int k = rhead + lanes_below(rm);
      if (k < rcap) {
        slot = k;
        DecRec& o = d.drec[k];
        o.move = ctr0 + lane;
        o.mol = P.mol;
        o.n = P.n;
        o.type = P.type;
        o.accepted = f_acc ? 1 : 0;
        o.lo = d.recs[lane].lo;
        o.hi = d.recs[lane].hi;
        o.contig = d.recs[lane].contig;
        o.evaluated = evaluated ? 1 : 0;
        o.early = f_early ? 1 : 0;
        o.pass = pass;
        o.pad0 = o.pad1 = 0;
        for (int k2 = 0; k2 < 8; k2++) o.terms[k2] = f_tt[k2];
        o.total = f_dE;
        o.de_s = des;
      }
    }
    if (mine) sm.s_drec[lane] = slot;
    if (lane == 0) d.drec_ctl[0] = rhead + (int)__popcll(rm);
  }
  // training samples in proposal order: the pair + k-space part the network
  // estimates
  int head = train ? d.tr_ctl[0] : 0;
  const int ring = train ? d.tr_ctl[1] : 0;
  const bool sample = valid && e >= 0 && train && !f_early && P.n > 0 && ring > 0;
  const unsigned long long smask = __ballot(sample);
  if (sample) {
    const int slot = (head + lanes_below(smask)) % ring;
    d.tr_target[slot] = f_target;
    d.tr_n[slot] = P.n;
    sm.s_train[e] = slot;
  }
  head += __popcll(smask);
  // the terms of the last proposal that reached the Metropolis test
  const unsigned long long lm = __ballot(valid && pass);
  double last[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  double last_total = sm.s_total;
  if (lm) {
    const int l = 63 - __builtin_clzll(lm);
    for (int k = 0; k < 8; k++) last[k] = lane_double(f_tt[k], l);
    last_total = lane_double(f_dE, l);
  }
  // the counters, one lane each: a read-modify-write is a round trip, so lane 0
  // adding to the sixteen of them in turn would wait sixteen times
  {
    const long long one[6] = {n_valid, skipped, s1r, s1p, tev, (long long)cut};
    long long inc = 0;
    for (int k = 0; k < 5; k++) {
      if (lane == k) inc = att[k];
      if (lane == 5 + k) inc = acc5[k];
    }
    for (int k = 0; k < 6; k++)
      if (lane == 10 + k) inc = one[k];
    if (lane < kCtlCounters) (&C->attempted[0])[lane] += inc;
  }
  if (lane == 0) {
    C->Mz = Mz;
    C->cur_dipl = cur_dipl;
    C->trial_dipl = cur_dipl;
    for (int k = 0; k < 8; k++) {
      C->running[k] = run[k];
      C->terms[k] = last[k];
    }
    C->total = last_total;
    C->move_counter = ctr0 + done;
    if (train) d.tr_ctl[0] = head;
    plan->acc_mask = mask;
    sm.s_mask = mask;
    sm.s_ndone = done;
  }
}

__global__ __launch_bounds__(kBlock) void k_resolve_spec(const Geo* __restrict__ G, const Dev* __restrict__ D,
                                                         const McDev* __restrict__ MC,
                                                         const RepCfg* __restrict__ RC, int R) {
  __shared__ ResSmem sm;
  const int r = blockIdx.x;
  if (r >= R) return;
  const Geo g = load_const(G, r);
  const Dev d = load_const(D, r);
  const McDev mc = load_const(MC, r);
  const RepCfg rc = load_const(RC, r);
  Ctl* C = d.ctl;
  SpecPlan* plan = d.plan;
  // everything the decisions read, fetched in parallel and before the counts
  // that say how much of it is in use are known
  const int t = threadIdx.x;
  const int np = plan->n_prop, ndec = plan->n_decide, nn = plan->n_near;
  const unsigned long long ctr0 = C->move_counter;
  int pp = 0, pq = 0;
  if (t < kMaxScreen) {
    const PropInfo P = d.prop[t];
    const double des = plan->de_s[t];
    const int pass = plan->pass1[t], exact = plan->exact_of[t];
    sm.s_prop[t] = P;
    sm.s_bcur[t] = P.bcur;
    sm.s_len[t] = P.len;
    sm.s_des[t] = des;
    sm.s_pass[t] = pass;
    sm.s_exact[t] = exact;
    const unsigned long long ctr = ctr0 + t;
    const uint4 u = Philox::gen(make_uint4((uint32_t)ctr, (uint32_t)(ctr >> 32), 0xACCu, 0u),
                                make_uint2((uint32_t)mc.seed, (uint32_t)(mc.seed >> 32)));
    sm.s_u[t] = u01_32(u.x);
  }
  if (t >= 64 && t < 64 + kKVals) {
    const int i = t - 64;
    double v = 0;
    if (i < kMaxProp) {
      v = plan->ksum[i];
    } else {
      const int parts = gram_parts(g.n_kh);
      for (int u0 = 0; u0 < parts; u0 += 16) {   // sixteen loads in flight
        double x[16];
#pragma unroll
        for (int u = 0; u < 16; u++) x[u] = plan->kx[min(u0 + u, parts - 1)][i - kMaxProp];
#pragma unroll
        for (int u = 0; u < 16; u++) v += u0 + u < parts ? x[u] : 0.0;
      }
    }
    sm.s_ksum[i] = v;
  }
  if (t >= 128 && t < 128 + kMaxPairs) {
    const int j = t - 128;
    pp = plan->pair_p[j];
    pq = plan->pair_q[j];
    sm.s_near[j] = -1;
    sm.s_xsum[j] = plan->xsum[j];
  }
  if (t >= 192 && t < 192 + kMaxProp) {
    sm.s_rsum[t - 192] = plan->rsum[t - 192];
    sm.s_screen[t - 192] = plan->screen_of[t - 192];
    sm.s_train[t - 192] = -1;
  }
  if (t >= 224 && t < 224 + kMaxScreen) sm.s_drec[t - 224] = -1;
  if (t == kBlock - 1) {
    sm.s_Mz = C->Mz;
    sm.s_dipl = C->cur_dipl;
    sm.s_total = C->total;
  }
  if (t >= kBlock - 9 && t < kBlock - 1) sm.s_run[t - (kBlock - 9)] = C->running[t - (kBlock - 9)];
  if (np == 0) return;
  __syncthreads();
  if (t >= 128 && t < 128 + nn) sm.s_near[pair_index(pp, pq)] = t - 128;
  __syncthreads();
  if (t < kWave) resolve_decide(g, d, rc, C, plan, np, ndec, ctr0, sm);
  __syncthreads();
  if (d.drec) {
    // trial positions and bead indices of the recorded proposals
    for (int s = 0; s < np; s++) {
      const int slot = sm.s_drec[s];
      if (slot < 0) continue;
      const int n = sm.s_prop[s].n;
      for (int i = t; i < n; i += kBlock) {
        d.drec_pos[(size_t)slot * rc.maxm + i] = d.mv_new[(size_t)s * rc.maxm + i];
        d.drec_idx[(size_t)slot * rc.maxm + i] = d.smv_idx[(size_t)s * rc.maxm + i];
      }
    }
  }
  // cell-list commits of the accepted slots, as many slots at a time as the
  // item arrays hold
  const unsigned mask = sm.s_mask;
  int e0 = 0;
  while (e0 < kMaxProp) {
    if (e0 > 0) __syncthreads();   // the last group's commit is done with the group arrays
    int ns = 0, n = 0, e = e0;
    for (; e < kMaxProp; e++) {
      if (!(mask & (1u << e))) continue;
      const int nm = sm.s_prop[sm.s_screen[e]].n;
      if (ns > 0 && n + nm > kMaxChainDev) break;
      if (t == 0) {
        sm.s_goff[ns] = n;
        sm.s_gscr[ns] = sm.s_screen[e];
      }
      ns++;
      n += nm;
    }
    e0 = e;
    if (ns == 0) break;
    if (t == 0) sm.s_goff[ns] = n;
    __syncthreads();
    commit_cells(g, d, SlotItems{d.mv_new, d.smv_idx, rc.maxm, sm.s_goff, sm.s_gscr, ns, n}, sm.cm);
  }
  if (rc.train) {
    // descriptor rows of the training samples (old rows, then new rows)
    for (int e = 0; e < kMaxProp; e++) {
      const int slot = sm.s_train[e];
      if (slot < 0) continue;
      const int s = sm.s_screen[e];
      const int n = sm.s_prop[s].n;
      const float* src = d.sur_x + (size_t)(2 * s) * rc.maxm * kDescr;
      float* dst = d.tr_x + (size_t)slot * 2 * rc.maxm * kDescr;
      for (int i = threadIdx.x; i < n * kDescr; i += kBlock) {
        dst[i] = src[i];
        dst[(size_t)rc.maxm * kDescr + i] = src[(size_t)rc.maxm * kDescr + i];
      }
    }
  }
}

// Folds the pending accepted dS_e(k) into S(k) (end of a run) and clears the
// mask, one block per system.
constexpr int kFlushThreads = 1024;
__global__ __launch_bounds__(kFlushThreads) void k_flush_spec(const Geo* __restrict__ G, const Dev* __restrict__ D) {
  const int r = blockIdx.x;
  const Geo& g = G[r];
  const Dev& d = D[r];
  const unsigned mask = d.plan->acc_mask;
  if (!mask) return;
  for (int k = threadIdx.x; k < g.n_kh; k += kFlushThreads) {
    double2 s = d.Sk[k];
    for (int e = 0; e < kMaxProp; e++)
      if (mask & (1u << e)) {
        const double2 ds = d.dS[(size_t)e * g.n_kh + k];
        s.x += ds.x;
        s.y += ds.y;
      }
    d.Sk[k] = s;
  }
  __syncthreads();
  if (threadIdx.x == 0) d.plan->acc_mask = 0;
}

// Tombstone compaction of every system's cells; cell_off is the exclusive
// prefix of the cell counts (R + 1 entries).  A cell is a chain of dependent
// reads (count, slots, their contents): by one thread, slot after slot, 50 to
// 130 us a launch whatever the number of cells (longest where few cells hold
// many beads); by a wave, 64 slots at a time.  A wave takes `per` (up to 64)
// cells, reads their counts together and visits the occupied ones: with a wave
// for every cell, 2.1 million nearly all empty took 190 us a launch, 8.7 so.
__global__ __launch_bounds__(kBlock) void k_compact_batch(const Geo* __restrict__ G, const Dev* __restrict__ D,
                                                          const int* __restrict__ cell_off, int R, int per) {
  const int lane = threadIdx.x % kWave;
  const int gid = (blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave) * per + lane;
  int cell = 0, lo = 0, cnt = 0;
  if (lane < per && gid < cell_off[R]) {
    int hi = R - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (cell_off[mid] <= gid) lo = mid;
      else hi = mid - 1;
    }
    cell = gid - cell_off[lo];
    cnt = D[lo].ccount[cell];
  }
  for (unsigned long long m = __ballot(cnt > 0); m; m &= m - 1) {
    const int l = __builtin_ctzll(m);
    const int r = __builtin_amdgcn_readlane(lo, l);
    compact_cell_wave(G[r], D[r], __builtin_amdgcn_readlane(cell, l));
  }
}

// Per system: overflow flag and moves still to propose (read by the host
// between graph replays).
__global__ void k_batch_status(const Dev* __restrict__ D, const McDev* __restrict__ MC, int R, int2* out) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= R) return;
  const unsigned long long c = D[r].ctl->move_counter, lim = MC[r].ctr_limit;
  out[r] = make_int2(D[r].ctl->overflow, c < lim ? (int)min(lim - c, 1ull << 30) : 0);
}

}  // namespace plum
