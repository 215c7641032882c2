// Configurational-bias growth of a whole chain on the device: every growth
// step of an insertion, a deletion or a Widom test insertion (cbmc.cc:213-533)
// is one launch, the trial draws made beforehand by the host in the
// reference's order.
//   k_grow_init    S_x(k) = S(k) - S_excluded(k), Rosenbluth weight 1
//   k_grow_step    launch s = 0 .. L - 1: every block first finishes step s - 1
//                  (grow_select: the trial energies from its partial sums, the
//                  weights, W *= W_s / K, the choice of the bead -- insertion:
//                  by the pre-drawn uniform; deletion: the existing bead, trial
//                  0), then does its part of step s: part 1 (cell list, LJ +
//                  real space), parts 2-4 (the grown chain, the bead-counterion
//                  pair, self images, walls; one block per trial) or the k-space
//                  sums of a trial bead and counterion, positions built from the
//                  bead just chosen.
//   k_grow_select  the end of the last step, and of every step where repeating
//                  it in each block costs more than a launch (many trials,
//                  grow_fused): by one block.
// With few trials the choice is a few hundred loads and K exponentials, so it
// is repeated in every block rather than made by one in a launch between the
// steps: at 16 trials, 3,200 beads, an insertion and a deletion of 32 beads take
// 1543 -> 1080 us, a step 24 -> 15 us; a step is latency (chains of dependent
// loads, the queue of the query, a launch), not bytes or operations.  All blocks
// compute the same bits, and so does the one block.  What a launch reads and
// the next one's value of (state, S_x, partial sums) live in two buffers used in
// turn; block 0 writes the state, the blocks of trial 0 write S_x.
// Step 0 is the first bead (and its counterion) alone, trial 0 of K.
#pragma once
#include "kernels_batch.h"
#include "kernels_cbmc.h"

namespace plum {

struct GrowIn {
  int K, L, mode, charged;   // mode 0 insertion, 1 deletion, 2 test insertion
  int type_c, type_i, ex_lo, ex_hi;
  double q_c, q_i;
};

static_assert(sizeof(GrowIn) % alignof(double) == 0, "the random numbers follow GrowIn in one buffer");

struct GrowOut {
  double W;       // Rosenbluth weight
  int stop;       // step at which the weight reached 0 (-1: grown to the end)
  int pad;
  // slab dipole: sum of q z over the system less the excluded beads plus the
  // chain beads chosen so far, and over the counterions chosen so far
  double mz_c, mz_i;
};

// Random numbers and known positions of one growth, one upload:
//   first[6]            first chain bead, its counterion (insertion)
//   disp[L K 3]         step s, trial t: bond vector from the bead of step s-1
//   ion[L K 3]          step s, trial t: counterion position
//   sel[L]              step s: uniform of the choice among the trials
//   act[2 L 3]          deletion: the chain's beads, then its counterions
__host__ __device__ inline size_t grow_rnd_size(int K, int L) { return 6 + 6 * (size_t)L * K + L + 6 * (size_t)L; }

struct GrowPtr {
  const double *first, *disp, *ion, *sel, *act;
};

__device__ __forceinline__ GrowPtr grow_ptr(const double* rnd, int K, int L) {
  GrowPtr p;
  p.first = rnd;
  p.disp = rnd + 6;
  p.ion = p.disp + 3 * (size_t)L * K;
  p.sel = p.ion + 3 * (size_t)L * K;
  p.act = p.sel + L;
  return p;
}

// Trial t of step s: chain bead r1 and counterion r2; prev is the chain bead
// of step s - 1.
__device__ __forceinline__ void grow_trial(const GrowIn& in, const GrowPtr& p, const double* prev, int s, int t,
                                           double r1[3], double r2[3]) {
  const int L = in.L, K = in.K;
  if (s == 0) {
    const double* a = in.mode == 1 ? p.act : p.first;
    const double* b = in.mode == 1 ? p.act + 3 * (size_t)L : p.first + 3;
#pragma unroll
    for (int k = 0; k < 3; k++) {
      r1[k] = a[k];
      r2[k] = b[k];
    }
  } else if (in.mode == 1 && t == 0) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
      r1[k] = p.act[3 * (size_t)s + k];
      r2[k] = p.act[3 * (size_t)(L + s) + k];
    }
  } else {
    const double* d = p.disp + 3 * ((size_t)s * K + t);
    const double* e = p.ion + 3 * ((size_t)s * K + t);
#pragma unroll
    for (int k = 0; k < 3; k++) {
      r1[k] = prev[k] + d[k];
      r2[k] = e[k];
    }
  }
}

constexpr int kInitK = 16;   // k vectors per block of k_grow_init, over 16 groups of excluded beads

__global__ __launch_bounds__(kBlock) void k_grow_init(Geo g, Dev d, const GrowIn* __restrict__ in,
                                                      double2* __restrict__ Sx, GrowOut* __restrict__ out) {
  __shared__ double sh[kBlock / kWave];
  if (blockIdx.x == 0 && g.dipole && g.use_ewald) {
    // M_z of the system less the excluded beads (DipoleEDiff's molecule
    // loop, potential_ewald_coul.cc:485-506)
    double m = 0;
    for (int j = threadIdx.x; j < g.n; j += kBlock)
      if (j < in->ex_lo || j > in->ex_hi) m += d.q[j] * d.z[j];
    m = block_sum<kBlock>(m, sh);
    if (threadIdx.x == 0) {
      out->mz_c = m;
      out->mz_i = 0;
    }
  }
  __shared__ double2 s_ex[kBlock / kInitK][kInitK];
  const int kk = threadIdx.x % kInitK, grp = threadIdx.x / kInitK, k = blockIdx.x * kInitK + kk;
  const bool in_k = g.use_ewald && k < g.n_kh;
  double2 ex = make_double2(0, 0);
  if (in_k) {
    const int4 l = d.kl[k];
    for (int j = in->ex_lo + grp; j <= in->ex_hi; j += kBlock / kInitK) {
      const double r[3] = {d.x[j], d.y[j], d.z[j]};
      const double2 e = phase(g, l, r);
      ex.x += d.q[j] * e.x;
      ex.y += d.q[j] * e.y;
    }
  }
  s_ex[grp][kk] = ex;
  __syncthreads();
  if (in_k && grp == 0) {
    double2 S = d.Sk[k];
    for (int u = 0; u < kBlock / kInitK; u++) {
      S.x -= s_ex[u][kk].x;
      S.y -= s_ex[u][kk].y;
    }
    Sx[k] = S;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    out->W = 1.0;
    out->stop = -1;
  }
}

// Parts 2-4 of trial t (cbmc.cc:52-151): LJ with the grown chain (not the
// bonded previous bead) and real space with it over every image within rc,
// the bead-counterion pair, the half self images, the walls, one thread per
// pair.  The beads of step cur - 1 are at prev (chain bead, counterion).
// Returns (pair energy, real-space energy) in thread 0.
__device__ double2 grow_explicit(const Geo& g, const Dev& d, const GrowIn& in, const double* grown, const double* prev,
                                 int cur, const double r1[3], const double r2[3], double* sh) {
  const int L = in.L, ch = in.charged, tc = in.type_c, ti = in.type_i, nt = g.n_types;
  const LJPair* lj = d.lj;
  double elj = 0, ere = 0;
  for (int q = threadIdx.x; q < 4 * cur + 3; q += kBlock) {
    if (q < 4 * cur) {
      const int i = q % cur, kind = q / cur;   // (r1|r2) x (chain|ion)
      if (kind > 0 && !ch) continue;
      const double* a = kind < 2 ? r1 : r2;
      const double* b = i == cur - 1 ? prev + 3 * (kind & 1) : grown + 3 * (size_t)((kind & 1) ? L + i : i);
      if (g.use_pair && !(kind == 0 && i == cur - 1))
        elj += lj_energy(bb_dist(a, b, g.Lsim, g.npbc), lj[((kind < 2) ? tc : ti) * nt + ((kind & 1) ? ti : tc)]);
      if (g.use_ewald) ere += real_pair(a, kind < 2 ? in.q_c : in.q_i, b, (kind & 1) ? in.q_i : in.q_c, g);
    } else if (g.use_ewald) {
      const int o = q - 4 * cur;   // self images of bead and counterion, their pair
      if (o > 0 && !ch) continue;
      const double* a = o == 0 ? r1 : r2;
      const double* b = o == 1 ? r2 : r1;
      ere += (o == 2 ? 1.0 : 0.5) * real_pair(a, o == 0 ? in.q_c : in.q_i, b, o == 1 ? in.q_i : in.q_c, g);
    }
  }
  const double a = block_sum<kBlock>(elj, sh);
  const double b = block_sum<kBlock>(ere, sh);
  double pair_e = a;
  if (threadIdx.x == 0) {
    if (g.use_pair && ch) pair_e += lj_energy(bb_dist(r1, r2, g.Lsim, g.npbc), lj[tc * nt + ti]);
    if (g.use_ext) {
      pair_e += wall_energy(r1[2], d.wall[tc], g);
      if (ch) pair_e += wall_energy(r2[2], d.wall[ti], g);
    }
  }
  return make_double2(pair_e, b);
}

constexpr int kMaxGrowSplit = 16;   // most blocks per trial bead's cell-list query

// Buffers of a growth; [2]: used in turn by the launches.
struct GrowBuf {
  const GrowIn* in;
  const double* rnd;
  double* grown;
  double2* Sx[2];
  GrowOut* out;        // two states: out[s & 1] before step s
  double2* cells[2];   // [bead][trial][split][wave]
  double2* expl[2];    // [trial]
  double* kpart[2];    // [trial][k block]
};

struct GrowSelSmem {
  double s_w[kCbmcMaxTrials];   // weights of the trials
  double s_pos[6];
  int s_go;
};

// The end of step s: its trial energies, weight and choice; the chosen bead
// and counterion in sm.s_pos.  Returns false when the growth stops (or has
// stopped).  Block 0 writes the state before step s + 1 and the chosen beads.
__device__ bool grow_select(const Geo& g, const GrowBuf& B, const GrowIn& in, const GrowPtr& p, int s, int nparts,
                            int nkb, GrowSelSmem& sm) {
  const GrowOut st = B.out[s & 1];
  if (st.stop >= 0) {
    if (blockIdx.x == 0 && threadIdx.x == 0) B.out[(s + 1) & 1] = st;
    return false;
  }
  const int K = in.K, L = in.L, Kt = s == 0 ? 1 : K, ch = in.charged;
  const double2* cells = B.cells[s & 1];
  const double* prev = s > 0 ? B.grown + 3 * (size_t)(s - 1) : nullptr;
  // 16 lanes per trial
  constexpr int G = 16;
  const int l16 = threadIdx.x % G;
  for (int t = threadIdx.x / G; t < Kt; t += blockDim.x / G) {
    double elj = 0, ere = 0, ek = 0;
    const int np = nparts * kQWaves;
    for (int i = l16; i < np; i += G) {
      const double2 a = cells[(size_t)t * np + i];
      elj += a.x;
      ere += a.y;
      if (ch) {
        const double2 b = cells[(size_t)(K + t) * np + i];
        elj += b.x;
        ere += b.y;
      }
    }
    for (int i = l16; i < nkb; i += G) ek += B.kpart[s & 1][(size_t)t * nkb + i];
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) {
      elj += __shfl_xor(elj, o, kWave);
      ere += __shfl_xor(ere, o, kWave);
      ek += __shfl_xor(ek, o, kWave);
    }
    if (l16 == 0) {
      const double2 x = B.expl[s & 1][t];
      const double pair_e = elj + x.x;
      double ewald_e = 0;
      if (g.use_ewald && pair_e < kVeryLargeEnergy) {
        ewald_e = ere + x.y + ek + g.self_coef * in.q_c * in.q_c;
        if (ch) ewald_e += g.self_coef * in.q_i * in.q_i;
        if (g.dipole) {
          double r1[3], r2[3];
          grow_trial(in, p, prev, s, t, r1, r2);
          ewald_e += dipole_ediff(g.dip_coef, st.mz_c + st.mz_i, in.q_c * r1[2], ch ? in.q_i * r2[2] : 0.0);
        }
      }
      const double e = pair_e >= kVeryLargeEnergy ? kVeryLargeEnergy : pair_e + ewald_e;
      sm.s_w[t] = exp(-g.beta * e);
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    // weights in trial order, summed as the reference sums them
    double Wi = 0;
    for (int t = 0; t < Kt; t++) Wi += sm.s_w[t];
    GrowOut o = st;
    int go = 1, cb = 0;
    if (s == 0) {
      o.W *= sm.s_w[0];
      if (in.mode == 0 && o.W <= 0) go = 0;
    } else {
      o.W *= Wi / K;
      if (in.mode != 1 && o.W <= 0) go = 0;
      if (go && in.mode != 1) {
        const double rn = p.sel[s] * Wi;
        double cum = sm.s_w[0];
        while (cum < rn && cb < K - 1) {
          cb++;
          cum += sm.s_w[cb];
        }
      }
    }
    if (!go) o.stop = s;
    sm.s_go = go;
    if (go) {
      double r1[3], r2[3];
      grow_trial(in, p, prev, s, cb, r1, r2);
      for (int k = 0; k < 3; k++) {
        sm.s_pos[k] = r1[k];
        sm.s_pos[3 + k] = r2[k];
      }
      if (g.dipole && g.use_ewald) {
        o.mz_c += in.q_c * r1[2];
        if (ch) o.mz_i += in.q_i * r2[2];
      }
      if (blockIdx.x == 0)
        for (int k = 0; k < 3; k++) {
          B.grown[3 * (size_t)s + k] = r1[k];
          B.grown[3 * (size_t)(L + s) + k] = r2[k];
        }
    }
    if (blockIdx.x == 0) B.out[(s + 1) & 1] = o;
  }
  __syncthreads();
  return sm.s_go != 0;
}

// The end of step s in a launch of its own (k_grow_step not fused).
constexpr int kSelThreads = 1024;
__global__ __launch_bounds__(kSelThreads) void k_grow_select(Geo g, Dev d, GrowBuf B, int s, int nparts, int nkb) {
  __shared__ GrowSelSmem sm;
  const GrowIn in = *B.in;
  grow_select(g, B, in, grow_ptr(B.rnd, in.K, in.L), s, nparts, nkb, sm);
}

// Launch s of a growth: (fused) step s - 1 finished, then blocks [0, 2 K nparts):
// part 1 of (bead b, trial t, split); then K blocks of parts 2-4, one per trial;
// then K x nkb blocks of k space, (trial, 256 vectors) each.  Step 0 evaluates
// trial 0 only.  A trial bead's query is a cluster query of one
// point (its trials are close together, its counterions anywhere, and each
// trial's energy is wanted): the pairs in range, a fifth of the candidates
// where the cells are coarse, meet in the queue instead of leaving most lanes
// idle in the erfc.
template <int P>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4))) void k_grow_step(Geo g, Dev d, GrowBuf B,
                                                                                              int s, int nparts,
                                                                                              int nkb, int fused) {
  __shared__ union {
    QueryShare<P, Q_MOVED> q;
    GrowSelSmem sel;
    double sh[kBlock / kWave];
  } sm;
  __shared__ double s_prev[6];   // the beads chosen at step s - 1
  const GrowIn in = *B.in;
  const GrowPtr p = grow_ptr(B.rnd, in.K, in.L);
  const int K = in.K, Kt = s == 0 ? 1 : K;
  if (s > 0) {
    if (fused) {
      if (!grow_select(g, B, in, p, s - 1, nparts, nkb, sm.sel)) return;
      if (threadIdx.x < 6) s_prev[threadIdx.x] = sm.sel.s_pos[threadIdx.x];
    } else {
      if (B.out[s & 1].stop >= 0) return;
      if (threadIdx.x < 6) {
        const size_t bead = threadIdx.x < 3 ? s - 1 : in.L + s - 1;
        s_prev[threadIdx.x] = B.grown[3 * bead + threadIdx.x % 3];
      }
    }
    __syncthreads();
  }
  const int ncell = 2 * K * nparts, cur = s & 1;
  if ((int)blockIdx.x < ncell) {
    const int q = blockIdx.x / nparts, sp = blockIdx.x - q * nparts;
    const int t = q % K, b = q / K;
    double2 e = make_double2(0, 0);
    if (t < Kt && (b == 0 || in.charged)) {
      double r1[3], r2[3];
      grow_trial(in, p, s_prev, s, t, r1, r2);
      const double4 pos = b ? make_double4(r2[0], r2[1], r2[2], in.q_i) : make_double4(r1[0], r1[1], r1[2], in.q_c);
      e = real_query_cluster<P, Q_MOVED>(g, d, pos, b ? in.type_i : in.type_c, threadIdx.x % kCluster == 0, 0, in.ex_lo,
                                         in.ex_hi, sp, nparts, sm.q);
    }
    if (threadIdx.x % kWave == 0) B.cells[cur][(size_t)blockIdx.x * kQWaves + threadIdx.x / kWave] = e;
    return;
  }
  if ((int)blockIdx.x < ncell + K) {
    const int t = blockIdx.x - ncell;
    if (t >= Kt) return;
    double r1[3], r2[3];
    grow_trial(in, p, s_prev, s, t, r1, r2);
    const double2 e = grow_explicit(g, d, in, B.grown, s_prev, s, r1, r2, sm.sh);
    if (threadIdx.x == 0) B.expl[cur][t] = e;
    return;
  }
  // k space: block (trial t, chunk kb of 256 vectors)
  const int b = blockIdx.x - ncell - K, t = b / nkb, kb = b - t * nkb;
  if (t >= Kt) return;
  const int k = kb * kBlock + threadIdx.x;
  double e = 0;
  if (k < g.n_kh) {
    const int4 l = d.kl[k];
    const double ck = d.ck[k];
    double2 S = B.Sx[s > 0 ? 1 - cur : 0][k];
    if (s > 0) {
      // the pair chosen at step s - 1 joins S_x
      const double2 e1 = phase(g, l, s_prev);
      S.x += in.q_c * e1.x;
      S.y += in.q_c * e1.y;
      if (in.charged) {
        const double2 e2 = phase(g, l, s_prev + 3);
        S.x += in.q_i * e2.x;
        S.y += in.q_i * e2.y;
      }
      if (t == 0) B.Sx[cur][k] = S;
    }
    double r1[3], r2[3];
    grow_trial(in, p, s_prev, s, t, r1, r2);
    const double2 e1 = phase(g, l, r1);
    e = 2.0 * in.q_c * ck * (e1.x * S.x + e1.y * S.y) + in.q_c * in.q_c * ck;
    if (in.charged) {
      const double2 e2 = phase(g, l, r2);
      e += 2.0 * in.q_i * ck * (e2.x * S.x + e2.y * S.y) + in.q_i * in.q_i * ck;
      e += 2.0 * in.q_c * in.q_i * ck * (e1.x * e2.x + e1.y * e2.y);
    }
  }
  const double r = block_sum<kBlock>(e, sm.sh);
  if (threadIdx.x == 0) B.kpart[cur][(size_t)t * nkb + kb] = r;
}

}  // namespace plum
