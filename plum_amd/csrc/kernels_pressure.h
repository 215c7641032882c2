// Volume-perturbation pressure: the energy change of one stretch of the box
// along z by kDz (ForceField::CalcPressureVolScalingHSELSlit,
// pressure.cc:187-387).  Beads' z are scaled by 1 + kDz/Lz (with the spring
// potential; grafted "L" beads stay, "R" beads move by kDz) or each molecule
// is shifted by kDz com_z / Lz (without it).  The pair part is summed new minus
// old per pair as the reference does, so the difference keeps its precision;
// the k-space part is summed per k vector from the change of S(k) and of c_k
// (k_vp_dsk).
#pragma once
#include "kernels_full.h"

namespace plum {

constexpr double kDz = 0.00001;   // utilities/constants.h:55

// Stretched z of bead j.  A bead that moves with its molecule sums the
// molecule's centre of mass itself, in the reference's bead order (beads of the
// spring potential do not).
__device__ double vp_z(const Geo& g, const Dev& d, int j) {
  const double Lz = g.Lsim[2], z = d.z[j];
  if (g.use_bond && d.wall[d.type[j]].kind == 0) return z * (1.0 + kDz / Lz);
  const int m = d.mol_of[j], a = d.mol_start[m], b = d.mol_start[m + 1];
  const int k0 = d.wall[d.type[a]].kind;
  double dcz = k0 == 2 ? kDz : 0.0;
  if (k0 == 0) {
    double com = 0;
    for (int i = a; i < b; i++) com += d.z[i];
    com /= (b - a);
    dcz = kDz * (com / Lz);
  }
  return z + dcz;
}

// Everything that goes over the beads, in one launch (a sample of a small
// system is launches): stretched z (zs), the displacement of the image that the
// cell list holds (dw), and block partials part[5 b ..] of the walls (mobile
// beads), the springs (each bond's change), the dipole moments before and after
// and the change of the mobile beads' own images (dself q^2).  Blocks past kVpBeadBlocks list the cells of k_vp_pairs.
constexpr int kVpBeadBlocks = 128, kVpSums = 5;
__global__ __launch_bounds__(kBlock) void k_vp_beads(Geo g, Dev d, CellList cl, double* zs, double* dw, int phantom,
                                                     double dself, double* part) {
  __shared__ double sh[kBlock / kWave];
  if (blockIdx.x >= kVpBeadBlocks) {
    scan_cells(g, d, cl, blockIdx.x - kVpBeadBlocks);
    return;
  }
  Geo gs = g;
  gs.Lsim[2] = g.Lsim[2] + kDz;
  double ew = 0, eb = 0, mo = 0, mn = 0, es = 0;
  for (int j = blockIdx.x * kBlock + threadIdx.x; j < g.n; j += kVpBeadBlocks * kBlock) {
    const int m = d.mol_of[j];
    const double z = d.z[j], zn = vp_z(g, d, j);
    // the displacement of the rounded z', exactly: z and z' are close
    const double disp = zn - z;
    zs[j] = zn;
    dw[j] = disp - rint((z - wrap_coord(z, g.L[2], g.inv_L[2])) * g.inv_L[2]) * kDz;
    if (g.use_ext && m >= phantom) {
      const WallType w = d.wall[d.type[j]];
      ew += wall_energy(zn, w, gs) - wall_energy(z, w, g);
    }
    const double q = d.q[j];
    if (m >= phantom) es += dself * q * q;
    mo += q * z;
    mn += q * zn;
    if (g.use_bond && j + 1 < d.mol_start[m + 1]) {
      const double dx = d.x[j] - d.x[j + 1], dy = d.y[j] - d.y[j + 1], dz = z - d.z[j + 1];
      const double disp1 = vp_z(g, d, j + 1) - d.z[j + 1];
      eb += spring_energy(g, dx, dy, dz + (disp - disp1)) - spring_energy(g, dx, dy, dz);
    }
  }
  const double v[kVpSums] = {ew, eb, mo, mn, es};
#pragma unroll
  for (int k = 0; k < kVpSums; k++) {
    const double t = block_sum<kBlock>(v[k], sh);
    if (threadIdx.x == 0) part[kVpSums * blockIdx.x + k] = t;
  }
}

// Ewald real-space and LJ pairs, stretched minus current: the from-scratch
// cluster queries (k_full_real) with both separations of each pair.  3,200
// beads with r_c = 42 and L = 60: 143 us, and linear in N; over all N (N + 1) /
// 2 bead pairs, the pair index decoded per pair and both image sums explicit,
// 250 us (432 us with all 27 images), quadratic in N.
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4))) void k_vp_pairs(
    Geo g, Dev d, CellList cl, const double* __restrict__ dw, int phantom, int nparts, double2* part_out) {
  __shared__ QueryShare<0, Q_STRETCH> sm;
  all_pairs<Q_STRETCH>(g, d, cl, nparts, sm, part_out, StretchArgs{dw, d.mol_of, kDz, phantom});
}

// The same for up to kVpDirect beads without Ewald, over the bead pairs a < b in
// turn: a query is some 15 us of dependent steps however few its candidates, and
// LJ has one image a pair.  A sample of neutral chains, pairs / queries: 27 / 41
// us at 100 beads, 32 / 57 at 1,020, 45 / 66 at 2,000.
constexpr int kVpDirect = 2048;
__global__ __launch_bounds__(kBlock) void k_vp_pairs_lj(Geo g, Dev d, const double* __restrict__ zs, int phantom,
                                                        double2* part_out) {
  const long long npair = (long long)g.n * g.n;
  const double cw = sqrt(g.lj2_max) + kStretchMargin, lj2 = cw * cw;
  double dlj = 0;
  for (long long p = blockIdx.x * (long long)kBlock + threadIdx.x; p < npair; p += (long long)gridDim.x * kBlock) {
    const int a = (int)(p / g.n), b = (int)(p - (long long)a * g.n);
    if (b <= a || !g.use_pair || d.mol_of[a] < phantom || d.mol_of[b] < phantom) continue;
    double s[3] = {d.x[b] - d.x[a], d.y[b] - d.y[a], d.z[b] - d.z[a]}, m[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
      m[k] = k < g.npbc ? rint(s[k] * g.inv_L[k]) : 0.0;
      s[k] -= m[k] * g.L[k];
    }
    const double r2 = s[0] * s[0] + s[1] * s[1] + s[2] * s[2];
    if (!(r2 < lj2)) continue;
    const double sn = s[2] + ((zs[b] - d.z[b]) - (zs[a] - d.z[a]) - m[2] * kDz);
    const LJPair lp = d.lj[d.type[a] * g.n_types + d.type[b]];
    dlj += lj_energy(sqrt(s[0] * s[0] + s[1] * s[1] + sn * sn), lp) - lj_energy(sqrt(r2), lp);
  }
  dlj = wave_sum(dlj);
  if (threadIdx.x % kWave == 0)
    part_out[(size_t)blockIdx.x * kQWaves + threadIdx.x / kWave] = make_double2(dlj, 0.0);
}

// k space of the stretch, per half-space l vector of the current or the
// stretched k list (their union): S_c(k) of the three bead sets the pair rule
// separates -- mobile beads, the first and the second half of the phantom
// sites -- and the change dS_c of each under the stretch, as sums of
// per-bead phase changes e^{i k'.r'} - e^{i k.r} = 2 i sin(d/2) e^{i (th + th')/2}
// with d = th' - th small (x and y phases are unchanged; z is wrapped in the
// current box and the same image is used in the stretched box), so dE_k
// keeps its precision instead of being a difference of two totals.
// Bead chunk blockIdx.y.
// `ncls` is 3 with surface sites, else 1.  The half phase change d/2 is at most
// l pi kDz / L, so its sine and cosine are the first terms of their series
// (below 1e-3 the next ones are under 1e-25) and a bead costs one sincos, not
// three; chunks are short, as a chunk is a serial chain (512 beads a chunk:
// 372 us for 3,200 beads on seven blocks).
__device__ __forceinline__ void half_phase(double h, double& sn, double& cs) {
  const double h2 = h * h;
  sn = h * (1.0 + h2 * (-1.0 / 6.0 + h2 * (1.0 / 120.0 - h2 * (1.0 / 5040.0))));
  cs = 1.0 + h2 * (-0.5 + h2 * (1.0 / 24.0 - h2 * (1.0 / 720.0)));
}

template <int NCLS>
__global__ __launch_bounds__(kBlock) void k_vp_dsk(Geo g, Dev d, const int4* __restrict__ kl, int nk,
                                                   const double* __restrict__ zs, int phantom, int chunk,
                                                   double2* part) {
  const int k = blockIdx.x * kBlock + threadIdx.x;
  if (k >= nk) return;
  const int4 l = kl[k];
  const double kx = (double)(l.x * 2) * kPi / g.L[0];
  const double ky = (double)(l.y * 2) * kPi / g.L[1];
  const double kz = (double)(l.z * 2) * kPi / g.L[2];
  const double Ls = g.L[2] + kDz;
  const double kzs = (double)(l.z * 2) * kPi / Ls;
  const int j0 = blockIdx.y * chunk, j1 = min(g.n, j0 + chunk);
  double2 S[NCLS], D[NCLS];
#pragma unroll
  for (int c = 0; c < NCLS; c++) S[c] = D[c] = make_double2(0, 0);
  for (int j = j0; j < j1; j++) {
    const double qj = d.q[j];
    if (qj == 0) continue;
    const int cls = NCLS == 1 ? 0 : stretch_class(d.mol_of[j], phantom);
    const double xw = wrap_coord(d.x[j], g.L[0], g.inv_L[0]);
    const double yw = wrap_coord(d.y[j], g.L[1], g.inv_L[1]);
    const double nz = floor(d.z[j] * g.inv_L[2]);
    const double zw = d.z[j] - nz * g.L[2];
    const double zws = zs[j] - nz * Ls;
    double sn, cs, sh, ch;
    sincos(kx * xw + ky * yw + kz * zw, &sn, &cs);
    half_phase(0.5 * (kzs * zws - kz * zw), sh, ch);
    // 2 i sin(d/2) e^{i (th + d/2)}
    const double s2 = 2.0 * qj * sh;
    const double dx = -s2 * (sn * ch + cs * sh), dy = s2 * (cs * ch - sn * sh);
#pragma unroll
    for (int c = 0; c < NCLS; c++)
      if (c == cls) {
        S[c].x += qj * cs;
        S[c].y += qj * sn;
        D[c].x += dx;
        D[c].y += dy;
      }
  }
#pragma unroll
  for (int c = 0; c < NCLS; c++) {
    part[((size_t)blockIdx.y * 2 * NCLS + c) * nk + k] = S[c];
    part[((size_t)blockIdx.y * 2 * NCLS + NCLS + c) * nk + k] = D[c];
  }
}

__device__ __forceinline__ double re_conj(double2 a, double2 b) { return a.x * b.x + a.y * b.y; }

// dE_k per l of the union list: c'(Q(S + dS)) - c Q(S) with
// Q(S) = |S_M|^2 + 2 Re(S_A* S_B) + 2 Re(S_A* S_M) (the included pairs),
// written as dc Q(S) + c' (Q(S + dS) - Q(S)) where l is in both lists
// (dc = c' - c, evaluated on the host without cancellation); block partials.
template <int NCLS>
__global__ __launch_bounds__(kBlock) void k_vp_dsk_energy(const double2* __restrict__ part, int nchunk, int nk,
                                                          const double* __restrict__ c_old,
                                                          const double* __restrict__ c_new,
                                                          const double* __restrict__ dc, double* epart) {
  __shared__ double sh[kBlock / kWave];
  const int k = blockIdx.x * kBlock + threadIdx.x;
  double e = 0;
  if (k < nk) {
    double2 S[3] = {make_double2(0, 0), make_double2(0, 0), make_double2(0, 0)};
    double2 D[3] = {make_double2(0, 0), make_double2(0, 0), make_double2(0, 0)};
#pragma unroll 8
    for (int ch = 0; ch < nchunk; ch++)
#pragma unroll
      for (int c = 0; c < NCLS; c++) {
        const double2 v = part[((size_t)ch * 2 * NCLS + c) * nk + k];
        const double2 w = part[((size_t)ch * 2 * NCLS + NCLS + c) * nk + k];
        S[c].x += v.x;
        S[c].y += v.y;
        D[c].x += w.x;
        D[c].y += w.y;
      }
    const double2 M = S[0], A = S[1], B = S[2], dM = D[0], dA = D[1], dB = D[2];
    const double q0 = re_conj(M, M) + 2.0 * re_conj(A, B) + 2.0 * re_conj(A, M);
    const double dq = 2.0 * re_conj(M, dM) + re_conj(dM, dM) +
                      2.0 * (re_conj(A, dB) + re_conj(dA, B) + re_conj(dA, dB)) +
                      2.0 * (re_conj(A, dM) + re_conj(dA, M) + re_conj(dA, dM));
    const double co = c_old[k], cn = c_new[k];
    if (co != 0 && cn != 0) e = dc[k] * q0 + cn * dq;
    else e = cn * (q0 + dq) - co * q0;
  }
  const double r = block_sum<kBlock>(e, sh);
  if (threadIdx.x == 0) epart[blockIdx.x] = r;
}

// Every partial into out[0..5] = Ewald pairs, LJ pairs, walls, springs,
// dipole, k space.
__global__ __launch_bounds__(kFinalThreads) void k_vp_final(Geo g, const double2* __restrict__ ppart, int npp,
                                                            const double* __restrict__ ekpart, int nkb,
                                                            const double* __restrict__ opart, int nob, double* out) {
  __shared__ double sh[kFinalThreads / kWave];
  double pe = 0, pl = 0, kk = 0, vo[kVpSums] = {0, 0, 0, 0, 0};
#pragma unroll 4
  for (int b = threadIdx.x; b < npp; b += kFinalThreads) {
    pl += ppart[b].x;
    pe += ppart[b].y;
  }
  for (int b = threadIdx.x; b < nkb; b += kFinalThreads) kk += ekpart[b];
  for (int b = threadIdx.x; b < nob; b += kFinalThreads)
#pragma unroll
    for (int k = 0; k < kVpSums; k++) vo[k] += opart[kVpSums * b + k];
  const double t_ew = block_sum<kFinalThreads>(vo[0], sh);
  const double t_eb = block_sum<kFinalThreads>(vo[1], sh);
  const double t_mo = block_sum<kFinalThreads>(vo[2], sh);
  const double t_mn = block_sum<kFinalThreads>(vo[3], sh);
  const double t_pe = block_sum<kFinalThreads>(pe + vo[4], sh);
  const double t_pl = block_sum<kFinalThreads>(pl, sh);
  const double t_kk = block_sum<kFinalThreads>(kk, sh);
  if (threadIdx.x == 0) {
    double dip = 0;
    if (g.use_ewald && g.dipole) {
      const double* L = g.Lsim;
      dip = (g.lB * 2 * kPi) * (t_mn * t_mn / (L[0] * L[1] * (L[2] + kDz)) - t_mo * t_mo / (L[0] * L[1] * L[2]));
    }
    out[0] = g.use_ewald ? t_pe : 0.0;
    out[1] = g.use_pair ? t_pl : 0.0;
    out[2] = g.use_ext ? t_ew : 0.0;
    out[3] = g.use_bond ? t_eb : 0.0;
    out[4] = dip;
    out[5] = g.use_ewald ? t_kk : 0.0;
  }
}

}  // namespace plum
