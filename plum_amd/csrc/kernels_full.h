// From-scratch kernels: the cell list, and the energy -- real space + LJ over
// all pairs through the cell list, S(k) by direct summation, springs / wall /
// self / dipole, and the reduction into the control block.
#pragma once
#include "kernels_batch.h"

namespace plum {

// ============================================================ cell list
// Built on the device in bead order: counts, then slots by atomics in any
// order, then each cell's beads put in order of their index by rank (the slot
// order a host counting sort gives).  On the host (download, sort, upload of
// every slot array) the list of 40,000 beads took 2.2 ms.
__global__ void k_cell_count(Geo g, Dev d) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= g.n) return;
  const double xw = wrap_coord(d.x[i], g.L[0], g.inv_L[0]);
  const double yw = wrap_coord(d.y[i], g.L[1], g.inv_L[1]);
  const double zw = wrap_coord(d.z[i], g.L[2], g.inv_L[2]);
  const int c = (cell_coord(xw, g.inv_h[0], g.nc[0]) * g.nc[1] + cell_coord(yw, g.inv_h[1], g.nc[1])) * g.nc[2] +
                cell_coord(zw, g.inv_h[2], g.nc[2]);
  d.bcell[i] = c;
  atomicAdd(&d.ccount[c], 1);
}

// Largest cell count into *out (zeroed by the caller).
__global__ __launch_bounds__(kBlock) void k_cell_max(Geo g, Dev d, int* out) {
  int m = 0;
  for (int c = blockIdx.x * kBlock + threadIdx.x; c < g.ncell; c += gridDim.x * kBlock) m = max(m, d.ccount[c]);
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o, kWave));
  if (threadIdx.x % kWave == 0) atomicMax(out, m);
}

// Bead i takes some slot of its cell (counts zeroed by the caller and counted
// again here); ctype holds the bead index until k_cell_order.
__global__ void k_cell_fill(Geo g, Dev d) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= g.n) return;
  const int c = d.bcell[i];
  d.ctype[(size_t)c * g.cap + atomicAdd(&d.ccount[c], 1)] = i;
}

// One block per cell: the bead of rank s among the cell's indices goes to
// slot s; the slots past the count are empty.
__global__ __launch_bounds__(kBlock) void k_cell_order(Geo g, Dev d) {
  __shared__ int s_idx[kBlock];
  const int c = blockIdx.x;
  const int cnt = d.ccount[c];
  const size_t c0 = (size_t)c * g.cap;
  for (int s0 = 0; s0 < cnt; s0 += kBlock) {
    const int s = s0 + threadIdx.x;
    const int j = s < cnt ? d.ctype[c0 + s] : 0;
    int rank = 0;
    for (int t0 = 0; t0 < cnt; t0 += kBlock) {
      __syncthreads();
      if (t0 + threadIdx.x < cnt) s_idx[threadIdx.x] = d.ctype[c0 + t0 + threadIdx.x];
      __syncthreads();
      const int m = min(kBlock, cnt - t0);
      for (int t = 0; t < m; t++) rank += s_idx[t] < j;
    }
    if (s < cnt) d.cbead[c0 + rank] = j;
  }
  for (int s = cnt + threadIdx.x; s < g.cap; s += kBlock) d.cbead[c0 + s] = -1;
  __syncthreads();   // the cell's slots are written, and its index copies read
  const int cx = c / (g.nc[1] * g.nc[2]), cy = (c / g.nc[2]) % g.nc[1], cz = c % g.nc[2];
  for (int s = threadIdx.x; s < cnt; s += kBlock) {
    const int j = d.cbead[c0 + s];
    const double xw = wrap_coord(d.x[j], g.L[0], g.inv_L[0]);
    const double yw = wrap_coord(d.y[j], g.L[1], g.inv_L[1]);
    const double zw = wrap_coord(d.z[j], g.L[2], g.inv_L[2]);
    const double q = d.q[j];
    d.cpos[c0 + s] = make_double4(xw, yw, zw, q);
    d.cpos32[c0 + s] = make_float4((float)(xw - cx * g.h[0]), (float)(yw - cy * g.h[1]), (float)(zw - cz * g.h[2]),
                                   (float)q);
    d.ctype[c0 + s] = d.type[j];
    d.bslot[j] = s;
  }
}

// ============================================================ from scratch
// Real space + LJ over all pairs: the cluster queries of the device loop with
// the beads of a cell, kCluster slots at a time, as the points.  Every ordered
// pair is tested and a pair counted from its lower index, which costs more distance tests than one thread per slot
// that walks the cells around it, and none of its waits: 2.6 ms for 40,000
// beads, and 8.5 ms for 3,200 beads in a box of 1.4 r_c, that way.
// Block (cells, slot group, share of the query's cells); its cells are cell
// blockIdx.x, or where most cells are empty the ones scan_cells listed for it.
struct CellList {
  int *cell, *count;
  int per;      // list entries of a block (0: a block per cell)
  int blocks;   // blocks that share the cells
};

// List of block b: the occupied ones of cells b, b + blocks, .. in that order,
// 256 counts read at a time (one block).
__device__ void scan_cells(const Geo& g, const Dev& d, const CellList& cl, int b) {
  __shared__ int s_wave[kQWaves];
  const int lane = threadIdx.x % kWave, wv = threadIdx.x / kWave;
  int* out = cl.cell + (size_t)b * cl.per;
  int n = 0;
  for (int base = 0; base < cl.per; base += kBlock) {
    const long long c = b + (long long)(base + threadIdx.x) * cl.blocks;
    const bool has = c < g.ncell && d.ccount[c] > 0;
    const unsigned long long m = __ballot(has);
    __syncthreads();   // the last counts are read
    if (lane == 0) s_wave[wv] = __popcll(m);
    __syncthreads();
    int at = n + lanes_below(m);
#pragma unroll
    for (int w = 0; w < kQWaves; w++) {
      if (w < wv) at += s_wave[w];
      n += s_wave[w];
    }
    if (has) out[at] = (int)c;
  }
  if (threadIdx.x == 0) cl.count[b] = n;
}

__global__ __launch_bounds__(kBlock) void k_cell_scan(Geo g, Dev d, CellList cl) { scan_cells(g, d, cl, blockIdx.x); }

// Sum over every bead pair of what real_query_cluster<0, MODE> evaluates, one
// partial per wave.  Of the blocks of 40,000 beads 85% lie past their cell's
// count, so what such a block does counts: with the set-up of the queries before
// the test 232 us, with it after 206.
template <int MODE>
__device__ __forceinline__ void all_pairs(const Geo& g, const Dev& d, const CellList& cl, int nparts,
                                          QueryShare<0, MODE>& sm, double2* out,
                                          const StretchArgs& st = StretchArgs{nullptr, nullptr, 0, 0}) {
  const int lane = threadIdx.x % kWave;
  const size_t b = ((size_t)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
  const int nc = cl.per ? uload(cl.count + blockIdx.x) : (int)blockIdx.y * kCluster < uload(d.ccount + blockIdx.x);
  if (nc == 0) {   // before the set-up of the queries
    if (threadIdx.x < kQWaves) out[b * kQWaves + threadIdx.x] = make_double2(0, 0);
    return;
  }
  double elj = 0, ere = 0;
  for (int i = 0; i < nc; i++) {
    const int cell = cl.per ? uload(cl.cell + (size_t)blockIdx.x * cl.per + i) : (int)blockIdx.x;
    const int cnt = uload(d.ccount + cell);
    for (int s0 = blockIdx.y * kCluster; s0 < cnt; s0 += gridDim.y * kCluster) {
      const int s = s0 + lane % kCluster;
      const size_t si = (size_t)cell * g.cap + min(s, cnt - 1);
      const int own = s < cnt ? d.cbead[si] : -1;
      if (!__ballot(own >= 0)) continue;
      const double2 e = real_query_cluster<0, MODE>(g, d, d.cpos[si], d.ctype[si], own >= 0, own, 0, -1, blockIdx.z,
                                                    nparts, sm, st);
      elj += e.x;
      ere += e.y;
      __syncthreads();   // the next group rewrites the points
    }
  }
  if (lane == 0) out[b * kQWaves + threadIdx.x / kWave] = make_double2(elj, ere);
}

__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4))) void k_full_real(Geo g, Dev d,
                                                                                              CellList cl,
                                                                                              int nparts) {
  __shared__ QueryShare<0, Q_ALL> sm;
  all_pairs<Q_ALL>(g, d, cl, nparts, sm, d.fpart);
}

// S(k) from scratch, bead chunk `blockIdx.y`: direct FP64 sincos per (k,
// bead), for phase tables that do not fit the LDS of k_full_sk_tile.
__global__ __launch_bounds__(kBlock) void k_full_sk_part(Geo g, Dev d, int chunk) {
  const int k = blockIdx.x * kBlock + threadIdx.x;
  if (k >= g.n_kh) return;
  const int4 l = d.kl[k];
  const double kx = (double)(l.x * 2) * kPi / g.L[0];
  const double ky = (double)(l.y * 2) * kPi / g.L[1];
  const double kz = (double)(l.z * 2) * kPi / g.L[2];
  const int j0 = blockIdx.y * chunk, j1 = min(g.n, j0 + chunk);
  double sr = 0, si = 0;
  for (int j = j0; j < j1; j++) {
    const double qj = d.q[j];
    if (qj == 0) continue;
    const double xw = wrap_coord(d.x[j], g.L[0], g.inv_L[0]);
    const double yw = wrap_coord(d.y[j], g.L[1], g.inv_L[1]);
    const double zw = wrap_coord(d.z[j], g.L[2], g.inv_L[2]);
    double s, c;
    sincos(kx * xw + ky * yw + kz * zw, &s, &c);
    sr += qj * c;
    si += qj * s;
  }
  d.sk_part[(size_t)blockIdx.y * g.n_kh + k] = make_double2(sr, si);
}

// The same on the matrix cores: block (four k tiles, bead chunk), a wave per
// tile.  The chunk's phase tables are built in LDS, `sub` beads at a time
// (tables_row, one thread per bead and dimension), and each wave adds its
// tile's products over them (kspace_spec_block's form, one position per bead).
// 40,000 beads and 10,683 vectors: 1.49 ms by sincos, 427 million of them.
constexpr int kSkStage = 3072;   // LDS table entries (48 KB)
__host__ __device__ __forceinline__ int sk_sub(int tab_w) { return min(kBlock / 4, kSkStage / (tab_w | 1)) / 4 * 4; }

__global__ __launch_bounds__(kBlock) void k_full_sk_tile(Geo g, Dev d, int chunk, int ntile) {
  __shared__ double2 s_tab[kSkStage];
  __shared__ double s_q[kBlock / 4];
  const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
  const int tile = blockIdx.x * kQWaves + w;
  const int ws = g.tab_w | 1, nsub = sk_sub(g.tab_w);
  const int col = lane % kKTile, sub = lane / kKTile;
  int4 row = make_int4(0, 0, 0, -1);
  int lz = 0;
  if (tile < ntile) {
    const int2 tl = d.ktile[tile];
    row = d.krow[tl.x + col];
    lz = tl.y + col;
  }
  const int ox = row.x, oy = g.nkx + 1 + abs(row.y), oz = g.nkx + 1 + g.nky + 1 + min(lz, g.nkz);
  const double sy = row.y < 0 ? -1.0 : 1.0;
  f64x4 rr = {0, 0, 0, 0}, ii = rr, ri = rr, ir = rr;
  const int j0 = blockIdx.y * chunk, j1 = min(g.n, j0 + chunk);
  for (int b0 = j0; b0 < j1; b0 += nsub) {
    const int nb = min(nsub, j1 - b0);
    __syncthreads();   // the last sub-chunk's tables are read
    for (int t = threadIdx.x; t < 3 * nsub; t += kBlock) {
      const int m = t / 3, dim = t - 3 * m;
      // (a place past the chunk repeats its last bead, with no charge)
      const int j = b0 + min(m, nb - 1);
      tables_row(g, dim, dim == 0 ? d.x[j] : (dim == 1 ? d.y[j] : d.z[j]), s_tab + (size_t)m * ws);
      if (dim == 0) s_q[m] = m < nb ? d.q[j] : 0.0;
    }
    __syncthreads();
    if (tile < ntile)
#pragma unroll 2
      for (int i0 = 0; i0 < nsub; i0 += 4) {
        const double2* t = s_tab + (size_t)(i0 + sub) * ws;
        const double2 X = t[ox], Y = t[oy], Z = t[oz];
        const double q = s_q[i0 + sub];
        const double yr = q * Y.x, yi = q * sy * Y.y;
        const double ar = X.x * yr - X.y * yi, ai = X.x * yi + X.y * yr;
        rr = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, Z.x, rr, 0, 0, 0);
        ii = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, Z.y, ii, 0, 0, 0);
        ri = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, Z.y, ri, 0, 0, 0);
        ir = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, Z.x, ir, 0, 0, 0);
      }
  }
  if (tile >= ntile) return;
  double2* out = d.sk_part + (size_t)blockIdx.y * g.n_kh;
#pragma unroll
  for (int v = 0; v < 4; v++) {
    const int src = 4 * v + sub;
    const int first = __shfl(row.z, src, kWave), m = __shfl(row.w, src, kWave);
    const int xy = __shfl(row.x | row.y, src, kWave);   // 0: the l_x = l_y = 0 row, which holds l_z > 0 only
    if (lz <= m) {
      const int k0 = xy ? first + m : first - 1;
      if (xy || lz > 0) out[k0 + lz] = make_double2(rr[v] - ii[v], ri[v] + ir[v]);
      if (xy && lz > 0) out[k0 - lz] = make_double2(rr[v] + ii[v], ir[v] - ri[v]);
    }
  }
}

__global__ __launch_bounds__(kBlock) void k_full_sk_reduce(Geo g, Dev d, int nchunk,
                                                           double* epart) {
  __shared__ double sh[kBlock / kWave];
  const int k = blockIdx.x * kBlock + threadIdx.x;
  double e = 0;
  if (k < g.n_kh) {
    double2 s = make_double2(0, 0);
#pragma unroll 8
    for (int c = 0; c < nchunk; c++) {
      const double2 v = d.sk_part[(size_t)c * g.n_kh + k];
      s.x += v.x;
      s.y += v.y;
    }
    d.Sk[k] = s;
    e = d.ck[k] * (s.x * s.x + s.y * s.y);
  }
  const double r = block_sum<kBlock>(e, sh);
  if (threadIdx.x == 0) epart[blockIdx.x] = r;
}

// Spring energy of a molecule at its current coordinates by one wave: the
// per-bond terms and the order of their sum are molecule_spring's (waves of
// 64 bonds, then the waves of a block in order, then the blocks), so the bits
// are the same.  Valid in lane 0.
__device__ double molecule_spring_wave(const Geo& g, const Dev& d, int a, int b) {
  const int lane = threadIdx.x % kWave;
  double acc = 0;
  for (int base = a; base < b - 1; base += kBlock) {
    double blk = 0;
    for (int w0 = base; w0 < min(base + kBlock, b - 1); w0 += kWave) {
      const int i = w0 + lane;
      double e = 0;
      if (i < b - 1) {
        const double dx = d.x[i] - d.x[i + 1], dy = d.y[i] - d.y[i + 1], dz = d.z[i] - d.z[i + 1];
        e = spring_energy(g, dx, dy, dz);
      }
      blk += wave_sum(e);
    }
    acc += blk;
  }
  return acc;
}

// Springs per molecule (a wave each, grid-stride), wall, self and dipole sums
// over the beads, the real-space sum of a bead's own images (self_img q^2) and
// the sum of k_full_real's partials: block partials opart[6 b ..] = springs,
// wall, self, M_z, LJ, real space.  (One block over all molecules
// in turn: 3.7 ms for 20,200 molecules; one block over 68,000 partials: 25 us of
// the 32 of k_full_final.)
constexpr int kSmallSums = 6;
__global__ __launch_bounds__(kBlock) void k_full_small(Geo g, Dev d, int nrealp, double self_img, double* opart) {
  __shared__ double sh[kBlock / kWave];
  const int lane = threadIdx.x % kWave;
  double eb = 0;
  if (g.use_bond)
    for (int m = blockIdx.x * kQWaves + threadIdx.x / kWave; m < g.n_mols; m += gridDim.x * kQWaves) {
      const int a = d.mol_start[m], b = d.mol_start[m + 1];
      const double e = b - a > 1 ? molecule_spring_wave(g, d, a, b) : 0.0;
      if (lane == 0) {
        d.bond_cur[m] = e;
        eb += e;
      }
    }
  double ew = 0, es = 0, mz = 0, el = 0, er = 0;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < g.n; i += gridDim.x * kBlock) {
    const double qi = d.q[i];
    if (g.use_ext) ew += wall_energy(d.z[i], d.wall[d.type[i]], g);
    es += g.self_coef * qi * qi;
    er += self_img * qi * qi;
    mz += qi * d.z[i];
  }
#pragma unroll 4
  for (int b = blockIdx.x * kBlock + threadIdx.x; b < nrealp; b += gridDim.x * kBlock) {
    const double2 e = d.fpart[b];
    el += e.x;
    er += e.y;
  }
  const double v[kSmallSums] = {eb, ew, es, mz, el, er};
#pragma unroll
  for (int k = 0; k < kSmallSums; k++) {
    const double t = block_sum<kBlock>(v[k], sh);
    if (threadIdx.x == 0) opart[kSmallSums * blockIdx.x + k] = t;
  }
}

// The final reduction of all from-scratch partials into the control block.
constexpr int kFinalThreads = 1024;
__global__ __launch_bounds__(kFinalThreads) void k_full_final(Geo g, Dev d, int nkb, int nob, const double* epart_k,
                                                              const double* opart, int set_running) {
  __shared__ double sh[kFinalThreads / kWave];
  Ctl* C = d.ctl;
  double vk = 0, vo[kSmallSums] = {0, 0, 0, 0, 0, 0};
  for (int b = threadIdx.x; b < nkb; b += kFinalThreads) vk += epart_k[b];
  for (int b = threadIdx.x; b < nob; b += kFinalThreads)
#pragma unroll
    for (int k = 0; k < kSmallSums; k++) vo[k] += opart[kSmallSums * b + k];
  const double ebt = block_sum<kFinalThreads>(vo[0], sh);
  const double ewt = block_sum<kFinalThreads>(vo[1], sh);
  const double est = block_sum<kFinalThreads>(vo[2], sh);
  const double mzt = block_sum<kFinalThreads>(vo[3], sh);
  const double lt = block_sum<kFinalThreads>(vo[4], sh);
  const double rt = block_sum<kFinalThreads>(vo[5], sh);
  const double kt = block_sum<kFinalThreads>(vk, sh);
  if (threadIdx.x == 0) {
    double f[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (g.use_pair) f[T_LJ] = lt;
    if (g.use_ewald) {
      f[T_REAL] = rt;
      f[T_KSPACE] = kt;
      f[T_SELF] = est;
      if (g.dipole) f[T_DIPOLE] = dipole_energy(g.dip_coef, mzt);
    }
    if (g.use_bond) f[T_BOND] = ebt;
    if (g.use_ext) f[T_WALL] = ewt;
    for (int k = 0; k < 8; k++) C->full[k] = f[k];
    if (set_running) {
      C->Mz = mzt;
      for (int k = 0; k < 8; k++) C->running[k] = f[k];
      C->cur_dipl = C->trial_dipl = f[T_DIPOLE];
    }
  }
}

}  // namespace plum
