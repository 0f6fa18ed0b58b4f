// Induced dipoles of small systems from a dense interaction matrix.
//
// The dipole field of one SOR iteration is linear in the dipoles with
// coefficients that stay fixed through the solve: the real-space tensors
// T(r_ij) (pot_ttm.f90:311-365) and the reciprocal-space sum
// -sum_k 4 pi A_k/V k k^T cos(k.(r_i - r_j)) (ewald.f90:56-119).  Where the
// matrix of all dipole sites of a bead is small, it is formed once per force
// call (k_dense_build) and an iteration is a matrix-vector product: the same
// iterates as the pass-by-pass kernels up to rounding, with the convergence
// test, the SOR update and the iteration counts of pot_ttm.f90:306-392.
//   dense 1: up to 64 dipole sites; one block per bead keeps the matrix in
//            registers and runs the whole loop (k_dense_solve)
//   dense 2: more sites; one launch per iteration, a wave per site
//            (k_dense_step), the matrix read from L2 / HBM
// Both leave the final dipoles in dip and the input of the last step in
// dip_prev, whose structure factor the reciprocal-space forces take
// (ewald.f90:184-193).
#include <algorithm>

#include "ttm_device.h"

namespace pimd {

// k_dense_build: a block takes an 8 x 8 tile of site pairs (i <= j), a lane
// per pair, and its waves deal the kx planes among themselves; their partial
// sums are added in wave order through LDS.  Bound by FP64 issue: per
// (pair, kz-column) three FMAs for each |kz| (the +-kz members of a column
// share cos and sin of kz z, held in registers with their kz and kz^2
// multiples; the column's weights are wave-uniform scalar loads) and about 12
// for the column's phase and its powers of ky.  LM: the largest |kz| index
// held.
constexpr int DB_W = 8;
template <int LM>
__global__ __launch_bounds__(64 * DB_W) void k_dense_build(const Rep *__restrict__ reps,
                                                          BlockMap bm) {
  static_assert(LM % 4 == 3, "weights come in fours");
  __shared__ double part[DB_W][6][64];
  const Blk bk = block_of(bm);
  const Rep &Rp = reps[bk.r];
  const SysConst &c = Rp.c;
  const int M = c.nd * c.N, b = bk.y;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // tile (ti, tj), ti <= tj, of the upper triangle: row ti holds nt - ti tiles
  const int nt = (M + 7) / 8;
  int ti = 0, t = bk.x;
  while (t >= nt - ti) {
    t -= nt - ti;
    ++ti;
  }
  const int tj = ti + t;
  const int i = ti * 8 + lane / 8, j = tj * 8 + lane % 8;
  const bool valid = i < M && j < M && i <= j;
  const int is = valid ? i : 0, js = valid ? j : 0;
  const double2 *__restrict__ tb = Rp.b.tabd + (size_t)b * c.T * M;
  // e^{i 2 pi h (x_i - x_j)/L} from the sites' table row
  auto diff = [&](int row) {
    const double2 a = tb[(size_t)row * M + is], d = tb[(size_t)row * M + js];
    return make_double2(a.x * d.x + a.y * d.y, a.y * d.x - a.x * d.y);
  };
  const int rowy = c.hmax + 1, rowz = c.hmax + c.kmax + 2;
  double cz[LM + 1], c2[LM + 1], s1[LM + 1];
  {
    const double2 z1 = c.lmax >= 1 ? diff(rowz + 1) : make_double2(1.0, 0.0);
    const double kz = TWOPI * c.boxi[2];
    double cc = 1.0, ss = 0.0;
#pragma unroll
    for (int l = 0; l <= LM; ++l) {
      const double k = kz * (double)l;
      cz[l] = cc;
      c2[l] = k * k * cc;
      s1[l] = k * ss;
      const double nc = cc * z1.x - ss * z1.y;
      ss = ss * z1.x + cc * z1.y;
      cc = nc;
    }
  }
  const double2 y1 = c.kmax >= 1 ? diff(rowy + 1) : make_double2(1.0, 0.0);
  const dptr<const int4> dcol = (dptr<const int4>)Rp.b.dcol;
  const dptr<const int> dkx = (dptr<const int>)Rp.b.dkx;
  const dptr<const double> dcoef = (dptr<const double>)Rp.b.dcoef;
  const double ty = TWOPI * c.boxi[1], tx = TWOPI * c.boxi[0];
  double K[6] = {0, 0, 0, 0, 0, 0};  // xx, xy, yy, zz, xz, yz
  for (int h = wv; h <= c.hmax; h += DB_W) {
    const int n0 = dkx[h], n1 = dkx[h + 1];
    if (n0 == n1) continue;
    const int ky0 = dcol[n0].y;
    const double2 X = diff(h);
    double2 Y = diff(rowy + abs(ky0));
    if (ky0 < 0) Y.y = -Y.y;
    double ca = X.x * Y.x - X.y * Y.y, sa = X.y * Y.x + X.x * Y.y;
    double T0 = 0, T1 = 0, T2 = 0, Z = 0, U0 = 0, U1 = 0;
    for (int n = n0; n < n1; ++n) {
      const int4 cl = dcol[n];  // kx, ky, |kz| count (a multiple of 4), first weight
      double S0 = 0, S1 = 0, S2 = 0;
#pragma unroll
      for (int q = 0; q < (LM + 1) / 4; ++q) {
        if (4 * q >= cl.z) break;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const double e = dcoef[cl.w + 4 * q + u];
          S0 = fma(e, cz[4 * q + u], S0);
          S2 = fma(e, c2[4 * q + u], S2);
          S1 = fma(e, s1[4 * q + u], S1);
        }
      }
      const double ky = ty * (double)cl.y;
      const double p0 = ca * S0, p1 = sa * S1;
      T0 += p0;
      T1 = fma(ky, p0, T1);
      T2 = fma(ky * ky, p0, T2);
      Z = fma(ca, S2, Z);
      U0 += p1;
      U1 = fma(ky, p1, U1);
      const double nc = ca * y1.x - sa * y1.y;
      sa = sa * y1.x + ca * y1.y;
      ca = nc;
    }
    const double kx = tx * (double)h;
    K[0] = fma(-kx * kx, T0, K[0]);
    K[1] = fma(-kx, T1, K[1]);
    K[2] -= T2;
    K[3] -= Z;
    K[4] = fma(kx, U0, K[4]);
    K[5] += U1;
  }
#pragma unroll
  for (int q = 0; q < 6; ++q) part[wv][q][lane] = K[q];
  __syncthreads();
  if (wv != 0 || !valid) return;
#pragma unroll
  for (int q = 0; q < 6; ++q) {
    double s = part[0][q][lane];
    for (int w = 1; w < DB_W; ++w) s += part[w][q][lane];
    K[q] = s;
  }
  // the real-space tensor: site pairs of molecules within the cut-off, and
  // those of one molecule
  const int mi = i / c.nd, mj = j / c.nd, ui = c.tdip + i % c.nd, uj = c.tdip + j % c.nd;
  const dptr<const Site> bs = (dptr<const Site>)Rp.b.site + (size_t)b * c.N * 4;
  bool on = mi == mj && i != j;
  if (mi != mj) {
    double x = bs[mi * 4].x - bs[mj * 4].x, y = bs[mi * 4].y - bs[mj * 4].y,
           z = bs[mi * 4].z - bs[mj * 4].z;
    minimg(c, x, y, z);
    on = norm2_exact(x, y, z) < c.rc2;
  }
  if (on) {
    double x = bs[mi * 4 + ui].x - bs[mj * 4 + uj].x, y = bs[mi * 4 + ui].y - bs[mj * 4 + uj].y,
           z = bs[mi * 4 + ui].z - bs[mj * 4 + uj].z;
    minimg(c, x, y, z);
    double ts1, ts2;
    smear2(c, norm2_exact(x, y, z), c.apolDD[ui][uj], ts1, ts2);
    const double t3 = 3.0 * ts2;
    K[0] += t3 * x * x - ts1;
    K[1] += t3 * x * y;
    K[2] += t3 * y * y - ts1;
    K[3] += t3 * z * z - ts1;
    K[4] += t3 * x * z;
    K[5] += t3 * y * z;
  }
  const size_t DS = dense_stride(c);
  dptr<double> m = Rp.b.dmat + (size_t)b * 3 * M * DS;
  const double v[3][3] = {{K[0], K[1], K[4]}, {K[1], K[2], K[5]}, {K[4], K[5], K[3]}};
  // the rows' padding, read with the last column (times a zero)
  if (j == M - 1 && DS != (size_t)3 * M)
    for (int a = 0; a < 3; ++a) m[(size_t)(3 * i + a) * DS + 3 * M] = 0.0;
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      m[(size_t)(3 * i + a) * DS + 3 * j + e] = v[a][e];
      if (i != j) m[(size_t)(3 * j + a) * DS + 3 * i + e] = v[a][e];
    }
}

// The whole SOR loop of one bead in one block: 64 groups of 16 lanes, group g
// holding rows g, g + 64, ... of the matrix in registers (lane u the columns
// u, u + 16, ...), the dipoles in LDS.  One barrier per iteration: dipoles and
// squared changes are double-buffered, and every wave forms the convergence
// test alike.  Bound by the latency of its chain of row sum, update, barrier
// and test, about 1 us per iteration (the four launches of an iteration of the
// pass-by-pass kernels take 40 us for 32 H2O).
template <int RPT, int CPT>
__global__ __launch_bounds__(1024) void k_dense_solve(const Rep *__restrict__ reps, BlockMap bm) {
  constexpr int DMAX = 64 * RPT;
  __shared__ double mu[2][16 * CPT], df2[2][DMAX], eq[DMAX], pol[DMAX];
  const Blk bk = block_of(bm);
  const Rep &Rp = reps[bk.r];
  const SysConst &c = Rp.c;
  const int M = c.nd * c.N, D = 3 * M, b = bk.x;
  const int g = threadIdx.x >> 4, u = threadIdx.x & 15, lane = threadIdx.x & 63;
  const size_t DS = dense_stride(c);
  const dptr<const double> m = (dptr<const double>)Rp.b.dmat + (size_t)b * D * DS;
  double A[RPT][CPT];
#pragma unroll
  for (int r = 0; r < RPT; ++r) {
    const int row = g + 64 * r;
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int col = u + 16 * k;
      A[r][k] = row < D && col < D ? m[(size_t)row * DS + col] : 0.0;
    }
  }
  dptr<double> dip = Rp.b.dip + (size_t)b * D, dip_prev = Rp.b.dip_prev + (size_t)b * D;
  for (int e = threadIdx.x; e < 16 * CPT; e += 1024) {
    mu[0][e] = e < D ? dip[e] : 0.0;
    mu[1][e] = 0.0;
  }
  for (int e = threadIdx.x; e < DMAX; e += 1024) {
    df2[0][e] = df2[1][e] = 0.0;
    const int s = min(e, D - 1) / 3, x = e % 3, type = c.tdip + s % c.nd;
    eq[e] = Rp.b.Efq[(((size_t)b * c.N + s / c.nd) * 4 + type) * 3 + x];
    pol[e] = c.polar[type];
  }
  __syncthreads();
  const double om = c.sor;
  int it = 1, cur = 0;
  bool conv = false;
  for (;; ++it) {
    const double *x = mu[cur];
    double *y = mu[cur ^ 1], *d2 = df2[cur ^ 1];
    double f[RPT];
#pragma unroll
    for (int r = 0; r < RPT; ++r) f[r] = 0.0;
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const double v = x[u + 16 * k];
#pragma unroll
      for (int r = 0; r < RPT; ++r) f[r] = fma(A[r][k], v, f[r]);
    }
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      f[r] = group_sum<16>(f[r]);
      const int row = g + 64 * r;
      if (u == 0 && row < D) {
        const double mr = x[row];
        const double nm = (1.0 - om) * mr + om * pol[row] * (f[r] + eq[row] + c.fac_dd * mr);
        const double d = nm - (it == 1 ? 0.0 : mr);
        y[row] = nm;
        d2[row] = d * d;
      }
    }
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int r = 0; r < RPT; ++r) s += d2[lane + 64 * r];
    s = group_sum<64>(s);
    conv = c.stath * sqrt(s) < c.peps;
    cur ^= 1;
    if (conv || it >= c.maxiter) break;
  }
  for (int e = threadIdx.x; e < D; e += 1024) {
    dip[e] = mu[cur][e];
    dip_prev[e] = mu[cur ^ 1][e];
  }
  if (threadIdx.x == 0) {
    Rp.b.active[b] = 0;
    Rp.b.iters[b] = conv ? it : -it;
  }
}

// One SOR iteration of every live bead, a wave per dipole site: its three
// rows against the bead's dipoles in LDS.  Odd iterations read dip and write
// dip_prev, even ones the other way round; the blocks first run the test of
// the previous iteration.  Reads 24 M bytes per site from L2 or the memory
// cache; 512 H2O, one bead (an 18.9 MB matrix): a few us, near the time of an
// empty launch.
constexpr int DS_W = 4;  // sites per block
__global__ __launch_bounds__(64 * DS_W) void k_dense_step(const Rep *__restrict__ reps, BlockMap bm,
                                                         int it) {
  extern __shared__ double2 lds_mu[];  // [DS / 2]
  __shared__ double red[256];
  __shared__ int act;
  const Blk bk = block_of(bm);
  const Rep &Rp = reps[bk.r];
  const SysConst &c = Rp.c;
  const int M = c.nd * c.N, D = 3 * M, b = bk.y;
  if (it > c.maxiter) return;
  if (it > 1) {
    // the squared changes are double-buffered: blocks of this launch write
    // iteration it's while others still test iteration it - 1's
    if (!sor_test(c, Rp.b.diff2 + (size_t)((it - 1) & 1) * c.P * M, Rp.b.active, Rp.b.iters,
                  Rp.b.nactive, b, it - 1, bk.x == 0, red, act))
      return;
  }
  const dptr<const double> src = (dptr<const double>)(it & 1 ? Rp.b.dip : Rp.b.dip_prev) +
                                 (size_t)b * D;
  dptr<double> dst = (it & 1 ? Rp.b.dip_prev : Rp.b.dip) + (size_t)b * D;
  const int DS = (int)dense_stride(c);
  double *mu = reinterpret_cast<double *>(lds_mu);
  for (int e = threadIdx.x; e < DS; e += 64 * DS_W) mu[e] = e < D ? src[e] : 0.0;
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int s = bk.x * DS_W + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (s >= M) return;
  const dptr<const double2> m =
      (dptr<const double2>)((dptr<const double>)Rp.b.dmat + ((size_t)b * D + 3 * s) * DS);
  const int n = DS / 2;
  double f[3] = {0.0, 0.0, 0.0};
#pragma unroll 4
  for (int e = lane; e < n; e += 64) {
    const double2 x = lds_mu[e];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      const double2 a = m[(size_t)r * n + e];
      f[r] = fma(a.x, x.x, fma(a.y, x.y, f[r]));
    }
  }
#pragma unroll
  for (int r = 0; r < 3; ++r) f[r] = group_sum<64>(f[r]);
  if (lane != 0) return;
  const int type = c.tdip + s % c.nd;
  const size_t ss = ((size_t)b * c.N + s / c.nd) * 4 + type;
  const double om = c.sor, pol = c.polar[type];
  double d2 = 0.0;
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const double mr = mu[3 * s + r];
    const double nm = (1.0 - om) * mr + om * pol * (f[r] + Rp.b.Efq[ss * 3 + r] + c.fac_dd * mr);
    const double d = nm - (it == 1 ? 0.0 : mr);
    d2 += d * d;
    dst[3 * s + r] = nm;
  }
  Rp.b.diff2[((size_t)(it & 1) * c.P + b) * M + s] = d2;
}

// After the last iteration of k_dense_step: its test for the beads still
// live, and the final dipoles into dip (the other buffer holds them after an
// odd count).
__global__ __launch_bounds__(256) void k_dense_done(const Rep *__restrict__ reps, BlockMap bm) {
  __shared__ double red[256];
  __shared__ int act;
  const Blk bk = block_of(bm);
  const Rep &Rp = reps[bk.r];
  const SysConst &c = Rp.c;
  const int M = c.nd * c.N, D = 3 * M, b = bk.x;
  (void)sor_test(c, Rp.b.diff2 + (size_t)(c.maxiter & 1) * c.P * M, Rp.b.active, Rp.b.iters,
                 Rp.b.nactive, b, c.maxiter, true, red, act);
  __threadfence_block();
  __syncthreads();
  const int n = abs(*(volatile int *)(Rp.b.iters + b));
  if (!(n & 1)) return;
  double *d = Rp.b.dip + (size_t)b * D, *p = Rp.b.dip_prev + (size_t)b * D;
  for (int e = threadIdx.x; e < D; e += 256) {
    const double t = d[e];
    d[e] = p[e];
    p[e] = t;
  }
}

void launch_dense_sor(const Group &g, int maxiter, hipStream_t s) {
  // variant: the |kz| bucket of the weights (7, 11, 15)
  launch_over(
      g,
      [](const SysConst &c, const MDConst &) {
        if (!c.dense) return Plan{-1, 0, 0, 0, 0};
        const int nt = (c.nd * c.N + 7) / 8;
        return Plan{c.lmax <= 7 ? 7 : c.lmax <= 11 ? 11 : 15, nt * (nt + 1) / 2, c.P, 1, 0};
      },
      [&](int v, dim3 grid, const BlockMap &m, size_t) {
        if (v == 7) hipLaunchKernelGGL(k_dense_build<7>, grid, dim3(64 * DB_W), 0, s, g.d, m);
        else if (v == 11) hipLaunchKernelGGL(k_dense_build<11>, grid, dim3(64 * DB_W), 0, s, g.d, m);
        else hipLaunchKernelGGL(k_dense_build<15>, grid, dim3(64 * DB_W), 0, s, g.d, m);
      });
  // variant: rows held per 16-lane group
  launch_over(
      g,
      [](const SysConst &c, const MDConst &) {
        if (c.dense != 1) return Plan{-1, 0, 0, 0, 0};
        const int D = 3 * c.nd * c.N;
        return Plan{D <= 64 ? 1 : D <= 128 ? 2 : 3, c.P, 1, 1, 0};
      },
      [&](int v, dim3 grid, const BlockMap &m, size_t) {
        if (v == 1) hipLaunchKernelGGL((k_dense_solve<1, 4>), grid, dim3(1024), 0, s, g.d, m);
        else if (v == 2) hipLaunchKernelGGL((k_dense_solve<2, 8>), grid, dim3(1024), 0, s, g.d, m);
        else hipLaunchKernelGGL((k_dense_solve<3, 12>), grid, dim3(1024), 0, s, g.d, m);
      });
  bool steps = false;
  for (const SysConst &c : g.hc) steps = steps || c.dense == 2;
  if (!steps) return;
  for (int it = 1; it <= maxiter; ++it)
    launch_over(
        g,
        [&](const SysConst &c, const MDConst &) {
          if (c.dense != 2 || it > c.maxiter) return Plan{-1, 0, 0, 0, 0};
          return Plan{0, (c.nd * c.N + DS_W - 1) / DS_W, c.P, 1, sizeof(double) * dense_stride(c)};
        },
        [&](int, dim3 grid, const BlockMap &m, size_t lds) {
          hipLaunchKernelGGL(k_dense_step, grid, dim3(64 * DS_W), lds, s, g.d, m, it);
        });
  launch_over(
      g,
      [](const SysConst &c, const MDConst &) { return Plan{c.dense == 2 ? 0 : -1, c.P, 1, 1, 0}; },
      [&](int, dim3 grid, const BlockMap &m, size_t) {
        hipLaunchKernelGGL(k_dense_done, grid, dim3(256), 0, s, g.d, m);
      });
}

}  // namespace pimd
