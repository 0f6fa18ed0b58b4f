// Ewald reciprocal space on matrix cores (ewald.f90:1-226, 403-437): phase
// tables, structure factors and the fields at the sites.
//
// e^{i k.r} = X(kx) Y(ky) Z(kz), and the k-vectors of one (kx, ky) form a
// kz-column symmetric about zero, or its positive half.  Both passes are
// matrix products with the columns along one side and cos / sin of kz z,
// kz = 0..lmax, along another:
//   structure factor  (column) x (cos, sin of each |kz|), summed over sites:
//       C + i S = sum_j w_j X_j Y_j (cos, sin)_j;  S(+-kz) = C +- i S
//   field             (column) x (site), summed over the (cos, sin) of each
//       |kz|: U = sum_kz w_k S_k conj(Z), V the same with kz, from which
//       every component follows by one product with X Y
// so that a k-vector costs a site 4 products (8 for the pair +-kz) in place of
// a phase, its advance and the sums, and the operands of 16 columns serve 16
// sites (16 k) from registers.  Sums are taken in the matrix cores' order;
// against 64-bit sums in the reference's order the difference is rounding.
// v_mfma_f64_16x16x4_f64: lane l holds A[l % 16][l / 16] and B[l / 16][l % 16],
// element i of D is row l / 16 + 4 i of column l % 16; the FP32 form holds row
// 4 (l / 16) + i there.
#include <algorithm>
#include <climits>

#include "ttm_device.h"

namespace pimd {

template <class R> struct Mf;
template <> struct Mf<double> {
  using v2 = double2;
  typedef double v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 mma(double a, double b, v4 d) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, d, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int q, int i) { return q + 4 * i; }
  // the sign of v flipped where sgn has the sign bit
  static __device__ __forceinline__ double flip(double v, int sgn) {
    return __hiloint2double(__double2hiint(v) ^ sgn, __double2loint(v));
  }
  // the value of the lane next to this one (even and odd lanes swapped)
  static __device__ __forceinline__ double swap1(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0xB1, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0xB1, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
  }
};
template <> struct Mf<float> {
  using v2 = float2;
  typedef float v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 mma(float a, float b, v4 d) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, d, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int q, int i) { return 4 * q + i; }
  static __device__ __forceinline__ float flip(float v, int sgn) {
    return __int_as_float(__float_as_int(v) ^ sgn);
  }
  static __device__ __forceinline__ float swap1(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xf, 0xf, true));
  }
};

// Per-site phase tables, the reference's ssincos recurrence (ewald.f90:403-437).
__global__ __launch_bounds__(256) void k_tables(const Rep *__restrict__ reps, BlockMap bm) {
  const Blk bk = block_of(bm);
  const Rep &Rp = reps[bk.r];
  const SysConst &c = Rp.c;
  const Site *__restrict__ site = Rp.b.site;
  double2 *tab = Rp.b.tab;
  const int S = 4 * c.N;
  const int s = bk.x * blockDim.x + threadIdx.x;
  const int b = bk.y;
  if (s >= S) return;
  const Site p = site[(size_t)b * S + s];
  const double xyz[3] = {p.x, p.y, p.z};
  const int hm[3] = {c.hmax, c.kmax, c.lmax};
  int row = 0;
  double2 *tb = tab + (size_t)b * c.T * S + s;
  // the dipole sites' rows again, contiguous in dipole-site order (mol * nd +
  // j), for the passes over dipole sites only; FP32 too in the mixed form
  const int type = s & 3, MD = c.nd * c.N;
  const bool dsite = type >= c.tdip && type < c.tdip + c.nd;
  const size_t dm = (size_t)b * c.T * MD + (size_t)(s >> 2) * c.nd + (type - c.tdip);
  double2 *td = Rp.b.tabd + dm;
  float2 *tf = c.mixed ? Rp.b.tabdf + dm : nullptr;
  auto put = [&](int r, double2 v) {
    tb[(size_t)r * S] = v;
    if (dsite) {
      td[(size_t)r * MD] = v;
      if (tf) tf[(size_t)r * MD] = make_float2((float)v.x, (float)v.y);
    }
  };
  for (int ax = 0; ax < 3; ++ax) {
    const double arg = TWOPI * c.boxi[ax] * xyz[ax];
    const double c1 = cos(arg), s1 = sin(arg);
    double cc = 1.0, ss = 0.0;
    put(row++, make_double2(1.0, 0.0));
    for (int h = 1; h <= hm[ax]; ++h) {
      double nc, ns;
      if (h == 1) {
        nc = c1;
        ns = s1;
      } else {
        nc = cc * c1 - ss * s1;
        ns = cc * s1 + ss * c1;
      }
      cc = nc;
      ss = ns;
      put(row++, make_double2(cc, ss));
    }
  }
}

// Site index of the m-th member of a site set.  SET_CHG: H1, H2, M of every
// molecule; SET_DIP: the dipole sites; SET_ALL: all four.
// SET_CHG_T / SET_ALL_T: the same sites as SET_CHG / SET_ALL, type-major
// (TTM3-F's M sites, then all H2, ...), so that a wave of the final
// reciprocal pass holds one site type and its dipole-site branch is uniform;
// the dipole sites, which take more products, come first.
enum SiteSet { SET_CHG = 0, SET_DIP = 1, SET_ALL = 2, SET_CHG_T = 3, SET_ALL_T = 4 };

__device__ __forceinline__ int set_size(const SysConst &c, int set) {
  return set == SET_CHG || set == SET_CHG_T ? 3 * c.N : set == SET_DIP ? c.nd * c.N : 4 * c.N;
}
__device__ __forceinline__ int set_site(const SysConst &c, int set, int m) {
  if (set == SET_CHG) return (m / 3) * 4 + 1 + m % 3;
  if (set == SET_DIP) return (m / c.nd) * 4 + c.tdip + m % c.nd;
  if (set == SET_CHG_T) return (m % c.N) * 4 + 3 - m / c.N;
  if (set == SET_ALL_T) return (m % c.N) * 4 + m / c.N;
  return m;
}

// Phase-table rows of the m-th member of a site set: the dipole sites from
// their contiguous table (FP32 in the mixed form's SOR iterations), the
// other sets from the all-site table.
template <class R, int SET>
__device__ __forceinline__ const typename Mf<R>::v2 *set_rows(const Rep &Rp, int b, int &stride) {
  const SysConst &c = Rp.c;
  if constexpr (SET == SET_DIP) {
    stride = c.nd * c.N;
    const size_t off = (size_t)b * c.T * stride;
    if constexpr (sizeof(R) == 4) return Rp.b.tabdf + off;
    else return Rp.b.tabd + off;
  } else {
    static_assert(sizeof(R) == 8, "the all-site table is FP64");
    stride = 4 * c.N;
    return Rp.b.tab + (size_t)b * c.T * stride;
  }
}
template <int SET>
__device__ __forceinline__ int row_index(const SysConst &c, int m) {
  return SET == SET_DIP ? m : set_site(c, SET, m);
}

// Steps of four (cos, sin) entries along kz = 0..l.
__host__ __device__ inline int kz_steps(int l) { return (l + 2) / 2; }
__host__ __device__ inline int col_tiles(const SysConst &c) { return (c.ncol + 15) / 16; }

// Field operands: [P][col_tiles][kz_steps(lmax)][components][64 lanes].
// First the 4 components U, V (re, im) of one structure factor, FP64; then the
// 6 components U, V, W of the total one (W with kz^2).  The mixed form's SOR
// iterations keep their FP32 operands in the second part, which is not
// written before they end.
constexpr int WK_A = 4, WK_B = 6;
__host__ __device__ inline size_t wk_elems(const SysConst &c, int comps) {
  return (size_t)c.P * col_tiles(c) * kz_steps(c.lmax) * comps * 64;
}

// Chunk partial sums of one structure factor: a wave takes 16 columns and the
// (cos, sin) of 8 consecutive |kz| (its task) over a block's chunk of sites,
// whose phase tables and weights are staged in LDS once for all tasks.  Lane
// l forms the weighted X Y of column l % 16 and site l / 16 of the step as
// the A operands of NC products, and reads one cos or sin as their common B.
//   SF_Q: (sum q cos, sum q sin)                      (ewald.f90:41-44)
//   SF_D: (-sum (k.mu) sin, sum (k.mu) cos)           (ewald.f90:99-110)
//   SF_V: (sum mu cos, sum mu sin) per component      (ewald.f90:208-213)
// stale (SF_D): of every bead's dip_prev, the input of its last SOR step, in
// place of its current dipoles (dense systems).
// Bound by the FP64 matrix rate (64 cycles per product on a SIMD) and the
// launch; 512 H2O x 32 beads, one kz-segment of 4 per lane / now: SF_D 16.8 /
// 13.0 us (4.3 us of it matrix time), SF_Q 43 / 22.7 (6.4), SF_V 30 / 18.7.
template <int MODE, class R>
__global__ __launch_bounds__(1024) void k_sfac(const Rep *__restrict__ reps, BlockMap bm, int stale,
                                               int groups) {
  using R2 = typename Mf<R>::v2;
  using V4 = typename Mf<R>::v4;
  constexpr int SET = MODE == SF_Q ? SET_CHG : SET_DIP;
  constexpr int NW = MODE == SF_Q ? 1 : 3;                      // weights per site
  constexpr int NC = MODE == SF_Q ? 2 : MODE == SF_D ? 4 : 6;   // products
  constexpr int NV = MODE == SF_V ? 6 : 2;                      // values per k
  extern __shared__ double2 lds_raw[];
  R2 *tabs = reinterpret_cast<R2 *>(lds_raw);  // [T][scp] tables, then [sc][NW] weights
  const Blk bk = block_of(bm);
  const Rep &Rp = reps[bk.r];
  const SysConst &c = Rp.c;
  const int b = bk.y;
  if (MODE == SF_D && !stale && !Rp.b.active[b]) return;
  const Site *__restrict__ site = Rp.b.site;
  const double *__restrict__ dip = stale ? Rp.b.dip_prev : Rp.b.dip;
  const int4 *__restrict__ cols = Rp.b.cols;
  const int *__restrict__ colk = Rp.b.colk;
  int nch, sc, scp;
  sfac_chunking(c, MODE, nch, sc, scp);
  R *lw = reinterpret_cast<R *>(tabs + (size_t)c.T * scp);
  const int S = 4 * c.N, M = set_size(c, SET);
  const int chunk = bk.x, m0 = chunk * sc, nt = min(sc, M - m0);
  int RS;
  const R2 *__restrict__ tb = set_rows<R, SET>(Rp, b, RS);
  // sites past the chunk's end: the last one's phases, with zero weights
  for (int e = threadIdx.x; e < c.T * sc; e += blockDim.x) {
    const int row = e / sc, l = e % sc;
    tabs[row * scp + l] = tb[(size_t)row * RS + row_index<SET>(c, m0 + min(l, nt - 1))];
  }
  for (int l = threadIdx.x; l < sc; l += blockDim.x) {
    if (MODE == SF_Q) {
      lw[l] = l < nt ? site[(size_t)b * S + set_site(c, SET, m0 + l)].q : 0.0;
    } else {
      const double *mu = dip + ((size_t)b * c.N * c.nd + m0 + l) * 3;
      for (int k = 0; k < 3; ++k) lw[l * 3 + k] = l < nt ? (R)mu[k] : (R)0.0;
    }
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, n = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
  const double tpz = TWOPI * c.boxi[2];
  for (int task = bk.z * nw + wave; task < c.sf_ntask; task += groups * nw) {
    const int tk = Rp.b.sftask[task], ct = tk & 0xffff, l0 = 8 * (tk >> 16);
    const ColRec cr = Rp.b.colrec[ct * 16 + n];
    const R2 *px = tabs + cr.rx * scp + q;
    const R2 *py = tabs + cr.ry * scp + q;
    const R *pz = reinterpret_cast<const R *>(
                      tabs + (c.hmax + c.kmax + 2 + min(l0 + (n >> 1), c.lmax)) * scp + q) + (n & 1);
    const R kx = (R)cr.kx, ky = (R)cr.ky;
    V4 acc[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) acc[i] = V4{0, 0, 0, 0};
    auto step = [&](int e) {
      const R2 x = px[e];
      R2 y = py[e];
      const R t = pz[2 * e];
      y.y = Mf<R>::flip(y.y, cr.sgn);
      const R xr = x.x * y.x - x.y * y.y, xi = x.y * y.x + x.x * y.y;
      const R *w = lw + (e + q) * NW;
      R a[NC];
      if constexpr (MODE == SF_Q) {
        a[0] = w[0] * xr;
        a[1] = w[0] * xi;
      } else if constexpr (MODE == SF_D) {
        const R wxy = kx * w[0] + ky * w[1];
        a[0] = wxy * xr;
        a[1] = wxy * xi;
        a[2] = w[2] * xr;
        a[3] = w[2] * xi;
      } else {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          a[2 * k] = w[k] * xr;
          a[2 * k + 1] = w[k] * xi;
        }
      }
#pragma unroll
      for (int i = 0; i < NC; ++i) acc[i] = Mf<R>::mma(a[i], t, acc[i]);
    };
    for (int e = 0; e < sc; e += 8) {
      step(e);
      step(e + 4);
    }
    // even lanes hold the cos sums of |kz| and write +kz, odd lanes the sin
    // sums and write -kz
    const bool odd = n & 1;
    const int l = l0 + (n >> 1), kz = odd ? -l : l;
    const R kzv = (R)(tpz * (double)kz);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      R re[NC / 2], im[NC / 2];
#pragma unroll
      for (int v = 0; v < NC / 2; ++v) {
        const R o_r = acc[2 * v][i], o_i = acc[2 * v + 1][i];
        const R p_r = Mf<R>::swap1(o_r), p_i = Mf<R>::swap1(o_i);
        re[v] = odd ? p_r + o_i : o_r - p_i;
        im[v] = odd ? p_i - o_r : o_i + p_r;
      }
      const int col = ct * 16 + Mf<R>::row(q, i);
      if (col >= c.ncol) continue;
      const int4 cw = cols[col];
      if ((odd && l == 0) || kz < cw.z || kz >= cw.z + cw.w) continue;
      double *o = Rp.b.part + (((size_t)b * nch + chunk) * c.nk + colk[col] + kz - cw.z) * NV;
      if constexpr (MODE == SF_Q) {
        o[0] = re[0];
        o[1] = im[0];
      } else if constexpr (MODE == SF_D) {
        o[0] = -(double)(im[0] + kzv * im[1]);
        o[1] = (double)(re[0] + kzv * re[1]);
      } else {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          o[k] = re[k];
          o[3 + k] = im[k];
        }
      }
    }
  }
}

// The structure factor from its chunk sums, added in order, and the operands
// the fields take from it (R: their type, FP32 in the mixed form's SOR
// iterations).  A thread takes the +-kz pair of one column.  SF_V stays where
// its first chunk's sums were, and its operands are those of the total structure
// factor Sq + Sm.
template <int MODE, class R>
__global__ __launch_bounds__(256) void k_sfac_reduce(const Rep *__restrict__ reps, BlockMap bm,
                                                     int stale) {
  constexpr int NV = MODE == SF_V ? 6 : 2;
  constexpr int NC = MODE == SF_V ? WK_B : WK_A;
  const Blk bk = block_of(bm);
  const Rep &Rp = reps[bk.r];
  const SysConst &c = Rp.c;
  const int b = bk.y;
  if (MODE == SF_D && !stale && !Rp.b.active[b]) return;
  const int nct = col_tiles(c), nks = kz_steps(c.lmax);
  const int e = bk.x * 256 + threadIdx.x;
  if (e >= nct * nks * 32) return;
  const int r = e & 15, hl = (e >> 4) & 1, st = e >> 5;  // st = tile * nks + step
  const int l = 2 * (st % nks) + hl, col = (st / nks) * 16 + r;
  int nch, sc, scp;
  sfac_chunking(c, MODE, nch, sc, scp);
  const double4 *__restrict__ kv = Rp.b.kv;
  double w[2][2] = {{0, 0}, {0, 0}};  // 4 pi A_k / V times S of +kz, -kz (re, im)
  if (col < c.ncol) {
    const int4 cl = Rp.b.cols[col];
    const int k0 = Rp.b.colk[col];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int kz = s ? -l : l;
      if ((s && l == 0) || kz < cl.z || kz >= cl.z + cl.w) continue;
      const int k = k0 + kz - cl.z;
      double v[NV];
      for (int i = 0; i < NV; ++i) v[i] = 0.0;
      double *pp = Rp.b.part + ((size_t)b * nch * c.nk + k) * NV;
#pragma unroll 4
      for (int h = 0; h < nch; ++h)
        for (int i = 0; i < NV; ++i) v[i] += pp[(size_t)h * c.nk * NV + i];
      const size_t o = ((size_t)b * c.nk + k) * 2;
      double *out = MODE == SF_Q ? Rp.b.Sq + o : MODE == SF_D ? Rp.b.Sm + o : pp;
      for (int i = 0; i < NV; ++i) out[i] = v[i];
      const double re = MODE == SF_V ? Rp.b.Sq[o] + Rp.b.Sm[o] : v[0];
      const double im = MODE == SF_V ? Rp.b.Sq[o + 1] + Rp.b.Sm[o + 1] : v[1];
      w[s][0] = kv[k].w * re;
      w[s][1] = kv[k].w * im;
    }
  }
  const double kz = TWOPI * c.boxi[2] * (double)l;
  const double pr = w[0][0] + w[1][0], pi = w[0][1] + w[1][1];
  const double mr = w[0][0] - w[1][0], mi = w[0][1] - w[1][1];
  R *o;
  if constexpr (MODE == SF_V) o = Rp.b.wk + wk_elems(c, WK_A);
  else if constexpr (sizeof(R) == 4) o = reinterpret_cast<float *>((double *)(Rp.b.wk + wk_elems(c, WK_A)));
  else o = Rp.b.wk;
  o += ((size_t)b * nct * nks + st) * NC * 64 + 32 * hl + r;
  // rows (kz, cos) and (kz, sin), 16 lanes apart
  const double cs[6] = {pr, pi, kz * mr, kz * mi, kz * kz * pr, kz * kz * pi};
  const double sn[6] = {mi, -mr, kz * pi, -kz * pr, kz * kz * mi, -kz * kz * mr};
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    o[i * 64] = (R)cs[i];
    o[i * 64 + 16] = (R)sn[i];
  }
}

static size_t sfac_lds(const SysConst &c, int mode, int sc, int scp, bool f32) {
  const size_t r = f32 ? sizeof(float) : sizeof(double);
  return 2 * r * c.T * scp + r * sc * (mode == SF_Q ? 1 : 3);
}

// Reciprocal-space fields at each site.  A block holds SG groups of NT tiles
// of 16 sites of one bead and CG column groups, one wave for each pair;
// a wave takes every CG-th tile of 16 columns (the waves of other site groups
// read the same operands at about the same time, from the cache next to the
// CU): U, V (and, for FD_QD at dipole sites, U, V, W of the total structure
// factor) of 16 columns x 16 NT sites are one matrix product each over the (cos,
// sin) of the tile's |kz|, with the operands from k_sfac_reduce read in lane
// order and the sites' phases from LDS.  Lane l then holds 4 columns of site
// l % 16 of each tile and adds their fields.
// The waves' and lane groups' parts are added in a fixed order.
//   FD_Q : Efq and phi from the charge structure factor (ewald.f90:45-49)
//   FD_D : Efd from the dipole structure factor (ewald.f90:114-117), then the
//          SOR update of the induced dipole (pot_ttm.f90:371-385)
//   FD_QD: phi and dR from the stale dipole and the total structure factors
//          (ewald.f90:184-193)
// iter: the SOR iteration (FD_D), or -1 for the mixed form's FP64
// refinement, the step after the replica's last (maxiter + 1).
// Bound by the FP64 matrix rate and, in the SOR iterations, the launch:
// 512 H2O x 32 beads, one site per lane walking the columns / now: FD_D 12.4 /
// 10.5 us (3.3 us of it matrix time), FD_Q 39 / 25 (9.8), FD_QD 64 / 47 (15).
constexpr int FD_SB = 32;     // sites per group of two tiles
constexpr int FD_WAVES = 8;   // waves per block at most
// Tiles per site group, site groups per block and column groups of one field
// launch over M sites.  Small systems, of up to 128 groups of two tiles, take
// one tile to a group, half the work per wave: one tile / two, us per call of
// 32 H2O (Rc 4.9 A), 1 bead 250 / 258, 8 beads (24 groups of charges) 275 / 285,
// 32 (96) 355 / 364, 48 (144) 374 / 373, 64 (192) 407 / 408.
// Column groups until the device has two waves per SIMD; blocks of 4 waves,
// of which a CU holds three, and of 8 only where every CU gets at most one
// block.  Of 4, 2 and 1 site groups the most that leave few CUs idle at the
// end.  (Waves per block 4 / 8: FD_D of TTM2.1-F 128 x 32 10.8 / 12.9 us, a
// whole call of 32 H2O x 32 beads 376 / 369 us.)
__host__ inline void field_groups(const SysConst &c, int M, int &nt, int &sg, int &cg) {
  long ng = (long)c.shapeP * ((M + FD_SB - 1) / FD_SB);
  nt = ng <= 128 ? 1 : 2;
  const int sb = 16 * nt;
  ng = (long)c.shapeP * ((M + sb - 1) / sb);
  const int most = ng <= 256 ? FD_WAVES : 4;
  cg = 1;
  while (cg < most && cg < col_tiles(c) && ng * cg < 2048) cg *= 2;
  if (c.fd_cg) cg = c.fd_cg < FD_WAVES ? c.fd_cg : FD_WAVES;
  auto idle = [&](int s) {
    const long nb = (long)c.shapeP * ((M + s * sb - 1) / (s * sb));
    return 1.0 - (double)nb / ((nb + 255) / 256 * 256);
  };
  for (sg = cg < 4 ? 4 / cg : 1; sg > 1; sg /= 2)
    if (idle(sg) <= 0.1 || idle(sg) <= idle(1)) break;
}
template <int MODE, int MODEL, class R, int NT>
__global__ __launch_bounds__(64 * FD_WAVES, MODE == FD_QD ? 2 : 3) void k_field(const Rep *__restrict__ reps, BlockMap bm,
                                                         int iter, int SG) {
  using R2 = typename Mf<R>::v2;
  using V4 = typename Mf<R>::v4;
  constexpr int SET = MODE == FD_D    ? SET_DIP
                      : MODE == FD_QD ? (MODEL == 2 ? SET_ALL_T : SET_CHG_T)
                                      : (MODEL == 2 ? SET_ALL : SET_CHG);
  extern __shared__ double2 lds_raw[];  // [T + 1][TS] phases, then the column groups' [CG][4][SB] parts
  R2 *tabs = reinterpret_cast<R2 *>(lds_raw);
  const Blk bk = block_of(bm);
  const Rep &Rp = reps[bk.r];
  const SysConst &c = Rp.c;
  const Site *__restrict__ site = Rp.b.site;
  const ColRec *__restrict__ rec = Rp.b.colrec;
  if (iter < 0) iter = c.maxiter + 1;
  const int b = bk.y;
  if (MODE == FD_D && !Rp.b.active[b]) return;
  const int lane = threadIdx.x & 63, n = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = wave / SG, CG = (blockDim.x >> 6) / SG;
  constexpr int FS = 16 * NT;  // sites per group
  const int SB = SG * FS, TS = phase_row(SB);
  const int M = set_size(c, SET), S = 4 * c.N, mbase = bk.x * SB, sbase = (wave % SG) * FS;
  int RS;
  const R2 *__restrict__ tb = set_rows<R, SET>(Rp, b, RS);
  // one row more than the tables': the last step may reach kz = lmax + 1,
  // where the operands are zero
  for (int e = threadIdx.x; e < (c.T + 1) * SB; e += blockDim.x) {
    const int row = e / SB, l = e % SB;
    tabs[row * TS + l] = tb[(size_t)min(row, c.T - 1) * RS + row_index<SET>(c, min(mbase + l, M - 1))];
  }
  // charge and dipole of this lane's site of each tile
  double qs[NT], mu[NT][3];
  for (int t = 0; t < NT; ++t) qs[t] = mu[t][0] = mu[t][1] = mu[t][2] = 0.0;
  bool any_q = true, any_d = false;
  if (MODE == FD_QD) {
    bool hq = false, hd = false;
    for (int t = 0; t < NT; ++t) {
      const int s = set_site(c, SET, min(mbase + sbase + 16 * t + n, M - 1)), type = s & 3;
      if (type != 0) {
        qs[t] = site[(size_t)b * S + s].q;
        hq = true;
      }
      if (type >= c.tdip && type < c.tdip + c.nd) {
        hd = true;
        const size_t d = ((size_t)b * c.N + (s >> 2)) * c.nd + (type - c.tdip);
        for (int k = 0; k < 3; ++k) mu[t][k] = Rp.b.dip[d * 3 + k];
      }
    }
    any_q = __any(hq);
    any_d = __any(hd);
  }
  __syncthreads();
  const int nct = col_tiles(c), nks = kz_steps(c.lmax);
  const R *wa, *wb = nullptr;
  if constexpr (sizeof(R) == 4) wa = reinterpret_cast<const float *>((const double *)(Rp.b.wk + wk_elems(c, WK_A)));
  else wa = Rp.b.wk;
  if constexpr (MODE == FD_QD) wb = Rp.b.wk + wk_elems(c, WK_A);
  // this lane's cos or sin row of the first step: kz = q / 2, then two on
  const R *pb = reinterpret_cast<const R *>(
                    tabs + (c.hmax + c.kmax + 2 + (q >> 1)) * TS + sbase + n) + (q & 1);
  double e[NT][4];  // field and potential at this lane's sites
  for (int t = 0; t < NT; ++t) e[t][0] = e[t][1] = e[t][2] = e[t][3] = 0.0;
  for (int ct = g; ct < nct; ct += CG) {
    // the columns are sorted by their reach along kz
    const int ks = kz_steps(rec[ct * 16].reach);
    double kx[4], ky[4];
    const R2 *px[4], *py[4];
    int sg[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const ColRec cr = rec[ct * 16 + Mf<R>::row(q, i)];
      kx[i] = cr.kx;
      ky[i] = cr.ky;
      px[i] = tabs + (__umul24(cr.rx, TS) + sbase + n);
      py[i] = tabs + (__umul24(cr.ry, TS) + sbase + n);
      sg[i] = cr.sgn;
    }
    const size_t wo = ((size_t)b * nct + ct) * nks;
    // the products of NC components with both site tiles, then done(column
    // element, site tile, a = Re X Y, d = Im X Y, values)
    auto gemm = [&](auto nc_tag, const R *w, auto &&done) {
      constexpr int NC = decltype(nc_tag)::value;
      const R *wp = w + wo * NC * 64 + lane;
      V4 D[NC][NT];
      R a[NC], an[NC];
      auto load = [&](R *to, int s) {
#pragma unroll
        for (int v = 0; v < NC; ++v) to[v] = wp[(s * NC + v) * 64];
      };
      auto step = [&](int s, auto first_tag) {
        constexpr bool FIRST = decltype(first_tag)::value;
        const R *p = pb + (size_t)s * (4 * TS);
        const R b0 = p[0], b1 = NT == 2 ? p[32] : (R)0.0;
#pragma unroll
        for (int v = 0; v < NC; ++v) {
          D[v][0] = Mf<R>::mma(a[v], b0, FIRST ? V4{0, 0, 0, 0} : D[v][0]);
          if constexpr (NT == 2) D[v][1] = Mf<R>::mma(a[v], b1, FIRST ? V4{0, 0, 0, 0} : D[v][NT - 1]);
        }
      };
      // the next step's operands in flight
      load(a, 0);
      if (ks > 1) load(an, 1);
      step(0, std::true_type{});
      for (int s = 1; s < ks; ++s) {
#pragma unroll
        for (int v = 0; v < NC; ++v) a[v] = an[v];
        if (s + 1 < ks) load(an, s + 1);
        step(s, std::false_type{});
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const R2 x = px[i][16 * t];
          R2 y = py[i][16 * t];
          y.y = Mf<R>::flip(y.y, sg[i]);
          R v[NC];
#pragma unroll
          for (int k = 0; k < NC; ++k) v[k] = D[k][t][i];
          done(i, t, x.x * y.x - x.y * y.y, x.y * y.x + x.x * y.y, v);
        }
    };
    if (any_q)
      gemm(std::integral_constant<int, 4>{}, wa, [&](int i, int t, R a, R d, const R *v) {
        // at = w (cos Im S - sin Re S) summed over the column, az with kz
        R at = a * v[1] - d * v[0], az = a * v[3] - d * v[2];
        if (MODE != FD_D) e[t][3] += a * v[0] + d * v[1];
        if (MODE == FD_QD) {
          at *= -qs[t];
          az *= -qs[t];
        }
        e[t][0] -= kx[i] * (double)at;
        e[t][1] -= ky[i] * (double)at;
        e[t][2] -= (double)az;
      });
    if constexpr (MODE == FD_QD)
      if (any_d)
        gemm(std::integral_constant<int, 6>{}, wb, [&](int i, int t, R a, R d, const R *v) {
          const double dxy = kx[i] * mu[t][0] + ky[i] * mu[t][1];
          const double u = a * v[0] + d * v[1], z = a * v[2] + d * v[3], zz = a * v[4] + d * v[5];
          const double at = dxy * u + mu[t][2] * z, az = dxy * z + mu[t][2] * zz;
          e[t][0] -= kx[i] * at;
          e[t][1] -= ky[i] * at;
          e[t][2] -= az;
        });
  }
  __syncthreads();
  double *red = reinterpret_cast<double *>(lds_raw);  // [CG][4][SB]
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int k = 0; k < (MODE == FD_D ? 3 : 4); ++k) {
      double v = e[t][k];
      v += __shfl_xor(v, 16);
      v += __shfl_xor(v, 32);
      if (q == 0) red[(g * 4 + k) * SB + sbase + 16 * t + n] = v;
    }
  __syncthreads();
  const int m = mbase + threadIdx.x;
  if (threadIdx.x >= SB || m >= M) return;
  double f[4] = {0, 0, 0, 0};
  for (int w = 0; w < CG; ++w)
#pragma unroll
    for (int k = 0; k < (MODE == FD_D ? 3 : 4); ++k) f[k] += red[(w * 4 + k) * SB + threadIdx.x];
  const int s = set_site(c, SET, m), type = s & 3;
  const size_t ss = (size_t)b * S + s;
  if (MODE != FD_D) {
    // into their own buffers (kE, kphi): the consumer adds them to the
    // real-space sums, which the pair kernels may be forming meanwhile
    for (int k = 0; k < 3; ++k) Rp.b.kE[ss * 3 + k] = f[k];
    Rp.b.kphi[ss] = type != 0 ? f[3] : 0.0;
  } else {
    const size_t d = (size_t)b * c.N * c.nd + m;
    double *__restrict__ dip = Rp.b.dip;
    const double om = c.sor, pol = c.polar[type];
    double d2 = 0.0;
    for (int k = 0; k < 3; ++k) {
      const double mk = dip[d * 3 + k];
      const double etot = (Rp.b.Efd[d * 3 + k] + f[k]) + Rp.b.Efq[ss * 3 + k] + c.fac_dd * mk;
      const double nm = (1.0 - om) * mk + om * pol * etot;
      const double df = nm - (iter == 1 ? 0.0 : mk);
      d2 += df * df;
      dip[d * 3 + k] = nm;
      if (c.mixed && iter <= c.maxiter) Rp.b.dip_prev[d * 3 + k] = mk;
    }
    Rp.b.diff2[d] = d2;
  }
}

static bool has_dipoles(const SysConst &c) { return c.model == PIMD_TTM21F || c.model == PIMD_TTM3F; }
static int idiv(long a, long b) { return (int)((a + b - 1) / b); }

// sel (SF_D): SFAC_ITER, the SOR iterations (not the dense systems; the mixed
// form's in FP32), SFAC_REFINE the mixed form's FP64 refinement step,
// SFAC_STALE the dense systems' last input.  part: 1 the chunk sums, 2 their
// reduction, 3 both.  Variant: bit 0 FP32, above it the waves per block: one
// per task up to 16, beyond as few rounds of tasks as 16 waves need; an even
// number, so that more replicas of a batch share launches.  Passes of up to 128
// chunks give each round a block of its own: so / one block for all rounds, us
// per call of 32 H2O (Rc 4.9 A), 1 bead (4 to 8 chunks) 245 / 250, 8 beads (32
// and 64) 268 / 275, 32 (128 dipole chunks) 350 / 355, 48 (192) 378 / 374.
template <int MODE>
static void launch_sfac_mode(const Group &g, int sel, int part, hipStream_t s) {
  const int stale = MODE == SF_D && sel == SFAC_STALE ? 1 : 0;
  auto plan = [&](const SysConst &c) {
    if (MODE != SF_Q && !has_dipoles(c)) return Plan{-1, 0, 0, 0, 0};
    if (sel == SFAC_REFINE && !c.mixed) return Plan{-1, 0, 0, 0, 0};
    if (MODE == SF_D && (c.dense != 0) != (sel == SFAC_STALE)) return Plan{-1, 0, 0, 0, 0};
    const bool f32 = MODE == SF_D && c.mixed && sel == SFAC_ITER;
    int nch, sc, scp;
    sfac_chunking(c, MODE, nch, sc, scp);
    const int rounds = std::max(1, idiv(c.sf_ntask, 16));
    const int waves = std::max(2, (idiv(c.sf_ntask, rounds) + 1) / 2 * 2);
    const int groups = (long)nch * c.shapeP <= 128 ? rounds : 1;
    return Plan{(f32 ? 1 : 0) | (waves << 1) | (groups << 6), nch, c.P, groups,
                sfac_lds(c, MODE, sc, scp, f32)};
  };
  if (part & 1)
    launch_over(
        g, [&](const SysConst &c, const MDConst &) { return plan(c); },
        [&](int v, dim3 grid, const BlockMap &m, size_t lds) {
          const dim3 block(64 * ((v >> 1) & 31));
          const int groups = v >> 6;
          if constexpr (MODE == SF_D)
            if (v & 1) {
              hipLaunchKernelGGL((k_sfac<MODE, float>), grid, block, lds, s, g.d, m, stale, groups);
              return;
            }
          hipLaunchKernelGGL((k_sfac<MODE, double>), grid, block, lds, s, g.d, m, stale, groups);
        });
  if (part & 2)
    launch_over(
        g,
        [&](const SysConst &c, const MDConst &) {
          const Plan p = plan(c);
          if (p.variant < 0) return p;
          return Plan{p.variant & 1, idiv(32L * col_tiles(c) * kz_steps(c.lmax), 256), c.P, 1, 0};
        },
        [&](int v, dim3 grid, const BlockMap &m, size_t) {
          if constexpr (MODE == SF_D)
            if (v & 1) {
              hipLaunchKernelGGL((k_sfac_reduce<MODE, float>), grid, dim3(256), 0, s, g.d, m, stale);
              return;
            }
          hipLaunchKernelGGL((k_sfac_reduce<MODE, double>), grid, dim3(256), 0, s, g.d, m, stale);
        });
}

// Variant: bit 0 TTM3-F site sets (the fixed-charge models share them), bit 1
// FP32 (the mixed form's SOR iterations; its refinement, iter < 0, in FP64),
// above them the
// site and column groups and the tiles per group.  sel_mixed: only the mixed-form replicas.
template <int MO>
static void launch_field_mode(const Group &g, int iter, bool sel_mixed, hipStream_t s) {
  launch_over(
      g,
      [&](const SysConst &c, const MDConst &) {
        if ((MO != FD_Q && !has_dipoles(c)) || (sel_mixed && !c.mixed) || (MO == FD_D && c.dense))
          return Plan{-1, 0, 0, 0, 0};
        const bool f32 = MO == FD_D && c.mixed && iter > 0;
        const int M = MO == FD_D ? c.nd * c.N : (c.model == 2 ? 4 : 3) * c.N;
        int nt, sg, cg;
        field_groups(c, M, nt, sg, cg);
        auto tab = [&] { return (f32 ? sizeof(float2) : sizeof(double2)) * (c.T + 1) * phase_row(sg * 16 * nt); };
        while (sg > 1 && tab() > 64 * 1024) sg /= 2;
        return Plan{(c.model == 2 ? 0 : 1) | (f32 ? 2 : 0) | (sg << 2) | (cg << 5) | (nt << 10),
                    idiv(M, sg * 16 * nt), c.P, 1,
                    std::max(tab(), sizeof(double) * cg * 4 * sg * 16 * nt)};
      },
      [&](int v, dim3 grid, const BlockMap &m, size_t lds) {
        const int sg = (v >> 2) & 7;
        const dim3 block(64 * sg * ((v >> 5) & 31));
        const bool two = (v >> 10) == 2;
#define PIMD_FIELD(ML, R)                                                                          \
  if (two) hipLaunchKernelGGL((k_field<MO, ML, R, 2>), grid, block, lds, s, g.d, m, iter, sg);     \
  else hipLaunchKernelGGL((k_field<MO, ML, R, 1>), grid, block, lds, s, g.d, m, iter, sg)
        if constexpr (MO == FD_D)
          if (v & 2) {
            if (v & 1) { PIMD_FIELD(3, float); } else { PIMD_FIELD(2, float); }
            return;
          }
        if (v & 1) { PIMD_FIELD(3, double); } else { PIMD_FIELD(2, double); }
#undef PIMD_FIELD
      });
}

// Buffer elements: the chunk sums (any_sites: enough for every sf_sites, which
// the batch tuning changes) and the field operands.
size_t sfac_part_elems(const SysConst &c0, bool any_sites) {
  SysConst c = c0;
  if (any_sites) c.sf_sites = 1;  // as many chunks as there may be
  size_t most = 0;
  for (int mode : {SF_Q, SF_D, SF_V}) {
    int nch, sc, scp;
    sfac_chunking(c, mode, nch, sc, scp);
    most = std::max(most, (size_t)nch * (mode == SF_V ? 6 : 2));
  }
  return c.P * (size_t)c.nk * most;
}
int sfac_chunks_max(const SysConst &c) {
  const int sites = std::min(64, sfac_cap(c));
  return std::max(32, (3 * c.N + sites - 1) / sites);
}
size_t field_operand_elems(const SysConst &c) {
  return wk_elems(c, WK_A + (has_dipoles(c) ? WK_B : 0));
}

// Structure-factor tasks: 16 columns (sorted by their reach) x 8 |kz| each.
std::vector<int> sfac_tasks(const std::vector<int4> &cols) {
  std::vector<int> t;
  for (int lt = 0;; ++lt) {
    const size_t before = t.size();
    for (size_t ct = 0; ct * 16 < cols.size(); ++ct) {
      const int4 cl = cols[ct * 16];
      if (std::max(std::abs(cl.z), std::abs(cl.z + cl.w - 1)) >= 8 * lt) t.push_back((int)ct | (lt << 16));
    }
    if (t.size() == before) return t;
  }
}

// The columns as the kernels read them, the last one repeated up to a whole tile.
std::vector<ColRec> column_records(const SysConst &c, const std::vector<int4> &cols) {
  std::vector<ColRec> r((size_t)col_tiles(c) * 16);
  for (size_t i = 0; i < r.size() && !cols.empty(); ++i) {
    const int4 cl = cols[std::min(i, cols.size() - 1)];
    r[i] = ColRec{TWOPI * c.boxi[0] * cl.x, TWOPI * c.boxi[1] * cl.y, cl.x,
                  c.hmax + 1 + std::abs(cl.y), cl.y < 0 ? INT_MIN : 0,
                  std::max(std::abs(cl.z), std::abs(cl.z + cl.w - 1))};
  }
  return r;
}

void launch_tables(const Group &g, hipStream_t s) {
  launch_over(
      g, [](const SysConst &c, const MDConst &) { return Plan{0, idiv(4 * c.N, 256), c.P, 1, 0}; },
      [&](int, dim3 grid, const BlockMap &m, size_t) {
        hipLaunchKernelGGL(k_tables, grid, dim3(256), 0, s, g.d, m);
      });
}

void launch_sfac(const Group &g, int mode, hipStream_t s, int sel, int part) {
  if (mode == SF_Q) launch_sfac_mode<SF_Q>(g, SFAC_ITER, part, s);
  else if (mode == SF_D) launch_sfac_mode<SF_D>(g, sel, part, s);
  else launch_sfac_mode<SF_V>(g, SFAC_ITER, part, s);
}

void launch_field(const Group &g, int mode, int iter, hipStream_t s, bool sel_mixed) {
  if (mode == FD_Q) launch_field_mode<FD_Q>(g, iter, sel_mixed, s);
  else if (mode == FD_D) launch_field_mode<FD_D>(g, iter, sel_mixed, s);
  else launch_field_mode<FD_QD>(g, iter, sel_mixed, s);
}

}  // namespace pimd
