// recip.hip -- reciprocal-space Ewald sums for gfx950.
//
// Reference: multipole_ES_rec (src/ewald_rec.f90:38-365) with the half-space
// k mesh of kpoint_sum_init (src/kspace.f90:143-207).  The reference loops
// over (k, atom) pairs and calls FP64 COS/SIN of k.r for each.  Here the
// mesh is treated as the box nx in [0,Kx], ny in [-Ky,Ky], nz in [-Kz,Kz]
// (entries outside the half space, and k = 0, carry A(n) = 0), and
// e^{i k.r} = X[nx] Y[ny] Z[nz] with per-dimension phase tables
// X[n] = e^{2 pi i n s_x} (s = B^double r, k.r = 2 pi n.s).  Every phase angle is
// formed in FP64, and all of it is summed in FP64, in the mixed form too: the
// sums over k cancel, and below the sizes that go to the mesh (mesh.hip) the
// FP64 matrix cores are the faster way to the same error.
//
//   phase 1  S(n) = sum_i a_i(n) X_i[nx] Y_i[ny] Z_i[nz],
//            a_i(n) = q_i + i 2 pi n.m_i,  m_i = B^double mu_i   (src/ewald_rec.f90:116-148)
//   reduce   S in FP64; W(n) = A(n) conj(S(n)); energy sum A|S|^2 and the
//            stress sum (delta - kcoe k k) A|S|^2              (:173-174, :252-263)
//   phase 2  per atom: U1_d = sum_n n_d Im(W e_i), M_de = sum_n n_d n_e Re(W e_i)
//            field = 2 (4 pi/V) 2 pi B U1; force = 2 (4 pi/V) [q_i 2 pi B U1
//            + (2 pi)^2 B M m_i]                               (:196-233, :300-358)
#include <cstdlib>
#include <type_traits>
#include <utility>

#include "common.h"
#include "reduce.h"

struct cplx {
  double re, im;
};

namespace {

__device__ __forceinline__ cplx cmul(cplx a, cplx b) {
  return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}

// Phase tables, layout [col][atom], col = 0..Kx (X), Kx+1..Kx+Ky+1 (Y), then Z.
// A thread writes a run of up to kTabRun consecutive columns of one
// direction: exp(2 pi i k0 s) by sincospi of the reduced angle k0 s - rint(k0 s),
// then E(k + 1) = E(k) E(1) in FP64 (at most kTabRun - 1 products, each
// within a few units of 2^-53).
constexpr int kTabRun = 8;

// runs of the three directions: blockIdx.y -> (first column, k0, count, which s)
struct TabRun {
  int col, k0, cnt, dir;
};
__device__ __forceinline__ TabRun tab_run(int y, int Kx, int Ky, int Kz) {
  const int rx = (Kx + kTabRun) / kTabRun, ry = (Ky + kTabRun) / kTabRun;
  TabRun r;
  int K, base;
  if (y < rx) { r.dir = 0; K = Kx; base = 0; }
  else if (y < rx + ry) { r.dir = 1; K = Ky; base = Kx + 1; y -= rx; }
  else { r.dir = 2; K = Kz; base = Kx + Ky + 2; y -= rx + ry; }
  r.k0 = y * kTabRun;
  r.cnt = min(kTabRun, K + 1 - r.k0);
  r.col = base + r.k0;
  return r;
}
static int tab_runs(const int* K) {
  return (K[0] + kTabRun) / kTabRun + (K[1] + kTabRun) / kTabRun + (K[2] + kTabRun) / kTabRun;
}

__device__ __forceinline__ void table_run(double s, const TabRun& r, int n, int i, cplx* __restrict__ tab) {
  double t = (double)r.k0 * s;
  t -= rint(t);
  double sn, cs;
  sincospi(2.0 * t, &sn, &cs);
  double t1 = s - rint(s);
  double s1, c1;
  sincospi(2.0 * t1, &s1, &c1);
  cplx* dst = tab + (size_t)r.col * n + i;
  dst[0] = {cs, sn};
  for (int u = 1; u < r.cnt; ++u) {
    const double c2 = cs * c1 - sn * s1, s2 = cs * s1 + sn * c1;
    cs = c2;
    sn = s2;
    dst[(size_t)u * n] = {cs, sn};
  }
}

__global__ void k_tables(int n, int Kx, int Ky, int Kz, const double* __restrict__ sx,
                         const double* __restrict__ sy, const double* __restrict__ sz,
                         cplx* __restrict__ tab) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const TabRun r = tab_run(blockIdx.y, Kx, Ky, Kz);
  const double s = r.dir == 0 ? sx[i] : (r.dir == 1 ? sy[i] : sz[i]);
  table_run(s, r, n, i, tab);
}

// The same tables straight from the Cartesian positions: s = B^double r formed
// as kardir does (src/lattice.f90:183-216, products and sums rounded
// separately, no fused multiply-add), so s is bit-identical to the list
// code's; the blocks of the first run (X columns from 0) also store s (sx,
// sy, sz).
struct TabRArgs {
  int n, Kx, Ky, Kz;
  const double *rx, *ry, *rz;
  double b[9];                   // B column-major
  double *sx, *sy, *sz;
  cplx* tab;
  // pack != 0: also the atoms in the cell order of the last list build
  // (rec[p], meta[p] of atom order[p], as pack_atoms)
  int pack;
  const int32_t* order;
  const double* q;
  const int32_t* itype;
  AtomRec* rec;
  int2* meta;
};

// fin_row >= 0: the blocks of row blockIdx.y == fin_row run the queued final
// sums of the previous MD step instead (block x: sum x).
__global__ void __launch_bounds__(256) k_tables_r(TabRArgs a, FinalBatch fb, int fin_row) {
  if ((int)blockIdx.y == fin_row) {
    __shared__ double sh[4 * kRedMaxCols];
    run_final_batch(fb, blockIdx.x, sh);
    return;
  }
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  auto dot = [](double x, double y, double z, double u, double v, double w) {
    return __dadd_rn(__dadd_rn(__dmul_rn(x, u), __dmul_rn(y, v)), __dmul_rn(z, w));
  };
  const double* b = a.b;
  const double x = a.rx[i], y = a.ry[i], z = a.rz[i];
  const TabRun r = tab_run(blockIdx.y, a.Kx, a.Ky, a.Kz);
  if (blockIdx.y == 0) {
    a.sx[i] = dot(x, y, z, b[0], b[1], b[2]);
    a.sy[i] = dot(x, y, z, b[3], b[4], b[5]);
    a.sz[i] = dot(x, y, z, b[6], b[7], b[8]);
    if (a.pack) {
      const int j = a.order[i];
      const double xj = a.rx[j], yj = a.ry[j], zj = a.rz[j];
      a.rec[i] = AtomRec{dot(xj, yj, zj, b[0], b[1], b[2]), dot(xj, yj, zj, b[3], b[4], b[5]),
                         dot(xj, yj, zj, b[6], b[7], b[8]), a.q[j]};
      a.meta[i] = make_int2(a.itype[j], j);
    }
  }
  const double s = r.dir == 0 ? dot(x, y, z, b[0], b[1], b[2])
                              : (r.dir == 1 ? dot(x, y, z, b[3], b[4], b[5]) : dot(x, y, z, b[6], b[7], b[8]));
  table_run(s, r, a.n, i, a.tab);
}

// A, k vector and kcoe on the box, A = 0 outside the half space (n_x > 0, or 0 and
// n_y > 0, or both 0 and n_z > 0)
struct BoxArgs {
  int K[3];
  double b[9], alpha2;
  double *A, *kvec;
};
__global__ void __launch_bounds__(256) k_box_weights(BoxArgs a) {
  const int NY = 2 * a.K[1] + 1, NZ = 2 * a.K[2] + 1;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= (a.K[0] + 1) * NY * NZ) return;
  const int z = i % NZ - a.K[2], xy = i / NZ, y = xy % NY - a.K[1], x = xy / NY;
  const bool half = x > 0 || (x == 0 && y > 0) || (x == 0 && y == 0 && z > 0);
  const KWeight w = k_weight(a.b, a.alpha2, x, y, z);
  a.A[i] = half ? w.A : 0.0;
  a.kvec[4 * (size_t)i] = w.kx;
  a.kvec[4 * (size_t)i + 1] = w.ky;
  a.kvec[4 * (size_t)i + 2] = w.kz;
  a.kvec[4 * (size_t)i + 3] = half ? w.kc : 0.0;
}

struct SkArgs {
  int n, Kx, Ky, Kz, NY, NZ, M, NG, GZ;
  int use_q, use_mu;
  int a0_step;                   // atoms per chunk
  int TA;                        // atoms per LDS tile
  const double* q;
  const double* mu;              // 3n AoS
  double b[9];                   // B column-major
  const cplx* tab;
  double* part;                  // [chunk][2*nk_box]
  int nk_box;
};

// Phase 1.  Work item = (g, m): m = nx*NY + (ny+Ky), g = group of GZ
// consecutive nz.  Consecutive lanes take consecutive m, so the Y loads are
// consecutive and the Z loads are wave-uniform (LDS broadcast).
template <int GZ>
__global__ void __launch_bounds__(256) k_sk(SkArgs a) {
  const int TA = a.TA;
  extern __shared__ unsigned char smem_raw[];
  const int ncol = a.Kx + 1 + a.Ky + 1 + a.Kz + 1;
  cplx* st = reinterpret_cast<cplx*>(smem_raw);          // [ncol][TA]
  double* sq = reinterpret_cast<double*>(st + (size_t)ncol * TA);         // q, mx, my, mz per atom
  const cplx* tab = a.tab;
  const int item = blockIdx.x * blockDim.x + threadIdx.x;
  const int m = item % a.M;
  const int g = item / a.M;
  const bool active = g < a.NG;
  const int nx = m / a.NY, ny = m % a.NY - a.Ky;
  const int nz0 = g * GZ - a.Kz;
  const double tp = 2.0 * MDFF_PI;
  cplx acc[GZ];
#pragma unroll
  for (int k = 0; k < GZ; ++k) acc[k] = {0.0, 0.0};
  const int abeg = blockIdx.y * a.a0_step;
  const int aend = min(a.n, abeg + a.a0_step);
  for (int t0 = abeg; t0 < aend; t0 += TA) {
    const int nt = min(TA, aend - t0);
    __syncthreads();
    for (int x = threadIdx.x; x < ncol * TA; x += blockDim.x) {
      int col = x / TA, ia = x % TA;
      st[x] = (ia < nt) ? tab[(size_t)col * a.n + t0 + ia] : cplx{0.0, 0.0};
    }
    for (int ia = threadIdx.x; ia < TA; ia += blockDim.x) {
      double qq = 0.0, mx = 0.0, my = 0.0, mz = 0.0;
      if (ia < nt) {
        int i = t0 + ia;
        if (a.use_q) qq = a.q[i];
        if (a.use_mu) {
          double u0 = a.mu[3 * i], u1 = a.mu[3 * i + 1], u2 = a.mu[3 * i + 2];
          // m = B^double mu
          mx = u0 * a.b[0] + u1 * a.b[1] + u2 * a.b[2];
          my = u0 * a.b[3] + u1 * a.b[4] + u2 * a.b[5];
          mz = u0 * a.b[6] + u1 * a.b[7] + u2 * a.b[8];
        }
      }
      sq[4 * ia] = qq;
      sq[4 * ia + 1] = mx;
      sq[4 * ia + 2] = my;
      sq[4 * ia + 3] = mz;
    }
    __syncthreads();
    if (active) {
      for (int ia = 0; ia < nt; ++ia) {
        const cplx X = st[nx * TA + ia];
        cplx Y = st[(a.Kx + 1 + (ny >= 0 ? ny : -ny)) * TA + ia];
        if (ny < 0) Y.im = -Y.im;
        const cplx XY = cmul(X, Y);
        const double qq = sq[4 * ia];
        cplx P, Pz{0.0, 0.0};
        if (a.use_mu) {
          // a = q + i 2pi (nx mx + ny my) ; the nz part is added per nz
          const double b = tp * ((double)nx * sq[4 * ia + 1] + (double)ny * sq[4 * ia + 2]);
          P = {qq * XY.re - b * XY.im, qq * XY.im + b * XY.re};
          const double c = tp * sq[4 * ia + 3];
          Pz = {-c * XY.im, c * XY.re};
        } else {
          P = {qq * XY.re, qq * XY.im};
        }
        const int zb = (a.Kx + 1 + a.Ky + 1) * TA + ia;
#pragma unroll
        for (int k = 0; k < GZ; ++k) {
          const int nz = nz0 + k;
          const int az = nz >= 0 ? nz : -nz;
          if (az > a.Kz) continue;
          cplx Z = st[zb + az * TA];
          if (nz < 0) Z.im = -Z.im;
          cplx Pk = P;
          if (a.use_mu) {
            Pk.re += (double)nz * Pz.re;
            Pk.im += (double)nz * Pz.im;
          }
          acc[k].re += Pk.re * Z.re - Pk.im * Z.im;
          acc[k].im += Pk.re * Z.im + Pk.im * Z.re;
        }
      }
    }
  }
  if (!active) return;
  double* out = a.part + (size_t)blockIdx.y * 2 * a.nk_box;
#pragma unroll
  for (int k = 0; k < GZ; ++k) {
    const int nz = nz0 + k;
    if (nz > a.Kz) continue;
    const int idx = m * a.NZ + (nz + a.Kz);
    out[2 * idx] = acc[k].re;
    out[2 * idx + 1] = acc[k].im;
  }
}

__host__ __device__ __forceinline__ int row_of(int ml, int comp);

// S(n) = sum of chunk partials (FP64, fixed order: a wave a quarter of the
// chunks of 64 k, so that few k still have loads enough in flight); W(n) = A conj(S);
// per-block sums of A|S|^2 and (delta_ab - kcoe k_a k_b) A|S|^2.  With amat,
// also the A operand of the matrix-core gather: amat[(mtile * nks + s) * 64
// + lane] holds, for m = 4 mtile + ml and K index kk = 4 s + lane / 16 =
// (nz index t, Re/Im cc), row R = lane % 16 = (ml, component comp):
// (Re, Im) of W Z as a real dot product with (Re Z, Im Z), times nz for
// comp >= 2.  Entries outside the mesh are never written (zero from setup).
__global__ void __launch_bounds__(256) k_sk_reduce(int nk_box, int nchunk, const double* __restrict__ part,
                                                   const double* __restrict__ kA,
                                                   const double* __restrict__ kvec,
                                                   double* __restrict__ wk, double* __restrict__ blk,
                                                   double* __restrict__ amat, int NZ, int Kz, int nks) {
  __shared__ double sh[4 * kRedMaxCols];
  __shared__ double2 quarter[4][64];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int k = blockIdx.x * 64 + lane;
  double v[kRedMaxCols];
#pragma unroll
  for (int c = 0; c < kRedMaxCols; ++c) v[c] = 0.0;
  {
    // chunks in order; the loads of 8 chunks are issued before their adds
    double2 t = {0.0, 0.0};
    const double2* src = reinterpret_cast<const double2*>(part) + min(k, nk_box - 1);
    const int per = (nchunk + 3) >> 2, c1 = min(nchunk, (wave + 1) * per);
    for (int c = wave * per; c < c1; c += 8) {
      double2 u8[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) u8[u] = src[(size_t)min(c + u, c1 - 1) * nk_box];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (c + u < c1) {
          t.x += u8[u].x;
          t.y += u8[u].y;
        }
    }
    quarter[wave][lane] = t;
  }
  __syncthreads();
  if (wave == 0 && k < nk_box) {
    double re = 0.0, im = 0.0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      re += quarter[w][lane].x;
      im += quarter[w][lane].y;
    }
    const double Ak = kA[k];
    wk[2 * k] = Ak * re;
    wk[2 * k + 1] = -Ak * im;
    if (amat) {
      const double wr = Ak * re, wi = -Ak * im;
      const int m = k / NZ, t = k - (k / NZ) * NZ;
      const int mt = m >> 2, ml = m & 3;
      const double fz = (double)(t - Kz);
#pragma unroll
      for (int cc = 0; cc < 2; ++cc) {
        const int kk = 2 * t + cc;
        double* dst = amat + ((size_t)mt * nks + (kk >> 2)) * 64 + 16 * (kk & 3);
#pragma unroll
        for (int comp = 0; comp < 4; ++comp) {
          double v = ((comp & 1) == 0) ? (cc == 0 ? wr : -wi) : (cc == 0 ? wi : wr);
          if (comp >= 2) v *= fz;
          dst[row_of(ml, comp)] = v;
        }
      }
    }
    const double str = (re * re + im * im) * Ak;
    const double kx = kvec[4 * k], ky = kvec[4 * k + 1], kz = kvec[4 * k + 2], kc = kvec[4 * k + 3];
    v[0] = str;
    v[1] = (1.0 - kc * kx * kx) * str;
    v[2] = (1.0 - kc * ky * ky) * str;
    v[3] = (1.0 - kc * kz * kz) * str;
    v[4] = -kc * kx * ky * str;
    v[5] = -kc * kx * kz * str;
    v[6] = -kc * ky * kz * str;
  }
  const double r = block_sum_cols(v, 7, sh);
  if (threadIdx.x < 7) blk[blockIdx.x * 7 + threadIdx.x] = r;
}

struct GaArgs {
  int n, Kx, Ky, Kz, NY, NZ, M, m_per_split;
  int moments;                   // 3 (field / charge forces) or 9 (dipole forces)
  const cplx* tab;
  const double* wk;              // W(n), 2 x nk_box
  double* out;                   // [split][moments][n]
};

// Phase 2: one thread per atom, W streamed through LDS (wave-uniform reads),
// the atom's own Z row held in LDS as [nz][thread] (conflict-free).
template <int MOM>
__global__ void __launch_bounds__(256) k_gather(GaArgs a) {
  extern __shared__ unsigned char smem_raw[];
  constexpr int MT = 8;                                     // m values per W tile
  const int nthr = blockDim.x;
  cplx* zt = reinterpret_cast<cplx*>(smem_raw);       // [Kz+1][nthr]
  cplx* wt = zt + (size_t)(a.Kz + 1) * nthr;             // [MT][NZ]
  const cplx* tab = a.tab;
  const cplx* W = reinterpret_cast<const cplx*>(a.wk);
  const int i = blockIdx.x * nthr + threadIdx.x;
  const bool act = i < a.n;
  const int zcol = a.Kx + 1 + a.Ky + 1;
  for (int k = 0; k <= a.Kz; ++k)
    zt[k * nthr + threadIdx.x] = act ? tab[(size_t)(zcol + k) * a.n + i] : cplx{0.0, 0.0};
  double u0 = 0, u1 = 0, u2 = 0, mxx = 0, myy = 0, mzz = 0, mxy = 0, mxz = 0, myz = 0;
  const int mbeg = blockIdx.y * a.m_per_split;
  const int mend = min(a.M, mbeg + a.m_per_split);
  for (int mt = mbeg; mt < mend; mt += MT) {
    const int nm = min(MT, mend - mt);
    __syncthreads();
    for (int x = threadIdx.x; x < nm * a.NZ; x += nthr) wt[x] = W[(size_t)mt * a.NZ + x];
    __syncthreads();
    if (!act) continue;
    for (int mm = 0; mm < nm; ++mm) {
      const int m = mt + mm;
      const int nx = m / a.NY, ny = m % a.NY - a.Ky;
      cplx X = tab[(size_t)nx * a.n + i];
      cplx Y = tab[(size_t)(a.Kx + 1 + (ny >= 0 ? ny : -ny)) * a.n + i];
      if (ny < 0) Y.im = -Y.im;
      const cplx XY = cmul(X, Y);
      double z0r = 0, z0i = 0, z1r = 0, z1i = 0, z2r = 0, z2i = 0;
      const cplx* wrow = wt + mm * a.NZ;
      // negative nz: Z = conj(Z[|nz|])
      for (int az = a.Kz; az >= 1; --az) {
        const cplx w = wrow[a.Kz - az];
        const cplx z = zt[az * nthr + threadIdx.x];
        const double tr = w.re * z.re + w.im * z.im;   // w * conj(z)
        const double ti = w.im * z.re - w.re * z.im;
        const double fz = -(double)az;
        z0r += tr; z0i += ti;
        z1r += fz * tr; z1i += fz * ti;
        if (MOM == 9) { z2r += fz * fz * tr; z2i += fz * fz * ti; }
      }
      for (int az = 0; az <= a.Kz; ++az) {
        const cplx w = wrow[a.Kz + az];
        const cplx z = zt[az * nthr + threadIdx.x];
        const double tr = w.re * z.re - w.im * z.im;
        const double ti = w.re * z.im + w.im * z.re;
        const double fz = (double)az;
        z0r += tr; z0i += ti;
        z1r += fz * tr; z1i += fz * ti;
        if (MOM == 9) { z2r += fz * fz * tr; z2i += fz * fz * ti; }
      }
      // Im and Re of XY * Z_p
      const double i0 = XY.re * z0i + XY.im * z0r, r0 = XY.re * z0r - XY.im * z0i;
      const double i1 = XY.re * z1i + XY.im * z1r, r1 = XY.re * z1r - XY.im * z1i;
      const double fx = (double)nx, fy = (double)ny;
      u0 += fx * i0;
      u1 += fy * i0;
      u2 += i1;
      if (MOM == 9) {
        const double r2 = XY.re * z2r - XY.im * z2i;
        mxx += fx * fx * r0;
        myy += fy * fy * r0;
        mxy += fx * fy * r0;
        mxz += fx * r1;
        myz += fy * r1;
        mzz += r2;
      }
    }
  }
  if (!act) return;
  double* o = a.out + (size_t)blockIdx.y * MOM * a.n;
  o[i] = u0;
  o[(size_t)a.n + i] = u1;
  o[(size_t)2 * a.n + i] = u2;
  if (MOM == 9) {
    o[(size_t)3 * a.n + i] = mxx;
    o[(size_t)4 * a.n + i] = myy;
    o[(size_t)5 * a.n + i] = mzz;
    o[(size_t)6 * a.n + i] = mxy;
    o[(size_t)7 * a.n + i] = mxz;
    o[(size_t)8 * a.n + i] = myz;
  }
}

// sum over splits, then field / force in Cartesian (src/ewald_rec.f90:196-233,
// scaled as :300-358: x2 for the half mesh, x 4pi/V)
__global__ void k_gather_final(RecFinal r, int field, int forces, double* __restrict__ ef,
                               double* __restrict__ f) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= r.n) return;
  double v[9], g[3];
  rec_final_moments(r, i, v, g);
  if (field) {
    double e[3];
    rec_final_field(r, g, e);
    ef[3 * i] = e[0];
    ef[3 * i + 1] = e[1];
    ef[3 * i + 2] = e[2];
  }
  if (forces) {
    double fv[3];
    rec_final_force(r, i, v, g, fv);
    f[3 * i] = fv[0];
    f[3 * i + 1] = fv[1];
    f[3 * i + 2] = fv[2];
  }
}


// ---------------------------------------------------------------------------
// Matrix-core form of phase 2.
//
// For one 16-atom tile the contraction over nz is a real GEMM on MFMA
// 16x16x4: rows R = (m_local, comp) of 4 values of m = (nx, ny) and four
// components comp = (Re U0, Im U0, Re U1, Im U1), U_p(i, m) = sum_nz nz^p
// W(m, nz) Z_i(nz); K = (nz, re/im of Z) padded to a multiple of 4; columns =
// the 16 atoms.  The A operand (W, arranged per lane) is written once per
// evaluation by k_sk_reduce; the B operand (the atom's Z row) stays in
// registers for the whole kernel.  With the row order below, lane l holds the
// four components of atom (l % 16) for m_local = l / 16 in its four
// accumulator registers, so the (nx, ny) epilogue (multiply by
// X_i[nx] Y_i[ny], weight by nx, ny) is lane-local; the four m_local lane
// groups are summed with two cross-lane shuffles at the very end.
//
// Second moments (MOM 9) need U2 too: a second product of the same A operand
// with nz Z has (U1, U2) in its rows, so it costs one multiply a step and no
// second A operand (a gradient evaluation of 480 ions 339 us with the
// vector-ALU gather, 217 with this; of 4,096 ions 437 and 364).
// Lane layouts (checked on gfx950): A(row = l%16, k = l/16), B(k = l/16,
// col = l%16); D f32: row = 4*(l/16) + r; D f64: row = 4*r + l/16.
// ---------------------------------------------------------------------------
typedef double f64x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f64x4 mfma(double a, double b, f64x4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
// row of the A operand for (m_local, comp)
__host__ __device__ __forceinline__ int row_of(int ml, int comp) { return 4 * comp + ml; }

struct GmArgs {
  int n, Kx, Ky, Kz, NY, NZ, M, nks, mt_per_split, mtiles;
  const cplx* tab;
  const double* amat;
  double* out;                   // [split][moments][n]
};

// Two waves per SIMD where the B operand, the double-buffered A operand and
// the accumulators fit in 256 registers without spills (the instances
// listed), one otherwise.
template <int CT, int NKS, int MOM>
constexpr int gather_waves() {
  return NKS <= 25 || (MOM == 3 && NKS <= 33) ? 2 : 1;
}

template <int CT, int NKS, int MOM>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(gather_waves<CT, NKS, MOM>())))
k_gather_mma(GmArgs a) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int g = lane >> 4, col = lane & 15;
  const int atom0 = (blockIdx.x * (blockDim.x >> 6) + wave) * (16 * CT);
  const cplx* tab = a.tab;
  const double* amat = a.amat;
  const int zcol = a.Kx + 1 + a.Ky + 1;
  // B operand: the Z row of this lane's atoms, zero beyond NZ.  Every load
  // reads a clamped, valid address and the zero is selected afterwards, so
  // all CT * NKS loads are in flight together.
  double breg[CT][NKS];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const int ia = atom0 + ct * 16 + col;
    const bool ok = ia < a.n;
    const int iac = min(ia, a.n - 1);
#pragma unroll
    for (int s = 0; s < NKS; ++s) {
      const int k = 4 * s + g;
      const int t = k >> 1;
      const int nz = t - a.Kz;
      const int az = min(nz < 0 ? -nz : nz, a.Kz);
      // Re (k even) or Im (k odd) of Z, conjugated for nz < 0
      const double v = reinterpret_cast<const double*>(tab + (size_t)(zcol + az) * a.n + iac)[k & 1];
      const double w = (ok && t < a.NZ) ? (((k & 1) && nz < 0) ? -1.0 : 1.0) : 0.0;
      breg[ct][s] = w * v;
    }
  }
  double ax[CT], ay[CT], az3[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) { ax[ct] = 0.0; ay[ct] = 0.0; az3[ct] = 0.0; }
  // MOM 9: xx, yy, zz, xy, xz, yz sums of n n Re(W e); nz of this lane's first K index
  double sec[MOM == 9 ? CT : 1][6] = {};
  const double nz0 = (double)((g >> 1) - a.Kz);
  const int mt0 = blockIdx.y * a.mt_per_split;
  const int mt1 = min(a.mtiles, mt0 + a.mt_per_split);
  // The A operand of tile mt+1 is loaded at the top of tile mt; the
  // epilogue's X[nx] Y[ny] rows of tile mt at its top, used after its MFMAs
  // (a scheduling barrier keeps their use, and so the wait for them, behind
  // the MFMAs).  Addresses are clamped to valid rows, lanes beyond M get a
  // zero weight, so nothing here branches.  The lane's m advances by 4 per
  // tile; (nx, ny + Ky) are stepped, not divided.
  int m = 4 * mt0 + g;
  int nx = min(m, a.M - 1) / a.NY;
  int nyo = min(m, a.M - 1) - nx * a.NY;                          // ny + Ky
  int iac[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) iac[ct] = min(atom0 + ct * 16 + col, a.n - 1);
  double abuf[NKS];
  auto load_a = [&](int mtl) {
    const double* ap = amat + (size_t)mtl * NKS * 64 + lane;
#pragma unroll
    for (int s = 0; s < NKS; ++s) abuf[s] = ap[(size_t)s * 64];
  };
  if (mt0 < mt1) load_a(mt0);
  for (int mt = mt0; mt < mt1; ++mt) {
    double cur[NKS];
#pragma unroll
    for (int s = 0; s < NKS; ++s) cur[s] = abuf[s];
    cplx Xv[CT], Yv[CT];
    {
      const int nyy = nyo - a.Ky;
      const size_t xrow = (size_t)min(nx, a.Kx) * a.n, yrow = (size_t)(a.Kx + 1 + (nyy >= 0 ? nyy : -nyy)) * a.n;
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        Xv[ct] = tab[xrow + iac[ct]];
        Yv[ct] = tab[yrow + iac[ct]];
      }
    }
    const double mw = m < a.M ? 1.0 : 0.0;
    const int ny = nyo - a.Ky;
    const double fx = (double)nx, fy = (double)ny;
    const double ysg = ny < 0 ? -1.0 : 1.0;
    // the next tile's m
    m += 4;
    nyo += 4;
    while (nyo >= a.NY) { nyo -= a.NY; ++nx; }          // NY = 2 Ky + 1 may be below 4
    if (mt + 1 < mt1) load_a(mt + 1);
    f64x4 acc[CT], acn[MOM == 9 ? CT : 1];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      acc[ct] = f64x4{0.0, 0.0, 0.0, 0.0};
      if (MOM == 9) acn[ct] = acc[ct];
    }
#pragma unroll
    for (int s = 0; s < NKS; ++s) {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        acc[ct] = mfma(cur[s], breg[ct][s], acc[ct]);
        if (MOM == 9) acn[ct] = mfma(cur[s], (nz0 + 2.0 * s) * breg[ct][s], acn[ct]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      cplx Y = Yv[ct];
      Y.im *= ysg;
      cplx XY = cmul(Xv[ct], Y);
      XY.re *= mw;
      XY.im *= mw;
      const double im0 = XY.re * acc[ct][1] + XY.im * acc[ct][0];
      const double im1 = XY.re * acc[ct][3] + XY.im * acc[ct][2];
      ax[ct] += fx * im0;
      ay[ct] += fy * im0;
      az3[ct] += im1;
      if (MOM == 9) {
        const double re0 = XY.re * acc[ct][0] - XY.im * acc[ct][1];
        const double re1 = XY.re * acc[ct][2] - XY.im * acc[ct][3];
        const double re2 = XY.re * acn[ct][2] - XY.im * acn[ct][3];
        sec[ct][0] += fx * fx * re0;
        sec[ct][1] += fy * fy * re0;
        sec[ct][2] += re2;
        sec[ct][3] += fx * fy * re0;
        sec[ct][4] += fx * re1;
        sec[ct][5] += fy * re1;
      }
    }
  }
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    ax[ct] += __shfl_xor(ax[ct], 16);
    ax[ct] += __shfl_xor(ax[ct], 32);
    ay[ct] += __shfl_xor(ay[ct], 16);
    ay[ct] += __shfl_xor(ay[ct], 32);
    az3[ct] += __shfl_xor(az3[ct], 16);
    az3[ct] += __shfl_xor(az3[ct], 32);
    if (MOM == 9)
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        sec[ct][k] += __shfl_xor(sec[ct][k], 16);
        sec[ct][k] += __shfl_xor(sec[ct][k], 32);
      }
  }
  if (g == 0) {
    double* o = a.out + (size_t)blockIdx.y * MOM * a.n;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      const int ia = atom0 + ct * 16 + col;
      if (ia < a.n) {
        o[ia] = ax[ct];
        o[(size_t)a.n + ia] = ay[ct];
        o[(size_t)2 * a.n + ia] = az3[ct];
        if (MOM == 9)
#pragma unroll
          for (int k = 0; k < 6; ++k) o[(size_t)(3 + k) * a.n + ia] = sec[ct][k];
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Matrix-core structure factor, transposed form: S^T(nz, m) = sum_i
// Z_i(nz) P_i(m), m = (nx, ny).  A block's four waves take 16 columns m each
// and RT row tiles of 16 rows (nz, Re/Im), 8 nz a tile; K = (atom, Re/Im of
// P).  Rows come straight from the Z table; P_i(m) = a_i X_i[nx] Y_i[ny] is
// made once per lane and K step and feeds all RT row tiles.
//   charges: a = q
//   dipoles: a = q + i 2pi (nx m_x + ny m_y), and the nz m_z part as a second
//            product into the same sums, rows nz Z against i 2pi m_z X Y
// FP64 partials per chunk of atoms.  What bounds it: the FP64 matrix rate
// where the blocks fill the chip, below that a block's own chain of staging
// (latency) and products, so the host weighs tile and chunk sizes (sk_plan).
// MgO 1,440 ions, kES 9, dipoles: 9.8 us (2 x 24 + 4.5 with 7 row tiles
// whatever kES(3), tiles of 64 atoms, and two launches and a combining one for
// dipoles); 216 ions, kES 5: 5.4 us (2 x 23 + 4.4); NaCl 512 7.1 us (14.4).
// ---------------------------------------------------------------------------
struct SmArgs {
  int n, Kx, Ky, Kz, NY, NZ, M, chunk, lta, nk_box;   // 1 << lta atoms a staged tile
  const double* q;
  const double* mu;
  double b[9];
  const cplx* tab;
  double* part;                  // [chunk][2*nk_box]
};

constexpr int kSkStep = 4;       // K steps unrolled: 8 atoms, the smallest tile

template <int RT, bool DIP>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) k_sk_mma(SmArgs a) {
  extern __shared__ unsigned char smem_raw[];
  const int ncol = a.Kx + a.Ky + a.Kz + 3;
  const int TA = 1 << a.lta, TAP = TA + 2;                       // padded atom stride of a staged column
  // staged tile, column-major: st[col * TAP + atom]; then the a-coefficients
  // sq[c * TAP + atom], c = 0..3.  A K step advances the atom by 2, a fixed
  // byte offset, so the unrolled step loop addresses LDS with immediates.
  cplx* st = reinterpret_cast<cplx*>(smem_raw);
  double* sq = reinterpret_cast<double*>(st + (size_t)ncol * TAP);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane >> 4, col = lane & 15;
  const int kk = g & 1, ja = g >> 1;                             // K: atom 2s+ja, Re/Im kk
  const int zcol = a.Kx + 1 + a.Ky + 1;
  // A rows of this lane (R = col): nz index and part per row tile.  A =
  // part 0: (Zr, -Zi); part 1: (Zi, Zr), with Z(-n) = conj Z(n).  Rows
  // beyond NZ read a valid column; their D rows are never stored.
  const int zoff = blockIdx.z * (RT * 8);                       // nz rows of this block
  const bool take_im = (col & 1) ^ kk;                           // which Z component feeds A
  const double* stT = reinterpret_cast<const double*>(st);
  const double* zp[RT];
  double zs[RT], zn[DIP ? RT : 1];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int nzi = zoff + rt * 8 + (col >> 1);
    const int part = col & 1;
    const int nz = nzi - a.Kz;
    const int zc = nzi < a.NZ ? zcol + (nz < 0 ? -nz : nz) : zcol;
    const double sgn_im = nz < 0 ? -1.0 : 1.0;
    zs[rt] = part == 0 ? (kk == 0 ? 1.0 : -sgn_im) : (kk == 0 ? sgn_im : 1.0);
    if (DIP) zn[rt] = nz;
    zp[rt] = stT + 2 * ((size_t)zc * TAP + ja) + (take_im ? 1 : 0);
  }
  // B column of this lane
  const int m = (blockIdx.x * (blockDim.x >> 6) + wave) * 16 + col;
  const bool bok = m < a.M;
  const int nx = bok ? m / a.NY : 0, ny = bok ? m % a.NY - a.Ky : 0;
  const cplx* xp = st + (size_t)nx * TAP + ja;
  const cplx* yp = st + (size_t)(a.Kx + 1 + (ny >= 0 ? ny : -ny)) * TAP + ja;
  const bool bneg = ny < 0;
  const double bnxf = nx, bnyf = ny;
  const double bw = bok ? 1.0 : 0.0;                            // columns beyond M: zero B (a multiply, no branch)
  const double* qp = sq + ja;
  f64x4 acc[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) acc[rt] = f64x4{0.0, 0.0, 0.0, 0.0};
  const int abeg = blockIdx.y * a.chunk;
  const int aend = min(a.n, abeg + a.chunk);
  // staging: thread -> (atom sia, columns scg, scg + CG, ...); loads from
  // clamped addresses in batches of 8, so they are in flight together
  const int CG = 256 >> a.lta;
  const int sia = threadIdx.x & (TA - 1), scg = threadIdx.x >> a.lta;
  for (int t0 = abeg; t0 < aend; t0 += TA) {
    const int nt = min(TA, aend - t0);
    const bool sok = sia < nt;
    const size_t src = (size_t)t0 + min(sia, nt - 1);
    __syncthreads();
    for (int c0 = scg; c0 < ncol; c0 += 8 * CG) {
      cplx v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = a.tab[(size_t)min(c0 + u * CG, ncol - 1) * a.n + src];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (c0 + u * CG < ncol) st[(size_t)(c0 + u * CG) * TAP + sia] = sok ? v[u] : cplx{0.0, 0.0};
    }
    if (threadIdx.x < TA) {
      const int ia = threadIdx.x;
      double c0 = 0.0, c1 = 0.0, c2 = 0.0, c3 = 0.0;
      if (ia < nt) {
        const int i = t0 + ia;
        c0 = a.q[i];
        if (DIP) {
          const double u0 = a.mu[3 * i], u1 = a.mu[3 * i + 1], u2 = a.mu[3 * i + 2];
          c1 = 2.0 * MDFF_PI * (u0 * a.b[0] + u1 * a.b[1] + u2 * a.b[2]);
          c2 = 2.0 * MDFF_PI * (u0 * a.b[3] + u1 * a.b[4] + u2 * a.b[5]);
          c3 = 2.0 * MDFF_PI * (u0 * a.b[6] + u1 * a.b[7] + u2 * a.b[8]);
        }
      }
      sq[ia] = c0;
      if (DIP) {
        sq[TAP + ia] = c1;
        sq[2 * TAP + ia] = c2;
        sq[3 * TAP + ia] = c3;
      }
    }
    __syncthreads();
    // K steps of 4: atoms 2s and 2s+1 (Re/Im of P).  Atoms beyond nt are the
    // zero padding of the staged tile: no step needs a mask.
    const int ns = (nt + 2 * kSkStep - 1) / (2 * kSkStep);
    for (int q8 = 0; q8 < ns; ++q8) {
      const int o = q8 * 2 * kSkStep;                            // first atom
#pragma unroll
      for (int s = 0; s < kSkStep; ++s) {
        double av[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) av[rt] = zs[rt] * zp[rt][2 * o + 4 * s];
        const cplx X = xp[o + 2 * s];
        const cplx Y = yp[o + 2 * s];
        const double yim = bneg ? -Y.im : Y.im;
        const double xyr = X.re * Y.re - X.im * yim;
        const double xyi = X.re * yim + X.im * Y.re;
        const double c0 = qp[o + 2 * s];
        double pre = c0 * xyr, pim = c0 * xyi;
        if (DIP) {
          // (c0 + i bb) XY, bb = 2pi (nx mx + ny my)
          const double bb = bnxf * qp[TAP + o + 2 * s] + bnyf * qp[2 * TAP + o + 2 * s];
          pre -= bb * xyi;
          pim += bb * xyr;
        }
        const double bv = bw * (kk == 0 ? pre : pim);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) acc[rt] = mfma(av[rt], bv, acc[rt]);
        if (DIP) {
          const double c3 = qp[3 * TAP + o + 2 * s];
          const double bz = bw * (kk == 0 ? -c3 * xyi : c3 * xyr);
#pragma unroll
          for (int rt = 0; rt < RT; ++rt) acc[rt] = mfma(zn[rt] * av[rt], bz, acc[rt]);
        }
      }
    }
  }
  if (!bok) return;
  // D: lane holds rows Rd(r) of column m; row Rd -> nz = rt*8 + Rd/2, part Rd%2
  double* out = a.part + (size_t)blockIdx.y * 2 * a.nk_box;
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int Rd = 4 * r + g;
      const int nzi = zoff + rt * 8 + (Rd >> 1);
      if (nzi >= a.NZ) continue;
      out[2 * ((size_t)m * a.NZ + nzi) + (Rd & 1)] = acc[rt][r];
    }
}

}  // namespace

// K-step counts compiled for the matrix-core gather (Kz + 1 rounded up)
static const int kMmaBuckets[] = {9, 13, 17, 19, 25, 33, 41, 57};
static int mma_bucket(int nks) {
  for (int b : kMmaBuckets)
    if (nks <= b) return b;
  return 0;
}
// atom tiles of 16 per wave: register budget of the B operand and the sums
static int mma_ct(int nks, int mom) { return mom == 3 && nks <= 25 ? 2 : 1; }

// the compiled matrix-core gather for NKS and the moments, or null
static const void* gather_kernel(int nks, int mom) {
#define GM_CASE(CTV, NKSV)                                                        \
  case NKSV:                                                                      \
    return mom == 9 ? reinterpret_cast<const void*>(&k_gather_mma<1, NKSV, 9>)    \
                    : reinterpret_cast<const void*>(&k_gather_mma<CTV, NKSV, 3>);
  switch (nks) {
    GM_CASE(2, 9) GM_CASE(2, 13) GM_CASE(2, 17) GM_CASE(2, 19) GM_CASE(2, 25)
    GM_CASE(1, 33) GM_CASE(1, 41) GM_CASE(1, 57)
    default: return nullptr;
  }
#undef GM_CASE
}

// the compiled matrix-core structure factor of rt row tiles (1..7)
static const void* sk_kernel(int rt, bool dip) {
#define SK_CASE(R) \
  case R: return dip ? reinterpret_cast<const void*>(&k_sk_mma<R, true>) : reinterpret_cast<const void*>(&k_sk_mma<R, false>);
  switch (rt) {
    SK_CASE(1) SK_CASE(2) SK_CASE(3) SK_CASE(4) SK_CASE(5) SK_CASE(6) SK_CASE(7)
    default: return nullptr;
  }
#undef SK_CASE
}

// Split count of a gather over mtiles m-tiles for atom_waves waves of atoms:
// every wave first loads its atoms' B operand (a prologue worth about
// kGatherPrologue m-tiles), then runs its share of the m-tiles; the time is
// taken as rounds of resident waves x (prologue + m-tiles per wave).  At
// least 4 m-tiles per wave; fewer splits win ties.  More than 64 only up to a
// block a CU, and where they pay for the longer sum over splits in the force
// kernel, kSplitCost m-tiles a split of one K step (few atoms in a large k mesh: 64
// at kES 80, 80, 50 192 -> 68 us).
constexpr double kGatherPrologue = 4.0, kSplitCost = 4.6;
static int gather_splits(int mtiles, int64_t atom_waves, int64_t conc, int cus, int nks) {
  int best_s = 1;
  double best = -1.0;
  const int most = (int)std::min<int64_t>(256, std::max<int64_t>(64, cus / div_up(atom_waves, 4)));
  for (int sp = 1; sp <= std::min(mtiles, most); ++sp) {
    if (sp > 1 && mtiles / sp < 4) break;
    const int mps = div_up(mtiles, sp);
    const int nsp = div_up(mtiles, mps);
    const int64_t rounds = (atom_waves * nsp + conc - 1) / conc;
    const double cost = (double)rounds * (kGatherPrologue + mps) + (nsp > 64 ? kSplitCost / nks * (nsp - 64) : 0.0);
    if (best < 0.0 || cost < best - 1e-9) {
      best = cost;
      best_s = nsp;
    }
  }
  return best_s;
}

// resident 256-thread blocks per CU of a kernel with `lds` bytes of LDS
static int blocks_per_cu(const void* fn, size_t lds) {
  int nb = 0;
  if (!fn || hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, fn, 256, lds) != hipSuccess || nb <= 0) nb = 1;
  return nb;
}

// LDS bytes of the matrix-core structure factor for a tile of ta atoms
static size_t sk_lds(int ncol, int ta) { return (16 * (size_t)ncol + 32) * (size_t)(ta + 2); }
// ... of the vector-ALU one
static size_t sk_valu_lds(int ncol, int ta) { return (16 * (size_t)ncol + 32) * (size_t)ta; }
// ... and of the vector-ALU gather with nthr threads a block
static size_t gather_lds(int Kz, int nthr) { return 16 * ((size_t)(Kz + 1) * nthr + 8 * (2 * (size_t)Kz + 1)); }

// LDS a block may take where no smaller tile fits: 64 KiB, 128 KiB in the mixed
// form.  This is what decides which k meshes a context is created for
// (direct_takes), the mixed form's reaching to twice the FP64 form's extent; it
// stays where it is so that the same ones are taken and refused.  Smaller tiles
// are used long before that.
static size_t lds_limit(const mdff_ctx* c) { return c->d.precision == MDFF_PREC_MIXED ? 131072 : 65536; }
static int allow_lds(mdff_ctx* c, const void* fn, size_t lds) {
  if (lds > 65536)
    HIP_TRY(c, hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  return MDFF_OK;
}

// table columns the matrix-core structure factor takes
static int sk_cols(const mdff_ctx* c) { return c->d.precision == MDFF_PREC_MIXED ? 817 : 408; }

// whether the direct kernels below take the k mesh (sums and gather both)
static bool direct_takes(const mdff_ctx* c) {
  const bool dip = c->task_qd || c->task_dd;
  const bool gather = gather_lds(c->K[2], 64) <= lds_limit(c) || (!dip && mma_bucket(c->K[2] + 1) > 0);
  return gather && c->K[0] + c->K[1] + c->K[2] + 3 <= sk_cols(c);
}

// Row tiles, staged tile and atom chunks of the matrix-core structure factor.
// Row tiles: kES(3) spread evenly over as few blocks of at most 7 as it needs.
// Tile and chunks: the least of a sum of what a launch waits for (us): a tile's
// staging kStage, its products (64 cycles each on a SIMD, shared by the blocks
// of a CU), kChunk a chunk for the reduction that adds them up, and for partial
// sums beyond the L2s' 32 MB their way to memory and back (kByte; 64 ions at kES
// 80, 80, 50, 21 MB a chunk: sums and reduction 141 -> 126 us; 512 at 40 101 -> 77).
static int sk_plan(mdff_ctx* c, int cus) {
  constexpr double kStage = 1.5, kChunk = 0.08, kProduct = 64.0 / 2400.0, kByte = 2.0 / 4e6, kCached = 32e6;
  const int ncol = c->K[0] + c->K[1] + c->K[2] + 3;
  c->sk_mma_ch = 1;
  if (ncol > sk_cols(c)) return MDFF_OK;          // refused at the first evaluation (sk_rt 0)
  const bool dip = c->task_qd || c->task_dd;
  const int nt = div_up(c->NZk, 8), zb = div_up(nt, 7);
  c->sk_rt = div_up(nt, zb);
  const int mblocks = div_up(div_up(c->NXk * c->NYk, 16), 4) * zb;
  double best = 0.0;
  for (int lta = 6; lta >= 3; --lta) {
    const int TA = 1 << lta;
    const size_t lds = sk_lds(ncol, TA);
    if (lds > (lta > 3 ? 65536 : 131072)) continue;
    for (int d = 0; d < 2; ++d) MDFF_TRY(allow_lds(c, sk_kernel(c->sk_rt, d), lds));
    const int64_t cap = (int64_t)cus * blocks_per_cu(sk_kernel(c->sk_rt, dip), lds);
    for (int ch = 1; ch <= 128 && (ch == 1 || div_up(c->n, ch) >= TA); ++ch) {
      const int per = div_up(c->n, ch), nch = div_up(c->n, per), tiles = div_up(per, TA);
      const int64_t blocks = (int64_t)mblocks * nch;
      const double t = (double)div_up(blocks, cap) * tiles * kStage + kChunk * nch +
                       kByte * std::max(0.0, 16.0 * c->nk_box * nch - kCached) +
                       (double)div_up(blocks, cus) * div_up(per, 8) * kSkStep * c->sk_rt * (dip ? 2 : 1) * kProduct;
      if (best == 0.0 || t < best) {
        best = t;
        c->sk_mma_ch = nch;
        c->sk_lta = lta;
      }
    }
  }
  return MDFF_OK;
}

// Whether the transforms are to hold FP64 accuracy: the FP64 form; the field
// gradient, which is FP64 in both; and of the mixed form the dipole systems that
// ask for it (MDFF_DIP_RECIP_FP64=1, read at context creation) or are large
// enough in x, y or z that the form has always summed them to FP64 rounding
// (more than 1,024 columns (nx, ny), or nz beyond 31, within |k| <= 2.5 alpha).
static bool recip_wide(const mdff_ctx* c) {
  if (c->d.precision != MDFF_PREC_MIXED || c->d.doefg) return true;
  if (!c->task_qd && !c->task_dd) return false;
  const char* ev = getenv("MDFF_DIP_RECIP_FP64");
  if (ev && ev[0] == '1') return true;
  int kin[3];
  for (int d = 0; d < 3; ++d) {
    const double* a = c->A + 3 * d;
    const double len = sqrt(a[0] * a[0] + a[1] * a[1] + a[2] * a[2]);
    kin[d] = std::min(c->K[d], (int)ceil(2.5 * c->alpha * len / (2.0 * MDFF_PI)));
  }
  return !c->task_qq || std::min({kin[0], kin[1], kin[2]}) < 1 || kin[2] > 31 || (kin[0] + 1) * (2 * kin[1] + 1) > 1024;
}

int recip_setup(mdff_ctx* c) {
  const int Kx = c->d.kES[0], Ky = c->d.kES[1], Kz = c->d.kES[2];
  c->K[0] = Kx; c->K[1] = Ky; c->K[2] = Kz;
  c->NXk = Kx + 1; c->NYk = 2 * Ky + 1; c->NZk = 2 * Kz + 1;
  c->nk_box = c->NXk * c->NYk * c->NZk;
  c->nk = Kz + Ky * (2 * Kz + 1) + Kx * (2 * Ky + 1) * (2 * Kz + 1);
  const int nb = c->nk_box;
  // The direct sums cost atoms x k vectors, the transforms some 60 us of short
  // kernels and a few us per 1,000 atoms (us a step or evaluation, direct / mesh):
  //   FP64   8e7 (silica 5,184) 160/164   1.5e8 (LiF 5,832) 157/145   1.8e8 (silica 8,232) 218/191
  //          dipoles, MgO 5,832 2662/2869   6,480 2834/2872   8,000 3379/2965
  //   mixed  5.4e7 (silica 4,320) 136/138   8e7 160/142
  //          dipoles, 4.3e7 (MgO 4,608) 1994/2407   5,832 2561/2458   8,000 3240/2898
  //   gradient  4e7 (NaCl 2,744) 162/164   9e7 (4,096) 207/184   (5,832) 320/194
  // The mixed form's narrower kernel (12 points, not 16) puts its line lower.
  // Few atoms in a large k mesh are another matter: the transforms' own work goes
  // with the mesh alone, and has to be less than what the direct sums spend on
  // atoms and k vectors (28 us a 1e8 terms, 220 us a 1e6 k vectors, fitted like
  // mesh_transform_us; FP64, us an evaluation, direct / mesh: 256 ions at kES 48
  // 247/508, 512 at 40 208/306, 128 at 200, 60, 20 341/1219, 1,728 at 28 224/183).
  // Not so for kES(3) > 56, whose direct gather is the vector-ALU one.
  {
    const char* ev = getenv("MDFF_RECIP_MESH");
    c->rec_wide = recip_wide(c) ? 1 : 0;
    const double line = c->d.doefg ? 8e7 : (c->rec_wide ? 1.1e8 : 7e7);
    const bool asked = ev && ev[0], on = asked ? ev[0] != '0' : (double)c->n * nb > line;
    const double direct_us = asked || mma_bucket(Kz + 1) == 0 ? INFINITY : 28e-8 * c->n * nb + 220e-6 * nb;
    if (on && c->use_mma && direct_takes(c)) {
      MDFF_TRY(mesh_setup(c, direct_us));
      if (c->mesh) return MDFF_OK;
    }
  }
  {
    HIP_TRY(c, hipMalloc((void**)&c->kA, sizeof(double) * nb));
    HIP_TRY(c, hipMalloc((void**)&c->kvec, sizeof(double) * 4 * (size_t)nb));
    BoxArgs a{};
    for (int d = 0; d < 3; ++d) a.K[d] = c->K[d];
    for (int k = 0; k < 9; ++k) a.b[k] = c->B[k];
    a.alpha2 = c->alpha * c->alpha;
    a.A = c->kA;
    a.kvec = c->kvec;
    hipLaunchKernelGGL(k_box_weights, dim3(div_up(nb, 256)), dim3(256), 0, c->stream, a);
    HIP_TRY(c, hipGetLastError());
  }
  const int ncol = Kx + Ky + Kz + 3;
  HIP_TRY(c, hipMalloc((void**)&c->tab, sizeof(cplx) * ncol * (size_t)c->n));
  // structure-factor chunks: enough work items to fill the GPU
  const int GZ = 8;
  const int NG = div_up(c->NZk, GZ);
  const int64_t items = (int64_t)c->NXk * c->NYk * NG;
  int chunks = (int)std::max<int64_t>(1, (int64_t)256 * 1024 * 8 / std::max<int64_t>(items, 1));
  chunks = std::min(chunks, std::max(1, c->n / 64));
  chunks = std::min(chunks, 64);
  c->sk_chunks = chunks;
  HIP_TRY(c, hipMalloc((void**)&c->wk, sizeof(double) * 2 * nb));
  // gather splits over (nx, ny): about 256k threads in flight
  const int M = c->NXk * c->NYk;
  int splits = std::max(1, std::min(M, div_up((int64_t)262144, c->n)));
  // matrix-core gather: A operand and its own split count
  c->mma_nks = mma_bucket(Kz + 1);
  c->mma_mtiles = div_up(M, 4);
  int cus = 256;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->device) != hipSuccess || cus <= 0)
    cus = 256;
  // splits over m-tiles (gather_splits), 3 and 9 moments
  for (int k = 0; k < 2; ++k) {
    const int mom = k ? 9 : 3;
    const int atom_waves = div_up(c->n, 16 * mma_ct(c->mma_nks, mom));
    const int64_t conc = 4 * (int64_t)cus * blocks_per_cu(gather_kernel(c->mma_nks, mom), 0);
    c->mma_splits[k] = gather_splits(c->mma_mtiles, atom_waves, conc, cus, std::max(c->mma_nks, 1));
  }
  MDFF_TRY(sk_plan(c, cus));
  const size_t na = (size_t)c->mma_mtiles * c->mma_nks * 64;
  HIP_TRY(c, hipMalloc((void**)&c->amat, sizeof(double) * na));
  // (on the context's stream, as the kernels: it does not wait for the null stream)
  HIP_TRY(c, hipMemsetAsync(c->amat, 0, sizeof(double) * na, c->stream));
  // block partials of the energy / stress: k-blocks of 64
  HIP_TRY(c, hipMalloc((void**)&c->rec_blk, sizeof(double) * 7 * (size_t)div_up(nb, 64)));
  HIP_TRY(c, hipMalloc((void**)&c->sk_part, sizeof(double) * 2 * (size_t)std::max(c->sk_chunks, c->sk_mma_ch) * nb));
  c->rec_splits = std::max({splits, c->mma_splits[0], c->mma_splits[1]});
  HIP_TRY(c, hipMalloc((void**)&c->rec_part, sizeof(double) * 9 * (size_t)c->rec_splits * c->n));
  return MDFF_OK;
}

void recip_free(mdff_ctx* c) {
  mesh_free(c);
  void* ps[] = {c->kA, c->kvec, c->tab, c->sk_part, c->wk, c->rec_part, c->amat, c->rec_blk};
  for (void* p : ps)
    if (p) (void)hipFree(p);
}

int recip_tables_from_r(mdff_ctx* c, bool pack) {
  if (c->mesh) return mesh_bin(c, true, pack);
  TabRArgs a{};
  a.n = c->n;
  a.Kx = c->K[0]; a.Ky = c->K[1]; a.Kz = c->K[2];
  a.rx = c->rx; a.ry = c->ry; a.rz = c->rz;
  for (int k = 0; k < 9; ++k) a.b[k] = c->B[k];
  a.sx = c->sx; a.sy = c->sy; a.sz = c->sz;
  a.tab = c->tab;
  a.pack = pack ? 1 : 0;
  a.order = c->cell_atoms;
  a.q = c->q;
  a.itype = c->itype;
  a.rec = c->arec;
  a.meta = c->ameta;
  // the previous MD step's final sums ride along as one more block row
  const int nbx = div_up(c->n, 256);
  if (c->nfin > nbx) MDFF_TRY(flush_finals(c));
  const FinalBatch fb = take_finals(c);
  const int runs = tab_runs(c->K);
  const bool extra = fb.nfin > 0 || fb.seq_out;
  PROF_LAUNCH(c, PK_TABLES,
              hipLaunchKernelGGL(k_tables_r, dim3(nbx, runs + (extra ? 1 : 0)), dim3(256), 0, c->stream, a, fb,
                                 extra ? runs : -1));
  HIP_TRY(c, hipGetLastError());
  return MDFF_OK;
}

int recip_tables(mdff_ctx* c) {
  if (c->mesh) return mesh_bin(c, false, false);
  PROF_LAUNCH(c, PK_TABLES,
              hipLaunchKernelGGL(k_tables, dim3(div_up(c->n, 256), tab_runs(c->K)), dim3(256), 0, c->stream, c->n,
                                 c->K[0], c->K[1], c->K[2], c->sx, c->sy, c->sz, c->tab));
  HIP_TRY(c, hipGetLastError());
  return MDFF_OK;
}

// the fields and forces from the moments of the splits; forces wanted with no
// output array: the caller's force kernel finishes them (c->rfin)
static int rec_finish(mdff_ctx* c, const double* part, int nsplit, int moments, const double* q, const double* mu,
                      bool use_q, bool forces, bool field, double* ef_out, double* f_out) {
  RecFinal rf{};
  rf.n = c->n;
  rf.nsplit = nsplit;
  rf.moments = moments;
  rf.use_q = use_q ? 1 : 0;
  rf.part = part;
  rf.q = q;
  rf.mu = mu;
  for (int k = 0; k < 9; ++k) rf.b[k] = c->B[k];
  rf.fpi_V = 2.0 * (2.0 * MDFF_PI / c->omega);
  const bool defer = forces && !f_out;
  if (defer) {
    c->rfin = rf;
    c->rfin_pending = 1;
  }
  if (field && !ef_out) {          // recip_moments
    c->rfin = rf;
    return MDFF_OK;
  }
  if (field || !defer)
    PROF_LAUNCH(c, PK_GFINAL,
                hipLaunchKernelGGL(k_gather_final, dim3(div_up(c->n, 256)), dim3(256), 0, c->stream, rf,
                                   field ? 1 : 0, (forces && !defer) ? 1 : 0, ef_out, f_out));
  HIP_TRY(c, hipGetLastError());
  return MDFF_OK;
}

int recip_eval(mdff_ctx* c, const double* q, const double* mu, bool use_q, bool use_mu, bool forces,
               bool field, double* ef_out, double* f_out, double* e_out) {
  // second moments: dipole forces, and the field gradient (efg.hip)
  const int moments = forces && (use_mu || c->d.doefg) ? 9 : 3;
  if (c->mesh) {
    const bool wanted = forces || field;
    const double* part = nullptr;
    MDFF_TRY(mesh_eval(c, mu, use_q, use_mu, wanted ? moments : 0, e_out, &part));
    return wanted ? rec_finish(c, part, 1, moments, q, mu, use_q, forces, field, ef_out, f_out) : MDFF_OK;
  }
  constexpr int GZ = 8;
  const int M = c->NXk * c->NYk, ncol = c->K[0] + c->K[1] + c->K[2] + 3;
  int chunks = c->sk_mma_ch;
  if (c->use_mma) {
    SmArgs sm{};
    sm.n = c->n;
    sm.Kx = c->K[0]; sm.Ky = c->K[1]; sm.Kz = c->K[2];
    sm.NY = c->NYk; sm.NZ = c->NZk; sm.M = M;
    sm.chunk = div_up(c->n, chunks);
    chunks = div_up(c->n, sm.chunk);
    sm.lta = c->sk_lta;
    sm.nk_box = c->nk_box;
    sm.q = use_q ? q : c->zeros;
    sm.mu = mu;
    for (int k = 0; k < 9; ++k) sm.b[k] = c->B[k];
    sm.tab = c->tab;
    sm.part = c->sk_part;
    if (c->sk_rt == 0) {
      c->err = "kES too large for the structure-factor kernel";
      return MDFF_ERR_UNSUPPORTED;
    }
    void* args[] = {&sm};
    PROF_LAUNCH(c, PK_SK,
                (void)hipLaunchKernel(sk_kernel(c->sk_rt, use_mu),
                                      dim3(div_up(div_up(M, 16), 4), chunks, div_up(c->NZk, 8 * c->sk_rt)), dim3(256),
                                      args, sk_lds(ncol, 1 << c->sk_lta), c->stream));
  } else {
    SkArgs s{};
    s.n = c->n;
    s.Kx = c->K[0]; s.Ky = c->K[1]; s.Kz = c->K[2];
    s.NY = c->NYk; s.NZ = c->NZk;
    s.M = M;
    s.NG = div_up(c->NZk, GZ);
    s.GZ = GZ;
    s.use_q = use_q; s.use_mu = use_mu;
    s.a0_step = div_up(c->n, c->sk_chunks);
    s.q = q; s.mu = mu;
    for (int k = 0; k < 9; ++k) s.b[k] = c->B[k];
    s.tab = c->tab;
    s.part = c->sk_part;
    s.nk_box = c->nk_box;
    // atoms per LDS tile within a 64 KiB budget
    s.TA = 32;
    while (s.TA > 1 && sk_valu_lds(ncol, s.TA) > 65536) s.TA /= 2;
    const size_t shm = sk_valu_lds(ncol, s.TA);
    if (shm > lds_limit(c)) {
      c->err = "kES too large for the structure-factor kernel";
      return MDFF_ERR_UNSUPPORTED;
    }
    MDFF_TRY(allow_lds(c, reinterpret_cast<const void*>(&k_sk<GZ>), shm));
    chunks = div_up(c->n, s.a0_step);
    const dim3 g1(div_up((int64_t)M * s.NG, 256), chunks);
    PROF_LAUNCH(c, PK_SK, hipLaunchKernelGGL(k_sk<GZ>, g1, dim3(256), shm, c->stream, s));
  }
  // the 7 energy / stress sums over the k-blocks: block partials here, the
  // final sum queued into e_out (device memory)
  const bool mma_gather = (forces || field) && c->mma_nks > 0 && c->use_mma;
  const int nb = div_up(c->nk_box, 64);
  MDFF_TRY(claim_partials(c, c->rec_blk));
  PROF_LAUNCH(c, PK_SKRED,
              hipLaunchKernelGGL(k_sk_reduce, dim3(nb), dim3(256), 0, c->stream, c->nk_box, chunks, c->sk_part, c->kA,
                                 c->kvec, c->wk, c->rec_blk, mma_gather ? c->amat : nullptr, c->NZk, c->K[2],
                                 c->mma_nks));
  if (e_out) MDFF_TRY(queue_final(c, c->rec_blk, nb, 7, e_out));
  if (!forces && !field) return MDFF_OK;
  int nsplit = 0;
  // the longest kES(3) of dipole forces is the vector-ALU gather's
  if ((!mma_gather || (forces && use_mu)) && gather_lds(c->K[2], 64) > lds_limit(c)) {
    c->err = "kES(3) too large for the reciprocal gather kernel";
    return MDFF_ERR_UNSUPPORTED;
  }
  if (mma_gather) {
    // matrix-core path (A operand written by k_sk_reduce)
    GmArgs gm{};
    gm.n = c->n;
    gm.Kx = c->K[0]; gm.Ky = c->K[1]; gm.Kz = c->K[2];
    gm.NY = c->NYk; gm.NZ = c->NZk; gm.M = M;
    gm.nks = c->mma_nks;
    gm.mtiles = c->mma_mtiles;
    gm.mt_per_split = div_up(c->mma_mtiles, c->mma_splits[moments == 9]);
    nsplit = div_up(c->mma_mtiles, gm.mt_per_split);
    gm.tab = c->tab;
    gm.amat = c->amat;
    gm.out = c->rec_part;
    void* args[] = {&gm};
    PROF_LAUNCH(c, PK_GATHER,
                (void)hipLaunchKernel(gather_kernel(gm.nks, moments),
                                      dim3(div_up(c->n, 4 * 16 * mma_ct(gm.nks, moments)), nsplit), dim3(256), args, 0,
                                      c->stream));
  } else {
    GaArgs g{};
    g.n = c->n;
    g.Kx = c->K[0]; g.Ky = c->K[1]; g.Kz = c->K[2];
    g.NY = c->NYk; g.NZ = c->NZk;
    g.M = M;
    g.m_per_split = div_up(M, c->rec_splits);
    nsplit = div_up(M, g.m_per_split);
    g.tab = c->tab;
    g.wk = c->wk;
    g.out = c->rec_part;
    // threads per block from the LDS budget (64 KiB)
    int nthr = 256;
    while (nthr > 64 && gather_lds(c->K[2], nthr) > 65536) nthr -= 64;
    const size_t shm = gather_lds(c->K[2], nthr);
    const auto fn = moments == 9 ? &k_gather<9> : &k_gather<3>;
    MDFF_TRY(allow_lds(c, reinterpret_cast<const void*>(fn), shm));
    PROF_LAUNCH(c, PK_GATHER, hipLaunchKernelGGL(fn, dim3(div_up(c->n, nthr), nsplit), dim3(nthr), shm, c->stream, g));
  }
  return rec_finish(c, c->rec_part, nsplit, moments, q, mu, use_q, forces, field, ef_out, f_out);
}

int recip_moments(mdff_ctx* c, const double* mu, RecFinal* rf) {
  MDFF_TRY(recip_eval(c, c->q, mu, false, true, false, true, nullptr, nullptr, nullptr));
  *rf = c->rfin;
  return MDFF_OK;
}
