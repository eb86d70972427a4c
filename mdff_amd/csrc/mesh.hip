// mesh.hip -- the reciprocal Ewald sums as non-uniform fast transforms in
// FP64 (gfx950).
//
// The sums are the reference's: S(k) over the whole half-space k mesh with
// its A(k) (multipole_ES_rec, src/ewald_rec.f90:38-365; mesh of
// src/kspace.f90:143-207), and per atom the sums over k of its fields and
// forces.  Evaluated term by term they cost N x nk; here each is a
// non-uniform Fourier transform to rounding accuracy, N w^3 + mesh work:
// the atoms are spread onto a regular grid with a kernel phi of w points a
// direction, the grid is transformed, and the kernel's own transform is
// divided out,
//   S(n) = sum_i a_i e^{2 pi i n.s_i} = 1/phih(n) sum_l b[l] e^{2 pi i n.l/G},
//   b[l] = sum_i a_i phi(l - G s_i),
// and the potential V(s) = Re sum_n W(n) e^{2 pi i n.s}, W = A conj(S), comes
// back the same way: sum_n n_d Im(W e_i) = -dV/ds_d / 2 pi and
// sum_n n_d n_e Re(W e_i) = -d2V/ds_d ds_e / 4 pi^2, with derivatives of phi.
// A dipole is the derivative of a charge: its amplitude i 2 pi n.m is
// m.d/ds on phi.
//
// phi(x) = s I1(beta s), s = sqrt(1 - (2x/w)^2): the Kaiser-Bessel family
// (R. M. Lewitt, J. Opt. Soc. Am. A 7, 1834 (1990)), continuous at its edge,
// which the derivatives need.  Its transform is elementary
// (2 h beta (z cosh z - sinh z) / z^3, z^2 = beta^2 - (2 pi f h)^2, h = w/2).
// The grid G and beta are chosen per direction from the alias error weighted
// with the decay of A(k) (mesh_error_above): below 4e-15 with w = 16 in the FP64
// form, which measured 1e-14 of the reciprocal force (its rounding), below
// 1e-9 with w = 12 in the mixed form, whose FP32 pair terms carry 1e-7 (16 points
// there too where recip_wide, recip.hip, asks for them).
//
// Launches of one evaluation: k_mesh_bin (s = B^T r, count per bin),
// k_mesh_scan, k_mesh_scatter, k_mesh_phi (order within the bins, phi
// values), k_mesh_spread, k_mesh_zy (z and y transforms), k_mesh_x (x
// transform, W, energy and stress, x transform back), k_mesh_yz, k_mesh_gather.
// Planes longer than LDS holds are transformed in slices (SLICED).  Every sum has
// a fixed order.  What an evaluation reads besides the atoms (weights, twiddles,
// deconvolution, A(k)) is formed on the device at creation (k_mesh_tables).
#include <algorithm>
#include <cmath>

#include "common.h"
#include "reduce.h"

namespace {

constexpr int kDeg = 15;        // degree of the piecewise polynomials of phi
constexpr int kPair = 8;        // even (odd) coefficients of a piece
constexpr int kTile = 16;       // grid points of a spread tile (and of a bin) a direction

typedef double f64x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f64x4 mma64(double a, double b, f64x4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ int div_up_dev(int a, int b) { return (a + b - 1) / b; }

// the wave's number in the block, as a scalar
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

struct MeshGrid {
  int G[3];
  int nyb, nzb;                 // bins (tiles) of y and z
};

// Grid coordinate of a fractional coordinate s: the first point l (in
// [0, G)) of the window of w points and t = l - (G s - w/2) in [0, 1).
// Rounded operation by operation, so that every kernel finds the same l.
template <int W>
__device__ __forceinline__ void mesh_coord(double s, int G, int& l, double& t) {
  const double f = s - floor(s);
  const double x = __dsub_rn(__dmul_rn(f, (double)G), 0.5 * W);
  const double c = ceil(x);
  t = c - x;
  l = 0;
  if (f >= 0.0 && f <= 1.0) {     // not NaN
    l = (int)c;
    l = l < 0 ? l + G : (l >= G ? l - G : l);
  }
}

// bin of a window start: x exactly, y and z by tiles, x fastest
__device__ __forceinline__ int mesh_bin(const MeshGrid& m, int lx, int ly, int lz) {
  return ((ly / kTile) * m.nzb + lz / kTile) * m.G[0] + lx;
}

// ---- atoms into bins -------------------------------------------------------

struct BinArgs {
  int n, from_r, pack;
  MeshGrid m;
  const double *rx, *ry, *rz;
  double b[9];                   // B column-major
  double *sx, *sy, *sz;          // written from r, or read
  int32_t* key;                  // bin of every atom
  int32_t* slot;                 // its arrival number in the bin (any order)
  int32_t* cnt;                  // atoms per bin (zero on entry)
  // pack: the atoms in the cell order of the last list build (pack_atoms)
  const int32_t* order;
  const double* q;
  const int32_t* itype;
  AtomRec* rec;
  int2* meta;
};

// One thread per atom.  fin_row >= 0: the blocks of that row run the queued
// final sums of the previous MD step (block x: sum x).  s = B^T r is rounded
// as kardir does (src/lattice.f90:183-216).
template <int W>
__global__ void __launch_bounds__(256) k_mesh_bin(BinArgs a, FinalBatch fb, int fin_row) {
  if ((int)blockIdx.y == fin_row) {
    __shared__ double sh[4 * kRedMaxCols];
    run_final_batch(fb, blockIdx.x, sh);
    return;
  }
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  const double* b = a.b;
  auto dot = [](double x, double y, double z, double u, double v, double w) {
    return __dadd_rn(__dadd_rn(__dmul_rn(x, u), __dmul_rn(y, v)), __dmul_rn(z, w));
  };
  double s0, s1, s2;
  if (a.from_r) {
    const double x = a.rx[i], y = a.ry[i], z = a.rz[i];
    s0 = dot(x, y, z, b[0], b[1], b[2]);
    s1 = dot(x, y, z, b[3], b[4], b[5]);
    s2 = dot(x, y, z, b[6], b[7], b[8]);
    a.sx[i] = s0;
    a.sy[i] = s1;
    a.sz[i] = s2;
  } else {
    s0 = a.sx[i];
    s1 = a.sy[i];
    s2 = a.sz[i];
  }
  int lx, ly, lz;
  double t;
  mesh_coord<W>(s0, a.m.G[0], lx, t);
  mesh_coord<W>(s1, a.m.G[1], ly, t);
  mesh_coord<W>(s2, a.m.G[2], lz, t);
  const int bin = mesh_bin(a.m, lx, ly, lz);
  a.key[i] = bin;
  a.slot[i] = atomicAdd(a.cnt + bin, 1);
  if (a.pack) {
    const int j = a.order[i];
    const double xj = a.rx[j], yj = a.ry[j], zj = a.rz[j];
    a.rec[i] = AtomRec{dot(xj, yj, zj, b[0], b[1], b[2]), dot(xj, yj, zj, b[3], b[4], b[5]),
                       dot(xj, yj, zj, b[6], b[7], b[8]), a.q[j]};
    a.meta[i] = make_int2(a.itype[j], j);
  }
}

// start[0..nb] = prefix sums of cnt[0..nb), one block (many bins; few: the
// scatter forms them)
__global__ void __launch_bounds__(1024) k_mesh_scan(int nb, const int32_t* __restrict__ cnt, int32_t* __restrict__ start) {
  __shared__ int ws[16];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int base = 0;
  for (int t0 = 0; t0 < nb; t0 += 4096) {
    const int k0 = t0 + 4 * threadIdx.x;
    int c[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) c[u] = k0 + u < nb ? cnt[k0 + u] : 0;
    const int mine = c[0] + c[1] + c[2] + c[3];
    int v = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int x = __shfl_up(v, o, 64);
      if (lane >= o) v += x;
    }
    if (lane == 63) ws[w] = v;
    __syncthreads();
    int before = 0, all = 0;
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      before += u < w ? ws[u] : 0;
      all += ws[u];
    }
    int at = base + before + v - mine;
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (k0 + u < nb) {
        start[k0 + u] = at;
        at += c[u];
      }
    base += all;
    __syncthreads();
  }
  if (threadIdx.x == 0) start[nb] = base;
}

__global__ void k_mesh_clear(int nb, int32_t* __restrict__ cnt) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < nb) cnt[k] = 0;
}

// an atom among those of its bin: fractional coordinates, index, bin
struct alignas(16) BinAtom {
  double x, y, z;
  int32_t i, bin;
};

struct ScatterArgs {
  int n, nb;
  const int32_t *key, *slot, *cnt;
  int32_t* start;                // prefix sums of cnt: read, or (SCAN) written
  const double *sx, *sy, *sz;
  BinAtom* order;
};

// SCAN: every block forms the prefix sums itself (a launch less: 4.5 us of a
// 24,000-ion step), 256 runs of bins, then the atom's bin within its run; block
// 0 stores them.  For up to kScanBins bins, whose counts the blocks can all
// read in the time of one launch.
constexpr int kScanBins = 8192;
template <bool SCAN>
__global__ void __launch_bounds__(256) k_mesh_scatter(ScatterArgs a) {
  __shared__ int base[257];
  __shared__ int ws[4];
  const int i = blockIdx.x * 256 + threadIdx.x;
  const int ic = min(i, a.n - 1);
  const int bin = a.key[ic], slot = a.slot[ic];
  const double x = a.sx[ic], y = a.sy[ic], z = a.sz[ic];
  int first;
  if constexpr (SCAN) {
    const int run = (a.nb + 255) / 256, k0 = threadIdx.x * run, k1 = min(a.nb, k0 + run);
    int mine = 0;
#pragma unroll 8
    for (int k = k0; k < k1; ++k) mine += a.cnt[k];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int v = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(v, o, 64);
      if (lane >= o) v += t;
    }
    if (lane == 63) ws[w] = v;
    __syncthreads();
    int before = v - mine;
    for (int u = 0; u < w; ++u) before += ws[u];
    base[threadIdx.x] = before;
    __syncthreads();
    const int r0 = bin / run;
    first = base[r0];
#pragma unroll 8
    for (int k = r0 * run; k < bin; ++k) first += a.cnt[k];
    if (blockIdx.x == 0) {
      int at = before;
      for (int k = k0; k < k1; ++k) {
        a.start[k] = at;
        at += a.cnt[k];
      }
      if (threadIdx.x == 0) a.start[a.nb] = a.n;
    }
  } else {
    first = a.start[bin];
  }
  if (i < a.n) a.order[first + slot] = BinAtom{x, y, z, i, bin};
}

struct PhiArgs {
  int n;
  MeshGrid m;
  const BinAtom* order;
  const int32_t* start;
  int32_t* cnt;                  // the bins' counts, cleared for the next evaluation
  int nb;
  const double* q;
  const double* coef;            // [W/2][2][kPair] pieces of phi, even and odd coefficients
  int4* at;                      // per sorted atom: window start (x, y, z), atom index
  double4* vt;                   // v = 2t - 1 of x, y, z, charge
  double* phi;                   // [atom][3][W], with dip [atom][6][W]: phi, then dphi/dv
};

// Sixteen lanes an atom.  Its place within the bin is the number of smaller
// indices there (the arrival order is not reproducible); then lane j
// evaluates window point j of each direction.  Piece W-1-j mirrors piece j
// (phi is even), so the upper lanes take the lower pieces at -v; the
// coefficients of a lane's piece stay in registers over the atoms.
template <int W>
__device__ __forceinline__ void load_piece(const double* coef, int j, double c[2 * kPair]) {
  const int jj = j < W / 2 ? j : W - 1 - j;
#pragma unroll
  for (int k = 0; k < 2 * kPair; ++k) c[k] = j < W ? coef[jj * 2 * kPair + k] : 0.0;
}

// E(v^2) + v O(v^2) at v (v times sg for a mirrored piece), its first
// derivative in v and, SECOND, its second
template <bool FIRST, bool SECOND>
__device__ __forceinline__ void piece(const double c[2 * kPair], double v, double sg, double& f, double& df,
                                      double& d2) {
  v *= sg;
  const double v2 = v * v;
  double e = c[kPair - 1], h = c[2 * kPair - 1], de = 0.0, dh = 0.0, ee = 0.0, hh = 0.0;
#pragma unroll
  for (int k = kPair - 2; k >= 0; --k) {
    if (SECOND) {
      ee = ee * v2 + de;
      hh = hh * v2 + dh;
    }
    if (FIRST) {
      de = de * v2 + e;
      dh = dh * v2 + h;
    }
    e = e * v2 + c[k];
    h = h * v2 + c[kPair + k];
  }
  f = e + v * h;
  if (FIRST) df = sg * (2.0 * v * de + h + 2.0 * v2 * dh);
  // ee, hh: half the second derivatives of E and O in v^2
  if (SECOND) d2 = 2.0 * de + 8.0 * v2 * ee + v * (6.0 * dh + 8.0 * v2 * hh);
}

template <int W, bool DIP>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(DIP ? 4 : 6))) k_mesh_phi(PhiArgs a) {
  constexpr int NR = DIP ? 6 : 3;
  const int j = threadIdx.x & 15, step = gridDim.x * 16;
  double c[2 * kPair];
  load_piece<W>(a.coef, j, c);
  const double sg = j < W / 2 ? 1.0 : -1.0;
  for (int k = blockIdx.x * 256 + threadIdx.x; k < a.nb; k += gridDim.x * 256) a.cnt[k] = 0;
  for (int p0 = blockIdx.x * 16 + (threadIdx.x >> 4); p0 < a.n; p0 += step) {
    const BinAtom me = a.order[p0];
    const int i = me.i;
    const double s[3] = {me.x, me.y, me.z}, qi = a.q[i];
    const int b0 = a.start[me.bin], b1 = a.start[me.bin + 1];
    int rank = 0;
    for (int k = b0 + j; k < b1; k += 16) rank += a.order[k].i < i ? 1 : 0;
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) rank += __shfl_xor(rank, o, 16);
    const size_t p = (size_t)b0 + rank;
    double* out = a.phi + p * (NR * W) + j;
    int l[3];
    double v[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      double t, f, df = 0.0, d2 = 0.0;
      mesh_coord<W>(s[d], a.m.G[d], l[d], t);
      v[d] = 2.0 * t - 1.0;
      piece<DIP, false>(c, v[d], sg, f, df, d2);
      if (j < W) {
        out[d * W] = f;
        if (DIP) out[(3 + d) * W] = df;
      }
    }
    if (j == 0) {
      a.at[p] = make_int4(l[0], l[1], l[2], i);
      a.vt[p] = make_double4(v[0], v[1], v[2], qi);
    }
  }
}

// charge and -2 G m (m = B^T mu) of every sorted atom: the amplitudes of phi
// and of its derivatives dphi/ds_d = -2 G_d dphi/dv
__global__ void __launch_bounds__(256) k_mesh_amp(int n, const int4* __restrict__ at, const double* __restrict__ q,
                                                  int use_q, const double* __restrict__ mu, double b0, double b1,
                                                  double b2, double b3, double b4, double b5, double b6, double b7,
                                                  double b8, double gx, double gy, double gz, double4* __restrict__ amp) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const int i = at[p].w;
  const double u0 = mu[3 * i], u1 = mu[3 * i + 1], u2 = mu[3 * i + 2];
  amp[p] = make_double4(use_q ? q[i] : 0.0, gx * (u0 * b0 + u1 * b1 + u2 * b2), gy * (u0 * b3 + u1 * b4 + u2 * b5),
                        gz * (u0 * b6 + u1 * b7 + u2 * b8));
}

// ---- spread ------------------------------------------------------------------
// One block per tile of 16^3 grid points (and share of the bin columns), one
// wave per x plane of the tile.  The atoms whose window touches the tile are
// in the four bin columns (its y and z tile and the ones before them), lx from
// x0 - W + 1 to x0 + 15: x is the fastest index of the bins, so each column
// has one contiguous range of atoms (two where x wraps).  A chunk of them
// enters LDS as rows of 16 already in the tile's coordinates, zero outside
// the window: four atoms a step then cost two reads of 16 values, one product
// and one v_mfma_f64_16x16x4, D(y, z) += [q phi(x) phi(y)] phi(z).  A wave
// takes the steps of its own plane's range.  The windows' zeros in y and z are
// multiplied along (W/32 of each direction is used); no atomics, fixed order.
struct SpreadArgs {
  int n, shares, pstride;        // pstride: doubles per atom of phi
  MeshGrid m;
  const int32_t* start;
  const int4* at;
  const double4* vt;             // .w: charge (without dipoles)
  const double* phi;
  const double4* amp;            // with dipoles
  double* out;                   // [share][Gx][Gy][Gz]
};

template <int W, bool DIP>
__global__ void __launch_bounds__(1024) k_mesh_spread(SpreadArgs a) {
  constexpr int U = DIP ? 1 : 2;                          // staging passes of a chunk
  constexpr int NA = 64 * U;                              // atoms of a chunk
  constexpr int NR = DIP ? 2 : 1;
  // per atom: y and z rows (phi, and for dipoles m phi'), and by x plane q phi
  // (+ m phi') and, for dipoles, phi (padded against bank conflicts)
  __shared__ double ry[NR][NA + 16][kTile], rz[NR][NA + 16][kTile], rx[NR][kTile][NA + 18];
  const int Gx = a.m.G[0], Gy = a.m.G[1], Gz = a.m.G[2];
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15, grp = threadIdx.x >> 4;
  const int wave = wave_id();
  // tiles x fastest, in XCD order: an XCD's tiles share bin columns
  const int ntx = Gx / kTile;
  const int lin = xcd_order(blockIdx.x, (int)gridDim.x);
  const int tx = lin % ntx, share = (lin / ntx) % a.shares, yz = lin / (ntx * a.shares);
  const int tz = yz % a.m.nzb, ty = yz / a.m.nzb;
  const int x0 = kTile * tx, x = x0 + wave;
  f64x4 acc = {0.0, 0.0, 0.0, 0.0};
  for (int col = share; col < 4; col += a.shares) {
    if (((col & 1) && a.m.nyb == 1) || ((col & 2) && a.m.nzb == 1)) continue;
    int by = ty - (col & 1), bz = tz - (col >> 1);
    by = by < 0 ? by + a.m.nyb : by;
    bz = bz < 0 ? bz + a.m.nzb : bz;
    // the window's offset in the tile: its own column, or the one before (a
    // single tile wraps onto itself: both, from one column)
    const int oy = c + ((col & 1) ? kTile : 0), oz = c + ((col & 2) ? kTile : 0);
    const bool wy = a.m.nyb == 1, wz = a.m.nzb == 1;
    const int32_t* st = a.start + (size_t)(by * a.m.nzb + bz) * Gx;
    // lx in [x0 - W + 1, x0 + 15]; below zero they are at the other end of
    // the row, from x0 + 16 at the earliest (part 1)
    for (int part = 0; part < 2; ++part) {
      const int lo = x0 - W + 1;
      if (part == 1 && lo >= 0) break;
      const int f0 = part == 0 ? max(lo, 0) : max(Gx + lo, x0 + kTile), f1 = part == 0 ? x0 + kTile : Gx;
      // the wave's own starts in this part
      const int wl = x - W + 1 + (part == 0 ? 0 : Gx);
      const int w0 = max(wl, f0), w1 = part == 0 ? x + 1 : Gx;
      const int q0 = st[f0], q1 = st[f1];
      if (q0 >= q1) continue;
      // (a grid of one tile wraps onto itself: every atom, for every plane)
      const bool whole = Gx == kTile;
      const int own0 = whole ? q0 : (w0 < w1 ? st[w0] : 0), own1 = whole ? q1 : (w0 < w1 ? st[w1] : 0);
      const int ox = x0 + c + (part == 0 ? 0 : Gx);
      // the next chunk's atoms and the chunk after's places are on their way
      // while a chunk is summed
      double vx[NR][U], vy[NR][U], vz[NR][U];
      int4 at[U];
      auto load_at = [&](int p0) {
#pragma unroll
        for (int u = 0; u < U; ++u) at[u] = a.at[min(p0 + grp + 64 * u, q1 - 1)];
      };
      auto load_phi = [&](int p0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int p = p0 + grp + 64 * u, pc = min(p, q1 - 1);
          const double* f = a.phi + (size_t)pc * a.pstride;
          int dx = ox - at[u].x, dy = oy - (at[u].y & (kTile - 1)), dz = oz - (at[u].z & (kTile - 1));
          if (whole) dx &= kTile - 1;
          if (wy) dy &= kTile - 1;
          if (wz) dz &= kTile - 1;
          const bool okx = p < q1 && (unsigned)dx < (unsigned)W, oky = (unsigned)dy < (unsigned)W,
                     okz = (unsigned)dz < (unsigned)W;
          const unsigned ux = min((unsigned)dx, W - 1u), uy = min((unsigned)dy, W - 1u), uz = min((unsigned)dz, W - 1u);
          const double fx = f[ux], fy = f[W + uy], fz = f[2 * W + uz];
          if constexpr (DIP) {
            const double4 m = a.amp[pc];
            const double gx = f[3 * W + ux], gy = f[4 * W + uy], gz = f[5 * W + uz];
            vx[0][u] = okx ? m.x * fx + m.y * gx : 0.0;
            vx[1][u] = okx ? fx : 0.0;
            vy[1][u] = oky ? m.z * gy : 0.0;
            vz[1][u] = okz ? m.w * gz : 0.0;
          } else {
            vx[0][u] = okx ? a.vt[pc].w * fx : 0.0;
          }
          vy[0][u] = oky ? fy : 0.0;
          vz[0][u] = okz ? fz : 0.0;
        }
      };
      load_at(q0);
      load_phi(q0);
      load_at(q0 + NA);
      for (int p0 = q0; p0 < q1; p0 += NA) {
        __syncthreads();
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int r = 0; r < NR; ++r) {
            rx[r][c][grp + 64 * u] = vx[r][u];
            ry[r][grp + 64 * u][c] = vy[r][u];
            rz[r][grp + 64 * u][c] = vz[r][u];
          }
        __syncthreads();
        if (p0 + NA < q1) {
          load_phi(p0 + NA);
          load_at(p0 + 2 * NA);
        }
        const int s0 = max(own0 - p0, 0) >> 2, s1 = (min(own1 - p0, NA) + 3) >> 2;
        const double* px = &rx[0][wave][g];
        const double* py = &ry[0][g][c];
        const double* pz = &rz[0][g][c];
        constexpr int SX = kTile * (NA + 18), SY = (NA + 16) * kTile;   // to the second row set
        for (int t = s0; t < s1; t += 4) {
          double av[4], bv[4], cv[4], dv[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const double ax = px[4 * (t + u)], ay = py[64 * (t + u)];
            bv[u] = pz[64 * (t + u)];
            if constexpr (DIP) {
              const double cx = px[SX + 4 * (t + u)];
              av[u] = ax * ay + cx * py[SY + 64 * (t + u)];
              cv[u] = cx * ay;
              dv[u] = pz[SY + 64 * (t + u)];
            } else {
              av[u] = ax * ay;
            }
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            if (t + u >= s1) break;
            acc = mma64(av[u], bv[u], acc);
            if constexpr (DIP) acc = mma64(cv[u], dv[u], acc);
          }
        }
      }
    }
  }
  double* o = a.out + (((size_t)share * Gx + x) * Gy + kTile * ty) * Gz + kTile * tz + c;
#pragma unroll
  for (int r = 0; r < 4; ++r) o[(size_t)(4 * r + g) * Gz] = acc[r];
}

// ---- transforms --------------------------------------------------------------
// Each direction is a product with its Fourier matrix on
// v_mfma_f64_16x16x4 (the matrices carry 1 / phih).  A block takes one x
// plane (k_mesh_zy, k_mesh_yz) or 16 columns (k_mesh_x) through two
// transforms with the data between them in LDS.  The matrices are stored in
// the order of the instruction's operands:
//  - "row" products (real: z), out[row][col] = sum_k in[row][k] M[k][col]: M as
//    [k / 16][column tile][step][lane]; lane group g takes k = 16 kc + 4 g +
//    step, so its four values of in are consecutive;
//  - "mid" products (complex: x, y), out[n][c] = sum_l E[n][l] in[l][c]: E as
//    [l / 4][n tile of 8][re in, im in][lane]; tile row R holds n = 4 (R >> 3)
//    + (R & 3) and part (R >> 2) & 1, so a lane ends with re and im of its two
//    n.  The re and im inputs go to neighbouring waves, which halves the chain
//    of a wave; their sums meet in LDS.
// The rows that a product sums over are staged all at once where they fit the
// block's LDS, else (Gy or Gx + NX beyond 576: LiF of 53 cells and more in a
// row) a slice of them at a time: the sums of the slices before are read back by
// the threads that wrote them (y and x forward, x back) or kept in registers (y
// back).  The direct sums, the alternative, took 2960 us for LiF 66 x 8 x 8
// (33,792 ions, mixed) and 10.06 s for 46^3 (778,688); in slices 541 us and 10 ms.
constexpr int kFtThreads = 1024, kFtWaves = 16;

// acc + the tile's operand (e, es doubles between steps of 4 l) times the LDS
// rows v over L (operand and rows up to the next 16)
__device__ __forceinline__ f64x4 mid_chain(const double* e, size_t es, const double* v, int L, f64x4 acc) {
  for (int l = 0; l < L; l += 16) {
    double ev[4], vv[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      ev[u] = e[(size_t)(l / 4 + u) * es];
      vv[u] = v[(size_t)(l + 4 * u) * 16];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) acc = mma64(ev[u], vv[u], acc);
  }
  return acc;
}

// in: LDS planes [re, im][l][16], rows up to the next 16 finite; out(n, c, value)
template <typename Out>
__device__ __forceinline__ void mid_product(const double* in, int lrows, int L, int ntiles, int N, const double* E,
                                            double* xb, Out out) {
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15, wave = wave_id();
  const int sp = wave & 1;
  const double* v = in + (size_t)sp * lrows * 16 + 16 * g + c;
  double* x = xb + (wave >> 1) * 256 + lane;
  for (int t0 = 0; t0 < ntiles; t0 += kFtWaves / 2) {
    const int t = t0 + (wave >> 1);
    f64x4 acc = {0.0, 0.0, 0.0, 0.0};
    if (t < ntiles) acc = mid_chain(E + ((size_t)t * 2 + sp) * 64 + lane, (size_t)ntiles * 128, v, L, acc);
    if (sp == 1) {
#pragma unroll
      for (int r = 0; r < 4; ++r) x[64 * r] = acc[r];
    }
    __syncthreads();
    if (sp == 0 && t < ntiles) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int n = 8 * t + 4 * h + g;
        if (n < N) out(n, c, acc[2 * h] + x[128 * h], acc[2 * h + 1] + x[128 * h + 64]);
      }
    }
    __syncthreads();
  }
}

struct ZyArgs {
  int Gy, Gz, CN, NY, ctiles;
  int slice;                     // SLICED: y rows in LDS (a multiple of 16)
  size_t sstride;                // between the shares of the grid, which are added
  const double* grid;
  const double* zf;              // row operand: column tile 2 ct + part
  const double* yf;
  double2* out;                  // [x][ny][nz]
};

// Block (nz tile, x): z transform of the plane's rows at 16 nz into LDS, then
// their y transform.  SH: shares of the grid
template <int SH, bool SLICED>
__global__ void __launch_bounds__(kFtThreads) k_mesh_zy(ZyArgs a) {
  extern __shared__ double lds[];
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15, wave = wave_id();
  const int ct = blockIdx.x, x = blockIdx.y;
  const int slice = SLICED ? a.slice : a.Gy;
  double* pl = lds;                                       // [part][slice][16]
  double* xb = lds + 2 * (size_t)slice * 16;
  double2* out = a.out + (size_t)x * a.NY * a.CN;
  const int cc = 16 * ct + c, ntiles = div_up_dev(a.NY, 8);
  int y0 = 0;
  do {
    const int ny = SLICED ? min(slice, a.Gy - y0) : a.Gy;
    for (int u = wave; u < ny / 8; u += kFtWaves) {
      const int rt = u >> 1, part = u & 1;
      const double* in = a.grid + ((size_t)x * a.Gy + y0 + 16 * rt + c) * a.Gz + 4 * g;
      const double* m = a.zf + ((size_t)2 * ct + part) * 256 + lane;
      f64x4 acc = {0.0, 0.0, 0.0, 0.0};
      for (int k0 = 0; k0 < a.Gz; k0 += 32) {
        // the second of the two steps repeats a valid one when Gz ends before it
        const int kk[2] = {k0, min(k0 + 16, a.Gz - 16)};
        double2 v[2][SH][2];
        double b[2][4];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
          for (int s = 0; s < SH; ++s) {
            v[h][s][0] = *reinterpret_cast<const double2*>(in + s * a.sstride + kk[h]);
            v[h][s][1] = *reinterpret_cast<const double2*>(in + s * a.sstride + kk[h] + 2);
          }
#pragma unroll
          for (int s = 0; s < 4; ++s) b[h][s] = m[(size_t)(kk[h] / 16) * a.ctiles * 512 + 64 * s];
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          if (h == 1 && k0 + 16 >= a.Gz) break;
          double2 v0 = v[h][0][0], v1 = v[h][0][1];
#pragma unroll
          for (int s = 1; s < SH; ++s) {
            v0.x += v[h][s][0].x; v0.y += v[h][s][0].y;
            v1.x += v[h][s][1].x; v1.y += v[h][s][1].y;
          }
          acc = mma64(v0.x, b[h][0], acc);
          acc = mma64(v0.y, b[h][1], acc);
          acc = mma64(v1.x, b[h][2], acc);
          acc = mma64(v1.y, b[h][3], acc);
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) pl[((size_t)part * slice + 16 * rt + 4 * r + g) * 16 + c] = acc[r];
    }
    __syncthreads();
    mid_product(pl, slice, ny, ntiles, a.NY, a.yf + (size_t)(y0 / 4) * ntiles * 128, xb,
                [&](int n, int, double re, double im) {
                  if (cc >= a.CN) return;
                  double2* o = out + (size_t)n * a.CN + cc;
                  *o = SLICED && y0 > 0 ? make_double2(o->x + re, o->y + im) : make_double2(re, im);
                });
  } while (SLICED && (y0 += slice) < a.Gy);
}

struct XArgs {
  int Gx, NX, C, back;           // C = NY CN columns
  int slice;                     // SLICED: rows in LDS (a multiple of 16)
  double2* s;                    // SLICED: S, then W, [nx][C]
  const double* xf;
  const double* xb;
  double2* t;                    // [x][C], in place
  const double* A;               // [nx][C]
  const double* kvec;            // kx, ky, kz, kcoe per (nx, c)
  double* blk;                   // 7 per block
};

// Block: 16 columns (ny, nz).  S(n); W = A conj(S); the energy and stress
// partials ((delta_ab - kcoe k_a k_b) A |S|^2, src/ewald_rec.f90:173-174,
// 252-263); W's x transform back in place (back).  S and W stay in LDS, or
// (SLICED) in global memory.
template <bool SLICED>
__global__ void __launch_bounds__(kFtThreads) k_mesh_x(XArgs a) {
  extern __shared__ double lds[];
  const int lane = threadIdx.x & 63, wave = wave_id(), c = lane & 15;
  const int nxp = (a.NX + 15) & ~15, ntiles = div_up_dev(a.NX, 8);
  const int rows = SLICED ? a.slice : a.Gx;
  double* pl = lds;                                       // [part][rows][16]
  double* wl = pl + 2 * (size_t)rows * 16;                // [part][nxp][16]
  double* xb = wl + (SLICED ? 0 : 2 * (size_t)nxp * 16);
  const int c0 = blockIdx.x * 16, cc = c0 + c;
  // rows from..from + cnt of src into LDS, zero beyond cnt up to the next 16
  auto stage = [&](const double2* src, int from, int cnt) {
    for (int k = threadIdx.x; k < ((cnt + 15) & ~15) * 16; k += kFtThreads) {
      double2 v = src[(size_t)(from + min(k >> 4, cnt - 1)) * a.C + min(c0 + (k & 15), a.C - 1)];
      if ((k >> 4) >= cnt) v = make_double2(0.0, 0.0);
      pl[k] = v.x;
      pl[(size_t)rows * 16 + k] = v.y;
    }
  };
  if constexpr (!SLICED)
    for (int k = a.NX * 16 + threadIdx.x; k < nxp * 16; k += kFtThreads) {
      wl[k] = 0.0;
      wl[(size_t)nxp * 16 + k] = 0.0;
    }
  double sum[7] = {0, 0, 0, 0, 0, 0, 0};
  // A conj(S) of entry (n, cc), and its part of the sums
  auto weigh = [&](int n, double re, double im) {
    const size_t at = (size_t)n * a.C + cc;
    const double Ak = a.A[at];
    const double* k = a.kvec + 4 * at;
    const double str = (re * re + im * im) * Ak;
    const double kx = k[0], ky = k[1], kz = k[2], kc = k[3];
    sum[0] += str;
    sum[1] += (1.0 - kc * kx * kx) * str;
    sum[2] += (1.0 - kc * ky * ky) * str;
    sum[3] += (1.0 - kc * kz * kz) * str;
    sum[4] += -kc * kx * ky * str;
    sum[5] += -kc * kx * kz * str;
    sum[6] += -kc * ky * kz * str;
    return make_double2(Ak * re, -Ak * im);
  };
  int g0 = 0;
  do {
    const int cnt = SLICED ? min(rows, a.Gx - g0) : a.Gx;
    stage(a.t, g0, cnt);
    __syncthreads();
    mid_product(pl, rows, cnt, ntiles, a.NX, a.xf + (size_t)(g0 / 4) * ntiles * 128, xb,
                [&](int n, int, double re, double im) {
                  if constexpr (SLICED) {
                    if (cc >= a.C) return;
                    double2* o = a.s + (size_t)n * a.C + cc;
                    if (g0 > 0) {
                      re += o->x;
                      im += o->y;
                    }
                    *o = g0 + rows < a.Gx ? make_double2(re, im) : weigh(n, re, im);
                  } else {
                    double2 w = {0.0, 0.0};
                    if (cc < a.C) w = weigh(n, re, im);
                    wl[n * 16 + c] = w.x;
                    wl[(size_t)nxp * 16 + n * 16 + c] = w.y;
                  }
                });
  } while (SLICED && (g0 += rows) < a.Gx);
  // wave sums, then the waves in order
#pragma unroll
  for (int k = 0; k < 7; ++k) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sum[k] += __shfl_down(sum[k], o, 64);
    if (lane == 0) xb[wave * 8 + k] = sum[k];
  }
  __syncthreads();
  if (threadIdx.x < 7) {
    double r = 0.0;
    for (int w = 0; w < kFtWaves; ++w) r += xb[w * 8 + threadIdx.x];
    a.blk[(size_t)blockIdx.x * 7 + threadIdx.x] = r;
  }
  if (!a.back) return;
  __syncthreads();
  if constexpr (SLICED) {
    for (int n0 = 0; n0 < a.NX; n0 += rows) {
      const int cnt = min(rows, a.NX - n0);
      stage(a.s, n0, cnt);
      __syncthreads();
      mid_product(pl, rows, cnt, a.Gx / 8, a.Gx, a.xb + (size_t)(n0 / 4) * (a.Gx / 8) * 128, xb,
                  [&](int n, int, double re, double im) {
                    if (cc >= a.C) return;
                    double2* o = a.t + (size_t)n * a.C + cc;
                    *o = n0 > 0 ? make_double2(o->x + re, o->y + im) : make_double2(re, im);
                  });
    }
  } else {
    mid_product(wl, nxp, a.NX, a.Gx / 8, a.Gx, a.xb, xb, [&](int n, int, double re, double im) {
      if (cc < a.C) a.t[(size_t)n * a.C + cc] = make_double2(re, im);
    });
  }
}

constexpr int kYzRows = 32;      // y rows of a k_mesh_yz block

struct YzArgs {
  int Gy, Gz, CN, NY, ctiles, ld;
  int slice;                     // SLICED: ny rows in LDS (a multiple of 16)
  const double2* in;             // [x][ny][nz]
  const double* yb;
  const double* zb;
  double* grid;
};

// Block (32 y, x): y transform back of those rows, 16 nz at a time, into LDS
// rows of (nz, re / im), then their z transform back
template <bool SLICED>
__global__ void __launch_bounds__(kFtThreads) k_mesh_yz(YzArgs a) {
  extern __shared__ double lds[];
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15, wave = wave_id();
  const int y0 = blockIdx.x * kYzRows, x = blockIdx.y;
  const int nyp = SLICED ? a.slice : (a.NY + 15) & ~15;
  const int ny = min(kYzRows, a.Gy - y0);
  double* rows = lds;                                     // [kYzRows][ld]
  double* pl = rows + (size_t)kYzRows * a.ld;             // [nz tile][part][nyp][16]
  double* xb = pl + 4 * (size_t)nyp * 16;
  const double2* in = a.in + (size_t)x * a.NY * a.CN;
  // the whole y operand has Gy / 8 tiles a step; this block's start at y0 / 8.
  // Two nz tiles at a time, eight waves each: (n tile, re / im input)
  const int sp = wave & 1, t = (wave >> 1) & 3, half = wave >> 3;
  double* xw = xb + (wave >> 1) * 256 + lane;
  for (int ct0 = 0; ct0 < a.ctiles; ct0 += 2) {
    const int nct = min(2, a.ctiles - ct0);
    f64x4 acc = {0.0, 0.0, 0.0, 0.0};
    const bool on = 8 * t < ny && half < nct;
    int l0 = 0;
    do {
      for (int k = threadIdx.x; k < nct * nyp * 16; k += kFtThreads) {
        const int h = k >= nyp * 16 ? 1 : 0, kk = k - h * nyp * 16;
        const int cc = 16 * (ct0 + h) + (kk & 15), l = l0 + (kk >> 4);
        double2 v = in[(size_t)min(l, a.NY - 1) * a.CN + min(cc, a.CN - 1)];
        if (l >= a.NY || cc >= a.CN) v = make_double2(0.0, 0.0);
        pl[(size_t)(2 * h) * nyp * 16 + kk] = v.x;
        pl[(size_t)(2 * h + 1) * nyp * 16 + kk] = v.y;
      }
      __syncthreads();
      if (on)
        acc = mid_chain(a.yb + (size_t)(l0 / 4) * (a.Gy / 8) * 128 + ((size_t)(y0 / 8 + t) * 2 + sp) * 64 + lane,
                        (size_t)(a.Gy / 8) * 128, pl + (size_t)(2 * half + sp) * nyp * 16 + 16 * g + c,
                        SLICED ? min(nyp, a.NY - l0) : a.NY, acc);
      if (SLICED && l0 + nyp < a.NY) __syncthreads();
    } while (SLICED && (l0 += nyp) < a.NY);
    if (on && sp == 1) {
#pragma unroll
      for (int r = 0; r < 4; ++r) xw[64 * r] = acc[r];
    }
    __syncthreads();
    if (sp == 0 && on) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        double* o = rows + (size_t)(8 * t + 4 * h + g) * a.ld + 2 * (16 * (ct0 + half) + c);
        o[0] = acc[2 * h] + xw[128 * h];
        o[1] = acc[2 * h + 1] + xw[128 * h + 64];
      }
    }
    __syncthreads();
  }
  const int ztiles = a.Gz / 16, units = (ny / 16) * ztiles;
  for (int u = wave; u < units; u += kFtWaves) {
    const int rt = u / ztiles, zt = u - rt * ztiles;
    const double* r = rows + (size_t)(16 * rt + c) * a.ld + 4 * g;
    const double* m = a.zb + (size_t)zt * 256 + lane;
    f64x4 acc = {0.0, 0.0, 0.0, 0.0};
    for (int k0 = 0; k0 < 32 * a.ctiles; k0 += 32) {
      double b[8], v[8];
#pragma unroll
      for (int s = 0; s < 8; ++s) b[s] = m[(size_t)(k0 / 16 + (s >> 2)) * ztiles * 256 + 64 * (s & 3)];
#pragma unroll
      for (int s = 0; s < 8; ++s) v[s] = r[k0 + 16 * (s >> 2) + (s & 3)];
#pragma unroll
      for (int s = 0; s < 8; ++s) acc = mma64(v[s], b[s], acc);
    }
    double* o = a.grid + ((size_t)x * a.Gy + y0 + 16 * rt) * a.Gz + 16 * zt + c;
#pragma unroll
    for (int q = 0; q < 4; ++q) o[(size_t)(4 * q + g) * a.Gz] = acc[q];
  }
}

// ---- gather -------------------------------------------------------------------
// V's derivatives at the atoms.  One block per bin column (y tile, z tile) and
// run of X window starts; the grid planes that its atoms' windows touch pass
// through LDS kPlanes at a time, sixteen lanes an atom, lane = z point of the
// window, so a group's reads are consecutive.  Each value serves phi and
// dphi/dv of y, which lane j holds for row j and broadcasts within its row of
// 16 lanes; x is applied per plane, z at the end.
constexpr int kGatherThreads = 512;
constexpr int kGatherAtoms = 2;  // atoms of a group in flight

struct GatherArgs {
  int n, X;
  MeshGrid m;
  const int32_t* start;
  const int4* at;
  const double4* vt;
  const double* coef;
  const double* grid;
  double* out;                   // [moments][n] by atom index
};

// t += sum over the window rows k of f(lane k of the row of 16 lanes) v[k], and
// u with d: the broadcast is part of the multiply.  The wait states that it
// needs after a write of f's or d's register are in the string.
__device__ __forceinline__ void fma_rows12(const double* v, double f, double d, double& t, double& u) {
  asm("s_nop 1\n\t"
      "v_fmac_f64_dpp %0, %2, %4 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %4 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %5 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %5 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %6 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %6 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %7 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %7 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %8 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %8 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %9 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %9 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %10 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %10 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %11 row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %11 row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %12 row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %12 row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %13 row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %13 row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %14 row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %14 row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %15 row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %15 row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
      : "+v"(t), "+v"(u)
      : "v"(f), "v"(d), "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "v"(v[4]), "v"(v[5]), "v"(v[6]), "v"(v[7]), "v"(v[8]), "v"(v[9]), "v"(v[10]), "v"(v[11]));
}
__device__ __forceinline__ void fma_rows16(const double* v, double f, double d, double& t, double& u) {
  asm("s_nop 1\n\t"
      "v_fmac_f64_dpp %0, %2, %4 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %4 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %5 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %5 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %6 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %6 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %7 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %7 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %8 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %8 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %9 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %9 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %10 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %10 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %11 row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %11 row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %12 row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %12 row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %13 row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %13 row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %14 row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %14 row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %15 row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %15 row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %16 row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %16 row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %17 row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %17 row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %18 row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %18 row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %19 row_newbcast:15 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %19 row_newbcast:15 row_mask:0xf bank_mask:0xf\n\t"
      : "+v"(t), "+v"(u)
      : "v"(f), "v"(d), "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "v"(v[4]), "v"(v[5]), "v"(v[6]), "v"(v[7]), "v"(v[8]), "v"(v[9]), "v"(v[10]), "v"(v[11]), "v"(v[12]), "v"(v[13]), "v"(v[14]), "v"(v[15]));
}

// sums over the W window rows of a plane: phi, dphi/dv and (SECOND)
// d2phi/dv2 of y times the plane's values at the lane's z
template <int W, int RZ, bool SECOND>
__device__ __forceinline__ void row_sums(const double* p, double f, double d, double dd, double& t0, double& t1,
                                         double& t2) {
  double v[W], unused = 0.0;
#pragma unroll
  for (int k = 0; k < W; ++k) v[k] = p[k * RZ];
  if constexpr (W == 16) {
    fma_rows16(v, f, d, t0, t1);
    if constexpr (SECOND) fma_rows16(v, dd, dd, t2, unused);
  } else {
    fma_rows12(v, f, d, t0, t1);
    if constexpr (SECOND) fma_rows12(v, dd, dd, t2, unused);
  }
}

constexpr int kPlanes = 8;       // staged planes

template <int W, int MOM>
__global__ void __launch_bounds__(kGatherThreads) __attribute__((amdgpu_waves_per_eu(MOM == 9 ? 2 : 4)))
k_mesh_gather(GatherArgs a) {
  constexpr bool SECOND = MOM == 9;
  constexpr int RY = kTile + W - 1, RZ = kTile + W;       // rows and padded row length of a staged plane
  constexpr int GRP = kGatherThreads / 16, NS = GRP * kGatherAtoms;
  __shared__ double plane[kPlanes * RY * RZ];
  __shared__ double px[NS][W][SECOND ? 4 : 2];            // phi, dphi/dv (, d2phi/dv2) of x per atom in flight
  const int Gx = a.m.G[0], Gy = a.m.G[1], Gz = a.m.G[2];
  // x runs fastest, in XCD order: an XCD's blocks share bin columns and planes
  const int lin = xcd_order(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
  const int col = lin / (int)gridDim.x, x0 = (lin % (int)gridDim.x) * a.X, x1 = min(Gx, x0 + a.X);
  const int ty = col / a.m.nzb, tz = col % a.m.nzb;
  const int32_t* st = a.start + (size_t)col * Gx;
  const int p0 = st[x0], p1 = st[x1];
  if (p0 >= p1) return;
  const int grp = threadIdx.x >> 4, j = threadIdx.x & 15;
  const double sg = j < W / 2 ? 1.0 : -1.0;
  const double fx = (double)Gx / MDFF_PI, fy = (double)Gy / MDFF_PI, fz = (double)Gz / MDFF_PI;
  // staging: half a wave per row of a plane, lane = z
  const int hz = threadIdx.x & 31, row0 = threadIdx.x >> 5;
  int gz = kTile * tz + min(hz, RZ - 1);
  gz = gz >= Gz ? gz - Gz : gz;
  const int xend = x1 - x0 + W - 1;                       // planes x0 .. x0 + xend - 1
  for (int base = p0; base < p1; base += NS) {
    double py[kGatherAtoms], dy[kGatherAtoms], ey[kGatherAtoms], pz[kGatherAtoms], dz[kGatherAtoms], ez[kGatherAtoms];
    double s0[kGatherAtoms], s1[kGatherAtoms], s2[kGatherAtoms], s3[kGatherAtoms], s4[kGatherAtoms], s5[kGatherAtoms];
    int off[kGatherAtoms], xs[kGatherAtoms], idx[kGatherAtoms];
    __syncthreads();                                      // the last round's planes and table are done with
    {
      double c[2 * kPair];
      load_piece<W>(a.coef, j, c);
#pragma unroll
      for (int r = 0; r < kGatherAtoms; ++r) {
        const int p = base + r * GRP + grp, slot = r * GRP + grp;
        const int4 at = a.at[min(p, p1 - 1)];
        const double4 vt = a.vt[min(p, p1 - 1)];
        idx[r] = p < p1 ? at.w : -1;
        off[r] = (at.y - kTile * ty) * RZ + (at.z - kTile * tz) + min(j, W - 1);
        s0[r] = s1[r] = s2[r] = s3[r] = s4[r] = s5[r] = 0.0;
        double f[3], df[3], d2[3];
        piece<true, SECOND>(c, vt.x, sg, f[0], df[0], d2[0]);
        piece<true, SECOND>(c, vt.y, sg, f[1], df[1], d2[1]);
        piece<true, SECOND>(c, vt.z, sg, f[2], df[2], d2[2]);
        xs[r] = p < p1 ? at.x - x0 : -4 * kTile;          // no plane touches an atom that is not there
        if (j < W) {
          px[slot][j][0] = f[0];
          px[slot][j][1] = df[0];
          if constexpr (SECOND) px[slot][j][2] = d2[0];
        }
        // lanes beyond the window hold zeros (their pieces have none)
        py[r] = f[1]; dy[r] = df[1]; ey[r] = SECOND ? d2[1] : 0.0;
        pz[r] = f[2]; dz[r] = df[2]; ez[r] = SECOND ? d2[2] : 0.0;
      }
    }
    for (int c0 = 0; c0 < xend; c0 += kPlanes) {
      const int nr = min(kPlanes, xend - c0) * RY;
      if (c0 > 0) __syncthreads();
      // (eight rows' loads in flight)
      for (int r0 = row0; r0 < nr; r0 += 8 * (kGatherThreads / 32)) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int row = min(r0 + u * (kGatherThreads / 32), nr - 1);
          const int pl = row / RY, yy = row - pl * RY;
          int gx = x0 + c0 + pl, gy = kTile * ty + yy;
          gx = gx >= 2 * Gx ? gx - 2 * Gx : (gx >= Gx ? gx - Gx : gx);
          gy = gy >= Gy ? gy - Gy : gy;
          v[u] = a.grid[((size_t)gx * Gy + gy) * Gz + gz];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int row = r0 + u * (kGatherThreads / 32);
          if (row < nr && hz < RZ) plane[row * RZ + hz] = v[u];
        }
      }
      __syncthreads();
#pragma unroll
      for (int r = 0; r < kGatherAtoms; ++r) {
        const int slot = r * GRP + grp;
        const int pb = max(0, xs[r] - c0), pe = min(min(kPlanes, xend - c0), xs[r] + W - c0);
        const double* pp = plane + off[r] + pb * (RY * RZ);
        const double* tx = px[slot][max(0, c0 - xs[r])];
        for (int pl = pb; pl < pe; ++pl) {
          double t0 = 0.0, t1 = 0.0, t2 = 0.0;
          row_sums<W, RZ, SECOND>(pp, py[r], dy[r], ey[r], t0, t1, t2);
          const double ax = tx[0], bx = tx[1];
          s0[r] = fma(bx, t0, s0[r]);                     // phi' phi
          s1[r] = fma(ax, t1, s1[r]);                     // phi  phi'
          s2[r] = fma(ax, t0, s2[r]);                     // phi  phi
          if constexpr (SECOND) {
            const double cx = tx[2];
            s3[r] = fma(cx, t0, s3[r]);                   // phi'' phi
            s4[r] = fma(ax, t2, s4[r]);                   // phi  phi''
            s5[r] = fma(bx, t1, s5[r]);                   // phi' phi'
          }
          pp += RY * RZ;
          tx += SECOND ? 4 : 2;
        }
      }
    }
#pragma unroll
    for (int r = 0; r < kGatherAtoms; ++r) {
      double m[9] = {fx * (pz[r] * s0[r]), fy * (pz[r] * s1[r]), fz * (dz[r] * s2[r])};
      if constexpr (SECOND) {
        m[3] = -(fx * fx) * (pz[r] * s3[r]);
        m[4] = -(fy * fy) * (pz[r] * s4[r]);
        m[5] = -(fz * fz) * (ez[r] * s2[r]);
        m[6] = -(fx * fy) * (pz[r] * s5[r]);
        m[7] = -(fx * fz) * (dz[r] * s0[r]);
        m[8] = -(fy * fz) * (dz[r] * s1[r]);
      }
#pragma unroll
      for (int k = 0; k < MOM; ++k) {
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) m[k] += __shfl_xor(m[k], o, 16);
        if (j == 0 && idx[r] >= 0) a.out[(size_t)k * a.n + idx[r]] = m[k];
      }
    }
  }
}

// ---- host: kernel, grid and tables ------------------------------------------

typedef long double ld;
const ld kPiL = 3.14159265358979323846264338327950288L;

// x I1(x): the kernel's profile up to a constant, by its series
ld bessel_xi1(ld x) {
  const ld y = x * x / 4;
  ld t = x * x / 2, s = t;
  for (int k = 1; k < 400 && t > s * 1e-22L; ++k) {
    t *= y / ((ld)k * (k + 1));
    s += t;
  }
  return s;
}

// transform of the kernel at frequency f (cycles per grid spacing), times a
// constant common to all f
template <typename R>
R kernel_hat(int w, R beta, R f) {
  const R h = (R)w / 2, a = 2 * (R)kPiL * f * h, z2 = beta * beta - a * a;
  if (std::fabs(z2) < (R)1e-6) return (R)1 / 3 + z2 / 30;
  const R z = std::sqrt(std::fabs(z2));
  if (z2 > 0) {
    const R e = std::exp(z);     // z cosh z - sinh z
    return ((z - 1) * e + (z + 1) / e) / (2 * z * z2);
  }
  return (std::sin(z) - z * std::cos(z)) / (z * -z2);
}

// Whether the alias error of the gradient of V from one direction, relative to
// the terms that carry the force, is above tol: mode n of weight a(n) >= A(n)/A(0)
// comes with modes n + jG of weight phih(n + jG) / phih(n), each differentiated.
// The force itself sits at n* = alpha |a| / (pi sqrt 2).  Measured errors are
// about 3 times this.  `first`: the mode looked at first, left at the one that was
// above, which is the likeliest to be so again.
bool mesh_error_above(int K, double aL, int G, int w, double beta, double tol, int& first) {
  const double pi = MDFF_PI, most = tol * std::max(1.0, aL / (pi * sqrt(2.0)));
  auto above = [&](int n) {
    double e = 0.0;
    for (int j = 1; j <= 2; ++j)
      for (int sg = -1; sg <= 1; sg += 2) {
        const double m = n + (double)sg * j * G;
        e += fabs(kernel_hat<double>(w, beta, m / G)) * fabs(m);
      }
    const double an = exp(-(pi * n / aL) * (pi * n / aL));
    return an * e / kernel_hat<double>(w, beta, (double)n / G) > most;
  };
  if (above(first)) return true;
  for (int n = K; n >= 0; --n)
    if (above(n)) {
      first = n;
      return true;
    }
  return false;
}

// Grids (multiples of the tile, at least the 2K + 1 modes and w) and the beta
// they share, with an error below tol in every direction: the beta whose
// grids have the fewest points.  false: none up to 4 (2K + 1) points.
bool choose_grid(const int* K, const double* aL, int w, double tol, int* G, double& beta) {
  double best = 0.0;
  int first[3] = {K[0], K[1], K[2]};
  for (double r = 1.5; r < 3.0; r += 0.05) {
    int g[3];
    double cells = 1.0;
    for (int d = 0; d < 3 && cells > 0.0; ++d) {
      if (d > 0 && K[d] == K[d - 1] && aL[d] == aL[d - 1]) {
        g[d] = g[d - 1];
      } else {
        const int lo = std::max(w, 2 * K[d] + 1), hi = 4 * lo + 2 * kTile;
        // the other directions have at least this one's size or their smallest
        // grid: no size is tried that could not beat the best
        double rest = 1.0;
        bool cube = true;
        for (int e = d + 1; e < 3; ++e) {
          cube = cube && K[e] == K[d] && aL[e] == aL[d];
          if (!cube) rest *= div_up(std::max(w, 2 * K[e] + 1), kTile) * kTile;
        }
        auto beaten = [&](int gd) {
          double c = cells * gd * rest;
          for (int e = d + 1; e < 3 && K[e] == K[d] && aL[e] == aL[d]; ++e) c *= gd;
          return best > 0.0 && c >= best;
        };
        g[d] = div_up(lo, kTile) * kTile;
        while (g[d] <= hi && !beaten(g[d]) && mesh_error_above(K[d], aL[d], g[d], w, r * w, tol, first[d])) g[d] += kTile;
        if (g[d] > hi || beaten(g[d])) cells = 0.0;
      }
      cells *= g[d];
      if (best > 0.0 && cells > best) cells = 0.0;
    }
    if (cells > 0.0 && (best == 0.0 || cells < best)) {
      best = cells;
      beta = r * w;
      for (int d = 0; d < 3; ++d) G[d] = g[d];
    }
  }
  return best > 0.0;
}

// pieces of phi on v in [-1, 1] (piece j: x = j - w/2 + (v + 1)/2) as
// polynomials through the Chebyshev nodes; coef[j][even | odd]
void kernel_pieces(int w, double beta, std::vector<double>& coef) {
  constexpr int M = kDeg + 1;
  ld T[M][M] = {};
  T[0][0] = 1;
  T[1][1] = 1;
  for (int k = 2; k < M; ++k)
    for (int c = 0; c < M; ++c) T[k][c] = (c ? 2 * T[k - 1][c - 1] : 0) - T[k - 2][c];
  ld cs[M][M];                             // cos(k (a + 1/2) pi / M)
  for (int k = 0; k < M; ++k)
    for (int a = 0; a < M; ++a) cs[k][a] = cosl(k * (a + 0.5L) * kPiL / M);
  const ld top = bessel_xi1(beta);
  coef.assign((size_t)(w / 2) * M, 0.0);
  for (int j = 0; j < w / 2; ++j) {
    ld y[M], mono[M] = {};
    for (int a = 0; a < M; ++a) {
      const ld v = cs[1][a];
      const ld x = (j - (ld)w / 2 + (v + 1) / 2) / ((ld)w / 2);
      const ld s2 = 1 - x * x;
      y[a] = s2 > 0 ? bessel_xi1((ld)beta * sqrtl(s2)) / top : 0;
    }
    for (int k = 0; k < M; ++k) {
      ld ck = 0;
      for (int a = 0; a < M; ++a) ck += y[a] * cs[k][a];
      ck *= (k ? 2.0L : 1.0L) / M;
      for (int c = 0; c <= k; ++c) mono[c] += ck * T[k][c];
    }
    for (int k = 0; k < M; ++k) coef[(size_t)j * M + (k & 1) * kPair + k / 2] = (double)mono[k];
  }
}

// x as the sum of two doubles
void push_split(std::vector<double>& v, ld x) {
  v.push_back((double)x);
  v.push_back((double)(x - (ld)(double)x));
}

// 1 / phih(n) for n = 0..K, phi as the pieces have it (x I1(x) over its top)
void push_deconv(std::vector<double>& v, int w, double beta, int K, int G) {
  const ld b = beta, top = bessel_xi1(b) / (w * b * b);
  for (int n = 0; n <= K; ++n) push_split(v, top / kernel_hat<ld>(w, b, (ld)n / G));
}

// e^{2 pi i a / G} for every a, as (cos, its rest, sin, its rest); G is a
// multiple of 16, so an eighth of the circle holds them all
void push_roots(std::vector<double>& v, int G) {
  std::vector<ld> c(G / 4 + 1), s(G / 4 + 1);
  for (int a = 0; a <= G / 8; ++a) {
    c[a] = s[G / 4 - a] = cosl(2 * kPiL * a / G);
    s[a] = c[G / 4 - a] = sinl(2 * kPiL * a / G);
  }
  for (int a = 0; a < G; ++a) {
    const int q = a / (G / 4), r = a % (G / 4);
    push_split(v, q == 0 ? c[r] : q == 1 ? -s[r] : q == 2 ? -c[r] : s[r]);
    push_split(v, q == 0 ? s[r] : q == 1 ? c[r] : q == 2 ? -s[r] : -c[r]);
  }
}

// ---- the matrices, made on the device: they and A(k) have as many entries as
// the k mesh, and made on the host they were most of a context's creation (LiF
// 195,112 24.5 ms, now 8.6; silica 24,000 FP64 3.2 ms, now 0.8).

struct TableArgs {
  int G[3], K[3], CN, ctiles;
  const double4* root[3];        // push_roots
  const double2* dec[3];         // 1 / phih(n), n = 0..K, as two doubles
  double *zf, *zb, *f[2], *b[2]; // f, b: x and y
  double *A, *kvec;
  double cell[9], alpha2;        // reciprocal matrix, column-major
};

// (x + its rest) times (d + its rest), rounded once
__device__ __forceinline__ double split_product(double x, double xl, double2 d) {
  const double p = x * d.x;
  return p + (fma(x, d.x, -p) + (x * d.y + xl * d.x));
}

// cos and sin of 2 pi a b / G over phih
__device__ __forceinline__ double2 table_entry(const TableArgs& a, int d, int mode, int point) {
  const long long G = a.G[d];
  const double4 r = a.root[d][(((long long)mode * point) % G + G) % G];
  const double2 w = a.dec[d][mode < 0 ? -mode : mode];
  return make_double2(split_product(r.x, r.y, w), split_product(r.z, r.w, w));
}

// blockIdx.y: 0 z forward, 1 z back, 2 and 3 x, 4 and 5 y forward and back, 6 the
// weights
__global__ void __launch_bounds__(256) k_mesh_tables(TableArgs a) {
  const int what = blockIdx.y, i0 = blockIdx.x * 256 + threadIdx.x, step = gridDim.x * 256;
  const int Gz = a.G[2];
  if (what < 2) {
    // operand order of a row product: [k / 16][column tile][step][lane].  Forward:
    // column tile 2 ct + part holds that part of nz = 16 ct ..; back: row k = 2 nz + part
    const int rows = what == 0 ? Gz : 32 * a.ctiles, nt = what == 0 ? 2 * a.ctiles : Gz / 16;
    double* out = what == 0 ? a.zf : a.zb;
    for (int i = i0; i < rows * nt * 16; i += step) {
      const int lane = i & 63, s = (i >> 6) & 3, tile = i >> 8;
      const int k = 16 * (tile / nt) + 4 * (lane >> 4) + s, col = 16 * (tile % nt) + (lane & 15);
      double v = 0.0;
      if (what == 0) {
        const int nz = 16 * (col >> 5) + (col & 15);
        if (nz < a.CN) {
          const double2 e = table_entry(a, 2, nz, k);
          v = (col & 16) ? e.y : e.x;
        }
      } else if (k < 2 * a.CN) {
        const double2 e = table_entry(a, 2, k >> 1, col);
        v = (k & 1) ? -e.y : e.x;
      }
      out[i] = v;
    }
  } else if (what < 6) {
    // operand order of a mid product: [l / 4][n tile of 8][re in, im in][lane]
    const int d = (what - 2) >> 1, G = a.G[d], K = a.K[d], M = 2 * K + 1;
    const bool back = what & 1;
    const int N = back ? G : M, L = back ? M : G, nt = (N + 7) / 8, lt = 4 * ((L + 15) / 16);
    double* out = back ? a.b[d] : a.f[d];
    for (int i = i0; i < lt * nt * 128; i += step) {
      const int lane = i & 63, im_in = (i >> 6) & 1, tile = i >> 7;
      const int R = lane & 15, part = (R >> 2) & 1;
      const int l = 4 * (tile / nt) + (lane >> 4), n = 8 * (tile % nt) + 4 * (R >> 3) + (R & 3);
      double v = 0.0;
      if (n < N && l < L) {
        const double2 e = table_entry(a, d, (back ? l : n) - K, back ? n : l);
        v = im_in ? (part ? e.x : -e.y) : (part ? e.y : e.x);
      }
      out[i] = v;
    }
  } else {
    // A and k on nz >= 0: an entry and its opposite are one term, so nz = 0 keeps
    // half of each of the two
    const int NX = 2 * a.K[0] + 1, NY = 2 * a.K[1] + 1;
    for (int i = i0; i < NX * NY * a.CN; i += step) {
      const int z = i % a.CN, xy = i / a.CN, y = xy % NY - a.K[1], x = xy / NY - a.K[0];
      const KWeight w = k_weight(a.cell, a.alpha2, x, y, z);
      a.A[i] = z == 0 ? 0.5 * w.A : w.A;
      a.kvec[4 * (size_t)i] = w.kx;
      a.kvec[4 * (size_t)i + 1] = w.ky;
      a.kvec[4 * (size_t)i + 2] = w.kz;
      a.kvec[4 * (size_t)i + 3] = w.kc;
    }
  }
}

}  // namespace

struct MeshRecip {
  int w = 0, dip = 0, second = 0;
  MeshGrid m{};
  int K[3] = {0, 0, 0}, CN = 0;            // CN = Kz + 1 complex columns
  int nbins = 0, shares = 1, X = 8, nblk = 0, ctiles = 0, ld = 0;
  int slice_zy = 0, slice_x = 0, slice_yz = 0;   // rows staged at a time, 0: all
  size_t lds_zy = 0, lds_x = 0, lds_yz = 0;
  int sorted = 0;                          // bins and phi belong to the current coordinates
  int counted = 0;                         // k_mesh_bin has run and the scan has not
  double *zf = nullptr, *zb = nullptr, *yf = nullptr, *yb = nullptr, *xf = nullptr, *xb = nullptr;
  void* mem = nullptr;                     // one allocation, the arrays its parts
  double *coef = nullptr, *A = nullptr, *kvec = nullptr;
  int32_t *key = nullptr, *slot = nullptr, *cnt = nullptr, *start = nullptr;
  BinAtom* order = nullptr;
  int4* at = nullptr;
  double4 *amp = nullptr, *vt = nullptr;
  double *phi = nullptr, *grid = nullptr, *mom = nullptr, *blk = nullptr;
  double2* t = nullptr;
};

// the transforms' kernels
static const void* zy_kernel(int shares, bool sliced) {
  switch (shares) {
    case 1: return sliced ? reinterpret_cast<const void*>(&k_mesh_zy<1, true>) : reinterpret_cast<const void*>(&k_mesh_zy<1, false>);
    case 2: return sliced ? reinterpret_cast<const void*>(&k_mesh_zy<2, true>) : reinterpret_cast<const void*>(&k_mesh_zy<2, false>);
    default: return sliced ? reinterpret_cast<const void*>(&k_mesh_zy<4, true>) : reinterpret_cast<const void*>(&k_mesh_zy<4, false>);
  }
}
static const void* x_kernel(bool sliced) {
  return sliced ? reinterpret_cast<const void*>(&k_mesh_x<true>) : reinterpret_cast<const void*>(&k_mesh_x<false>);
}
static const void* yz_kernel(bool sliced) {
  return sliced ? reinterpret_cast<const void*>(&k_mesh_yz<true>) : reinterpret_cast<const void*>(&k_mesh_yz<false>);
}

void mesh_free(mdff_ctx* c) {
  MeshRecip* m = c->mesh;
  if (!m) return;
  if (m->mem) (void)hipFree(m->mem);
  delete m;
  c->mesh = nullptr;
}

// Time (us) of an evaluation's transforms beyond their launches: by the
// operations of their products, and the grid's points.  Fitted over grids of
// 64^3 to 1104 x 144 x 96 (FP64, 64 to 4,096 ions: 160^3 154 of 156 us measured,
// 208 x 208 x 192 365 of 353, 272 x 272 x 224 732 of 698, 736 x 272 x 112 1074 of
// 1070; the longest, 1104 x 144 x 96, 790 of 1126).
static double mesh_transform_us(const int* G, const int* K) {
  const double NX = 2 * K[0] + 1, NY = 2 * K[1] + 1, CN = K[2] + 1, cp = 16 * div_up(K[2] + 1, 16);
  const double points = (double)G[0] * G[1] * G[2];
  const double ops = 2.0 * (4.0 * points * cp + 8.0 * G[0] * G[1] * NY * cp + 8.0 * G[0] * NX * NY * CN);
  return 30e-9 * ops + 8e-6 * points;
}

// Leaves c->mesh null where no grid meets the error bound, or the transforms of
// the one that does would take more than most_us.
int mesh_setup(mdff_ctx* c, double most_us) {
  const int n = c->n;
  const bool wide = c->rec_wide != 0;
  const int w = wide ? 16 : 12;
  // the gradient's second derivatives weigh the alias error by k^2: with
  // 4e-15 its error at 1,728 ions would be 4e-14, with 5e-16 it is 1.3e-14, the
  // direct sums' 1e-14 (4,096 ions 4.3e-14 and 4.1e-14; 338 against 318 us)
  const double tol = c->d.doefg ? 5e-16 : (wide ? 4e-15 : 1e-9);
  int G[3];
  double aL[3], beta = 0.0;
  for (int d = 0; d < 3; ++d) {
    const double* a = c->A + 3 * d;
    aL[d] = c->alpha * sqrt(a[0] * a[0] + a[1] * a[1] + a[2] * a[2]);
  }
  if (!choose_grid(c->K, aL, w, tol, G, beta)) return MDFF_OK;
  if ((double)G[0] * G[1] * G[2] > 536870912.0) return MDFF_OK;   // 4 GiB of grid
  if (mesh_transform_us(G, c->K) > most_us) return MDFF_OK;
  // LDS of the transforms (doubles: planes and the waves' exchange), and the
  // rows that fit
  const int nyp = (2 * c->K[1] + 16) & ~15, nxp = (2 * c->K[0] + 16) & ~15;
  const int ctiles = div_up(c->K[2] + 1, 16), yld = 32 * ctiles + 2;
  int maxlds = 0;
  HIP_TRY(c, hipDeviceGetAttribute(&maxlds, hipDeviceAttributeMaxSharedMemoryPerBlock, c->device));
  const int xch = kFtWaves / 2 * 256, room = maxlds / 8 - xch;
  const int fit = (room / 32) & ~15, fit_yz = std::max(0, room - kYzRows * yld) / 64 & ~15;
  if (fit_yz < 16) return MDFF_OK;         // kES(3) beyond 270
  const int slice_zy = G[1] <= fit ? 0 : fit, slice_x = G[0] + nxp <= fit ? 0 : fit, slice_yz = nyp <= fit_yz ? 0 : fit_yz;
  const size_t lds_zy = 8 * (32 * (size_t)std::min(G[1], fit) + xch), lds_x = 8 * (32 * (size_t)std::min(G[0] + nxp, fit) + xch),
               lds_yz = 8 * ((size_t)kYzRows * yld + 64 * (size_t)std::min(nyp, fit_yz) + xch);
  for (int sl = 0; sl < 2; ++sl)
    for (const void* fn : {zy_kernel(1, sl), zy_kernel(2, sl), zy_kernel(4, sl), x_kernel(sl), yz_kernel(sl)})
      HIP_TRY(c, hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, maxlds));
  MeshRecip* m = new MeshRecip();
  c->mesh = m;
  m->w = w;
  m->ctiles = ctiles;
  m->ld = yld;
  m->slice_zy = slice_zy;
  m->slice_x = slice_x;
  m->slice_yz = slice_yz;
  m->lds_zy = lds_zy;
  m->lds_x = lds_x;
  m->lds_yz = lds_yz;
  m->dip = (c->task_qd || c->task_dd) ? 1 : 0;
  for (int d = 0; d < 3; ++d) {
    m->m.G[d] = G[d];
    m->K[d] = c->K[d];
  }
  m->m.nyb = G[1] / kTile;
  m->m.nzb = G[2] / kTile;
  m->nbins = G[0] * m->m.nyb * m->m.nzb;
  const int tiles = (G[0] / kTile) * m->m.nyb * m->m.nzb;
  // blocks of the spread: shares of a tile's four bin columns until every
  // CU has a block
  m->shares = tiles >= 192 ? 1 : (tiles >= 96 ? 2 : 4);
  // window starts per gather block: about as many atoms as it has in flight
  const double per_x = (double)n / m->nbins;
  const int flight = kGatherThreads / 16 * kGatherAtoms;
  m->X = std::max(2, std::min(16, (int)(0.9 * flight / std::max(per_x, 1e-3))));
  m->CN = c->K[2] + 1;
  const int CN = m->CN, NX = 2 * c->K[0] + 1, NY = 2 * c->K[1] + 1;
  // what the host makes: the pieces of phi, roots and deconvolution, one copy
  std::vector<double> small;
  kernel_pieces(w, beta, small);
  size_t root_at[3], dec_at[3];
  for (int d = 0; d < 3; ++d) {
    int same = 0;
    while (same < d && G[same] != G[d]) ++same;
    root_at[d] = same < d ? root_at[same] : small.size();
    if (same == d) push_roots(small, G[d]);
  }
  for (int d = 0; d < 3; ++d) {
    int same = 0;
    while (same < d && (G[same] != G[d] || c->K[same] != c->K[d])) ++same;
    dec_at[d] = same < d ? dec_at[same] : small.size();
    if (same == d) push_deconv(small, w, beta, c->K[d], G[d]);
  }
  m->nblk = div_up((int64_t)NY * CN, 16);
  std::vector<std::pair<void**, size_t>> parts;
  auto part = [&](auto** p, size_t count) { parts.push_back({(void**)p, (sizeof(**p) * count + 255) & ~(size_t)255}); };
  const int nr = m->dip ? 6 : 3;
  const size_t nk = (size_t)NX * NY * CN, zt = (size_t)32 * ctiles * G[2];
  auto mid_size = [](int N, int L) { return (size_t)4 * div_up(L, 16) * div_up(N, 8) * 128; };
  part(&m->coef, small.size());
  part(&m->zf, zt);
  part(&m->zb, zt);
  part(&m->yf, mid_size(NY, G[1]));
  part(&m->yb, mid_size(G[1], NY));
  part(&m->xf, mid_size(NX, G[0]));
  part(&m->xb, mid_size(G[0], NX));
  part(&m->A, nk);
  part(&m->kvec, 4 * nk);
  part(&m->key, n);
  part(&m->slot, n);
  part(&m->order, n);
  part(&m->cnt, m->nbins);
  part(&m->start, m->nbins + 1);
  part(&m->at, n);
  part(&m->phi, (size_t)nr * w * n);
  part(&m->vt, n);
  if (m->dip) part(&m->amp, n);
  part(&m->grid, (size_t)G[0] * G[1] * G[2] * m->shares);
  part(&m->t, (size_t)G[0] * NY * CN);
  part(&m->mom, 9 * (size_t)n);
  part(&m->blk, 7 * (size_t)m->nblk);
  size_t total = 0;
  for (const auto& p : parts) total += p.second;
  HIP_TRY(c, hipMalloc(&m->mem, total));
  total = 0;
  for (const auto& p : parts) {
    *p.first = (char*)m->mem + total;
    total += p.second;
  }
  HIP_TRY(c, hipMemcpy(m->coef, small.data(), sizeof(double) * small.size(), hipMemcpyHostToDevice));
  // (on the context's stream: hipMemset may return before the null stream has done
  // it, and this stream does not wait for that one)
  HIP_TRY(c, hipMemsetAsync(m->cnt, 0, sizeof(int32_t) * m->nbins, c->stream));
  TableArgs ta{};
  for (int d = 0; d < 3; ++d) {
    ta.G[d] = G[d];
    ta.K[d] = c->K[d];
    ta.root[d] = reinterpret_cast<const double4*>(m->coef + root_at[d]);
    ta.dec[d] = reinterpret_cast<const double2*>(m->coef + dec_at[d]);
  }
  ta.CN = CN;
  ta.ctiles = ctiles;
  ta.zf = m->zf; ta.zb = m->zb;
  ta.f[0] = m->xf; ta.b[0] = m->xb;
  ta.f[1] = m->yf; ta.b[1] = m->yb;
  ta.A = m->A; ta.kvec = m->kvec;
  for (int k = 0; k < 9; ++k) ta.cell[k] = c->B[k];
  ta.alpha2 = c->alpha * c->alpha;
  hipLaunchKernelGGL(k_mesh_tables, dim3(std::min(256, div_up(nk, 256)), 7), dim3(256), 0, c->stream, ta);
  HIP_TRY(c, hipGetLastError());
  return MDFF_OK;
}

// s = B^T r (from_r) and the bin counts; pack: also the pair kernel's atoms.
// The previous MD step's queued sums ride along.
int mesh_bin(mdff_ctx* c, bool from_r, bool pack) {
  MeshRecip* m = c->mesh;
  if (m->counted)   // an evaluation that ended early left its counts
    hipLaunchKernelGGL(k_mesh_clear, dim3(div_up(m->nbins, 256)), dim3(256), 0, c->stream, m->nbins, m->cnt);
  BinArgs a{};
  a.n = c->n;
  a.from_r = from_r ? 1 : 0;
  a.pack = pack ? 1 : 0;
  a.m = m->m;
  a.rx = c->rx; a.ry = c->ry; a.rz = c->rz;
  for (int k = 0; k < 9; ++k) a.b[k] = c->B[k];
  a.sx = c->sx; a.sy = c->sy; a.sz = c->sz;
  a.key = m->key;
  a.slot = m->slot;
  a.cnt = m->cnt;
  a.order = c->cell_atoms;
  a.q = c->q;
  a.itype = c->itype;
  a.rec = c->arec;
  a.meta = c->ameta;
  const int nbx = div_up(c->n, 256);
  if (c->nfin > nbx) MDFF_TRY(flush_finals(c));
  const FinalBatch fb = from_r ? take_finals(c) : FinalBatch{};
  const bool extra = fb.nfin > 0 || fb.seq_out;
  const dim3 grid(nbx, extra ? 2 : 1);
  m->counted = 1;
  m->sorted = 0;
  if (m->w == 16)
    PROF_LAUNCH(c, PK_TABLES,
                hipLaunchKernelGGL(k_mesh_bin<16>, grid, dim3(256), 0, c->stream, a, fb, extra ? 1 : -1));
  else
    PROF_LAUNCH(c, PK_TABLES,
                hipLaunchKernelGGL(k_mesh_bin<12>, grid, dim3(256), 0, c->stream, a, fb, extra ? 1 : -1));
  HIP_TRY(c, hipGetLastError());
  return MDFF_OK;
}

// bins to sorted atoms and their kernel values
static int mesh_sort(mdff_ctx* c) {
  MeshRecip* m = c->mesh;
  if (m->sorted) return MDFF_OK;
  const int n = c->n;
  ScatterArgs sc{};
  sc.n = n;
  sc.nb = m->nbins;
  sc.key = m->key; sc.slot = m->slot; sc.cnt = m->cnt;
  sc.start = m->start;
  sc.sx = c->sx; sc.sy = c->sy; sc.sz = c->sz;
  sc.order = m->order;
  if (m->nbins <= kScanBins) {
    PROF_LAUNCH(c, PK_TABLES, hipLaunchKernelGGL(k_mesh_scatter<true>, dim3(div_up(n, 256)), dim3(256), 0, c->stream, sc));
  } else {
    PROF_LAUNCH(c, PK_TABLES,
                hipLaunchKernelGGL(k_mesh_scan, dim3(1), dim3(1024), 0, c->stream, m->nbins, m->cnt, m->start));
    PROF_LAUNCH(c, PK_TABLES, hipLaunchKernelGGL(k_mesh_scatter<false>, dim3(div_up(n, 256)), dim3(256), 0, c->stream, sc));
  }
  PhiArgs a{};
  a.n = n;
  a.m = m->m;
  a.start = m->start;
  a.cnt = m->cnt;
  a.nb = m->nbins;
  a.order = m->order;
  a.q = c->q;
  a.coef = m->coef;
  a.at = m->at;
  a.vt = m->vt;
  a.phi = m->phi;
  const dim3 grid(std::min(2048, div_up(n, 16)));
  if (m->w == 16) {
    if (m->dip) PROF_LAUNCH(c, PK_TABLES, hipLaunchKernelGGL((k_mesh_phi<16, true>), grid, dim3(256), 0, c->stream, a));
    else PROF_LAUNCH(c, PK_TABLES, hipLaunchKernelGGL((k_mesh_phi<16, false>), grid, dim3(256), 0, c->stream, a));
  } else {
    if (m->dip) PROF_LAUNCH(c, PK_TABLES, hipLaunchKernelGGL((k_mesh_phi<12, true>), grid, dim3(256), 0, c->stream, a));
    else PROF_LAUNCH(c, PK_TABLES, hipLaunchKernelGGL((k_mesh_phi<12, false>), grid, dim3(256), 0, c->stream, a));
  }
  HIP_TRY(c, hipGetLastError());
  m->counted = 0;
  m->sorted = 1;
  return MDFF_OK;
}

template <int W>
static void launch_spread(mdff_ctx* c, const SpreadArgs& a, bool dip, dim3 grid) {
  if (dip) PROF_LAUNCH(c, PK_SK, hipLaunchKernelGGL((k_mesh_spread<W, true>), grid, dim3(1024), 0, c->stream, a));
  else PROF_LAUNCH(c, PK_SK, hipLaunchKernelGGL((k_mesh_spread<W, false>), grid, dim3(1024), 0, c->stream, a));
}

template <int W>
static void launch_gather(mdff_ctx* c, const GatherArgs& a, int mom, dim3 grid) {
  if (mom == 9)
    PROF_LAUNCH(c, PK_GATHER, hipLaunchKernelGGL((k_mesh_gather<W, 9>), grid, dim3(kGatherThreads), 0, c->stream, a));
  else
    PROF_LAUNCH(c, PK_GATHER, hipLaunchKernelGGL((k_mesh_gather<W, 3>), grid, dim3(kGatherThreads), 0, c->stream, a));
}

// S of the charges or (use_mu) of the dipoles mu and, use_q, the charges; W, the
// 7 energy / stress sums into e_out (queued), and with mom = 3 or 9 the moments
// of every atom; *out: [mom][n]
int mesh_eval(mdff_ctx* c, const double* mu, bool use_q, bool use_mu, int mom, double* e_out, const double** out) {
  MeshRecip* m = c->mesh;
  MDFF_TRY(mesh_sort(c));
  const int n = c->n;
  const int Gx = m->m.G[0], Gy = m->m.G[1], Gz = m->m.G[2];
  const int NX = 2 * m->K[0] + 1, NY = 2 * m->K[1] + 1, CN = m->CN;
  if (use_mu) {
    const double* b = c->B;
    PROF_LAUNCH(c, PK_SK, hipLaunchKernelGGL(k_mesh_amp, dim3(div_up(n, 256)), dim3(256), 0, c->stream, n, m->at, c->q,
                                             use_q ? 1 : 0, mu, b[0], b[1], b[2], b[3], b[4], b[5], b[6], b[7], b[8],
                                             -2.0 * Gx, -2.0 * Gy, -2.0 * Gz, m->amp));
  }
  SpreadArgs sa{};
  sa.n = n;
  sa.shares = m->shares;
  sa.m = m->m;
  sa.start = m->start;
  sa.at = m->at;
  sa.phi = m->phi;
  sa.vt = m->vt;
  sa.pstride = (m->dip ? 6 : 3) * m->w;
  sa.amp = m->amp;
  sa.out = m->grid;
  const dim3 sg((Gx / kTile) * m->m.nyb * m->m.nzb * m->shares);
  if (m->w == 16) launch_spread<16>(c, sa, use_mu, sg);
  else launch_spread<12>(c, sa, use_mu, sg);
  ZyArgs za{};
  za.Gy = Gy; za.Gz = Gz; za.CN = CN; za.NY = NY;
  za.ctiles = m->ctiles;
  za.slice = m->slice_zy;
  za.sstride = (size_t)Gx * Gy * Gz;
  za.grid = m->grid;
  za.zf = m->zf; za.yf = m->yf;
  za.out = m->t;
  void* zargs[] = {&za};
  PROF_LAUNCH(c, PK_SKRED, (void)hipLaunchKernel(zy_kernel(m->shares, m->slice_zy > 0), dim3(m->ctiles, Gx), dim3(kFtThreads),
                                                 zargs, m->lds_zy, c->stream));
  MDFF_TRY(claim_partials(c, m->blk));
  XArgs xa{};
  xa.Gx = Gx; xa.NX = NX; xa.C = NY * CN;
  xa.back = mom > 0 ? 1 : 0;
  xa.slice = m->slice_x;
  // (the grid is free between the plane transforms, and at least as large:
  // NX <= Gx, NY <= Gy, 2 CN <= Gz)
  xa.s = reinterpret_cast<double2*>(m->grid);
  xa.xf = m->xf; xa.xb = m->xb;
  xa.t = m->t;
  xa.A = m->A; xa.kvec = m->kvec; xa.blk = m->blk;
  void* xargs[] = {&xa};
  PROF_LAUNCH(c, PK_SKRED, (void)hipLaunchKernel(x_kernel(m->slice_x > 0), dim3(m->nblk), dim3(kFtThreads), xargs, m->lds_x,
                                                 c->stream));
  if (e_out) MDFF_TRY(queue_final(c, m->blk, m->nblk, 7, e_out));
  if (mom > 0) {
    YzArgs ya{};
    ya.Gy = Gy; ya.Gz = Gz; ya.CN = CN; ya.NY = NY;
    ya.ctiles = m->ctiles;
    ya.ld = m->ld;
    ya.slice = m->slice_yz;
    ya.in = m->t;
    ya.yb = m->yb; ya.zb = m->zb;
    ya.grid = m->grid;
    void* yargs[] = {&ya};
    PROF_LAUNCH(c, PK_SKRED, (void)hipLaunchKernel(yz_kernel(m->slice_yz > 0), dim3(div_up(Gy, kYzRows), Gx), dim3(kFtThreads),
                                                   yargs, m->lds_yz, c->stream));
    GatherArgs ga{};
    ga.n = n;
    ga.X = m->X;
    ga.m = m->m;
    ga.start = m->start;
    ga.at = m->at;
    ga.vt = m->vt;
    ga.coef = m->coef;
    ga.grid = m->grid;
    ga.out = m->mom;
    const dim3 gg(div_up(Gx, m->X), m->m.nyb * m->m.nzb);
    if (m->w == 16) launch_gather<16>(c, ga, mom, gg);
    else launch_gather<12>(c, ga, mom, gg);
    *out = m->mom;
  }
  HIP_TRY(c, hipGetLastError());
  return MDFF_OK;
}
