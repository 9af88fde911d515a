// FP64 far field of large meshes by tile expansions (gz, and gz + FTG).
//
// The mesh is cut into tiles of 8 x 8 x 8 cells.  A site farther than kRatio half-diagonals from
// a tile's centre sees the tile through its solid-harmonic moments up to degree kDeg; nearer
// tiles are summed with the closed form, corner by corner.  With t = (s - centre) / half-diagonal,
//
//   phi(s) = (1/a) Re sum_{l,m} M_l^m I_l^m(t),   M_l^m = sum_cells rho int conj(R_l^m),
//   I_n^m = (-1)^m (2n-1)!! h_{n,m} E_m,  E_m = (x + i y)^m / r^{2m+1},
//   h_{m,m} = 1,  h_{n+1,m} = (z/r^2) h_{n,m} - (n^2-m^2)/((2n+1)(2n-1)) h_{n-1,m} / r^2,
//
// R and I the regular and irregular solid harmonics r^l P_l^m e^{im phi} / (l+m)! and
// (l-m)! P_l^m e^{im phi} / r^{l+1}.  Derivatives shift the indices: d/dz I_l^m = -I_{l+1}^m and
// (d/dx + i d/dy) I_l^m = I_{l+1}^{m+1}, so gz and the tensor are sums over I_{l+1} and I_{l+2}.
// The gradient is the transpose: local coefficients Lambda_l^m per tile, summed over the far
// sites, then integrated over each cell as a polynomial.
//
// Truncation: it is largest for a body of one cell in a corner of its tile, seen in that corner's
// direction from kRatio half-diagonals.  Of the body's largest value at that distance it is at most
// 9e-13 there, in every tensor component and in gz, for tiles of any shape (1 to 8 cells a side,
// cells of 1 : 4 to 4 : 1); 2 x 2 x 2 cells of a whole tile leave 2e-13, 4 x 4 x 4 2e-14, the tile
// itself 2e-15.  The closed form's own rounding is no smaller: 8e-13 to 2e-12 (median over
// directions) of one cell's diagonal components there, 5e-12 of the others, 1e-11 of gz, and less
// as the body grows.  So no density loses accuracy to the expansions.  (Degree 16 from 4
// half-diagonals on takes 6.8 instead of 9.4 ms for data and gradient of 2048 tiles and 4096 sites,
// but leaves 6e-10 of one cell and 1e-11 of 4 x 4 x 4; degree 22 from 4 on takes 9.3 ms, but 16.4
// instead of 14.2 for eight models and 1024 sites.)
//
// A site-tile pair takes about 4700 FP64 operations (gz + FTG; 1600 for gz) in the data and 9200
// (3900) in the gradient, against 512 cells at 250 (170) and as many corners.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <complex>
#include <type_traits>
#include <vector>

#include "context.hpp"
#include "epilogue.hpp"
#include "prism_device.hpp"

namespace jgm {

namespace {

constexpr int kBlock = 256;
constexpr int kT = 8;                       // cells per tile and axis
constexpr int kTC = kT + 1;                 // corners per tile and axis
constexpr int kTCorners = kTC * kTC * kTC;  // 729
constexpr int kDeg = 20;                    // largest degree of the moments
constexpr int kK = kDeg + 1;
// nearest far site, in tile half-diagonals
template <int MASK>
constexpr double kRatio = MASK == kMaskScalar ? 3.95 : 4.4;
constexpr int kMono = kK * (kK + 1) * (kK + 2) / 6;  // monomials of degree <= kDeg: 1771
constexpr int kPairs = kK * (kK + 1) / 2;            // (l, m), 0 <= m <= l: 231
constexpr int kRows = 2 * kPairs;
// (n, m) of the irregular harmonics: n = 1 .. kDeg + 2, m = 0 .. n, m-major
constexpr int kOrders = kDeg + 3;
constexpr int kNM = (kOrders + 1) * kOrders / 2 - 1;

inline unsigned blocks_for(long n) { return (unsigned)((n + kBlock - 1) / kBlock); }

__host__ __device__ constexpr int lm_index(int l, int m) { return l * (l + 1) / 2 + m; }
__host__ __device__ constexpr double odd_factorial(int n) {  // (2n - 1)!!
  double f = 1.0;
  for (int k = 1; k < n; ++k) f *= 2 * k + 1;
  return f;
}
__host__ __device__ constexpr double gamma_nm(int n, int m) {
  return (double)(n * n - m * m) / (double)((2 * n + 1) * (2 * n - 1));
}

struct TileGrid {
  const double *Xc, *Yc, *Zc;
  int nx, ny, nz, tx, ty, tz;
};

// Tile t: its cells' first indices and counts, centre and inverse half-diagonal.
struct Tile {
  int i0, j0, k0, ni, nj, nk;
  double cx, cy, cz, a, inva;
};

__device__ __forceinline__ Tile tile_of(const TileGrid& g, int t) {
  Tile q;
  const int k = t % g.tz, ij = t / g.tz, j = ij % g.ty, i = ij / g.ty;
  q.i0 = i * kT;
  q.j0 = j * kT;
  q.k0 = k * kT;
  q.ni = min(kT, g.nx - q.i0);
  q.nj = min(kT, g.ny - q.j0);
  q.nk = min(kT, g.nz - q.k0);
  const double x0 = g.Xc[q.i0], x1 = g.Xc[q.i0 + q.ni];
  const double y0 = g.Yc[q.j0], y1 = g.Yc[q.j0 + q.nj];
  const double z0 = g.Zc[q.k0], z1 = g.Zc[q.k0 + q.nk];
  q.cx = 0.5 * (x0 + x1);
  q.cy = 0.5 * (y0 + y1);
  q.cz = 0.5 * (z0 + z1);
  const double dx = x1 - x0, dy = y1 - y0, dz = z1 - z0;
  q.a = 0.5 * sqrt(fma(dx, dx, fma(dy, dy, dz * dz)));
  q.inva = 1.0 / q.a;
  return q;
}

// Workgroup b of the kernels that take a tile each: layer by layer from the top.  Workgroups go
// to the eight XCDs in turn, and in the tiles' own order (z fastest) a mesh of eight layers of
// tiles gives each XCD one layer, the uppermost with nearly all near sites (near gradient of
// 2048 tiles and 4096 sites 5.8 ms, 2.0 ms this way).
__device__ __forceinline__ int tile_of_block(const TileGrid& g, int b) {
  const int columns = g.tx * g.ty;
  return b % columns * g.tz + b / columns;
}

// centre and inverse half-diagonal of every tile, for the kernels that only test distances
__global__ __launch_bounds__(kBlock) void k_tile_centres(TileGrid g, int ntiles,
                                                         double4* __restrict__ geo) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ntiles) return;
  const Tile q = tile_of(g, t);
  geo[t] = make_double4(q.cx, q.cy, q.cz, q.inva);
}

// Offset of a site from a tile's centre in half-diagonals; far from kRatio of them on.  Every
// kernel decides with these operations, so a pair is near in one pass and far in the other.
struct Offset {
  double x, y, z, r2;
  template <int MASK>
  __device__ __forceinline__ bool far() const {
    return r2 >= kRatio<MASK> * kRatio<MASK>;
  }
};
__device__ __forceinline__ Offset offset_of(double px, double py, double pz, double4 c) {
  Offset o;
  o.x = (px - c.x) * c.w;
  o.y = (py - c.y) * c.w;
  o.z = (pz - c.z) * c.w;
  o.r2 = fma(o.x, o.x, fma(o.y, o.y, o.z * o.z));
  return o;
}

// Mean of 1024 cells spread over the mesh.  The tiles carry the densities less this value and
// the whole mesh as one box carries it: what a nearly uniform model's cells have in common
// cancels before any truncation, as it does in the corner weights of the closed form.
__global__ __launch_bounds__(1024) void k_reference_density(const double* __restrict__ rho,
                                                            long ld, long n,
                                                            double* __restrict__ ref) {
  __shared__ double red[1024];
  rho += blockIdx.x * ld;
  red[threadIdx.x] = rho[(long)((2.0 * threadIdx.x + 1.0) * (double)n / 2048.0)];
  __syncthreads();
  for (int w = 512; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) ref[blockIdx.x] = red[0] * (1.0 / 1024.0);
}

// Corner sums of the mesh as one box of the reference density: one row of partial a model.
template <int MASK>
__global__ __launch_bounds__(kBlock) void k_reference_box(
    const double* __restrict__ sx, const double* __restrict__ sy, const double* __restrict__ sz,
    int S, TileGrid g, const double* __restrict__ ref, int nb, double* __restrict__ partial,
    long ld) {
  constexpr int NC = Ncomp<MASK>::value;
  __shared__ LogTableShared tab;
  const LogTable lg = tab.fill();
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= S) return;
  double acc[NC];
#pragma unroll
  for (int m = 0; m < NC; ++m) acc[m] = 0.0;
  for (int c = 0; c < 8; ++c) {
    double v[NC];
    corner_terms_f64<MASK>(sx[s] - g.Xc[c & 1 ? g.nx : 0], sy[s] - g.Yc[c & 2 ? g.ny : 0],
                           sz[s] - g.Zc[c & 4 ? g.nz : 0], v, lg);
    const bool plus = ((c ^ c >> 1 ^ c >> 2) & 1) != 0;
#pragma unroll
    for (int m = 0; m < NC; ++m) acc[m] += plus ? v[m] : -v[m];
  }
  for (int b = 0; b < nb; ++b)
#pragma unroll
    for (int m = 0; m < NC; ++m) partial[b * ld + (long)m * S + s] = acc[m] * ref[b];
}

// Integrals over the tile's cells of powers of the scaled coordinate:
// m[axis][cell][k] = (t1^{k+1} - t0^{k+1}) / (k + 1); cells past the tile's end are zero.
__device__ inline void axis_moments(const TileGrid& g, const Tile& q, double (*m)[kT][kK]) {
  for (int e = threadIdx.x; e < 3 * kT; e += blockDim.x) {
    const int axis = e / kT, c = e % kT;
    const double* C = axis == 0 ? g.Xc + q.i0 : axis == 1 ? g.Yc + q.j0 : g.Zc + q.k0;
    const double centre = axis == 0 ? q.cx : axis == 1 ? q.cy : q.cz;
    const int n = axis == 0 ? q.ni : axis == 1 ? q.nj : q.nk;
    if (c >= n) {
      for (int k = 0; k < kK; ++k) m[axis][c][k] = 0.0;
      continue;
    }
    const double t0 = (C[c] - centre) * q.inva, t1 = (C[c + 1] - centre) * q.inva;
    double p0 = t0, p1 = t1;
    for (int k = 0; k < kK; ++k) {
      m[axis][c][k] = (p1 - p0) / (k + 1);
      p0 *= t0;
      p1 *= t1;
    }
  }
}

// pair index of (b, c) with b + c <= kDeg, c-major
__device__ __forceinline__ int bc_index(int b, int c) { return c * kK - c * (c - 1) / 2 + b; }

// Sparse harmonic polynomials: row r (2 lm for Re R_l^m, 2 lm + 1 for Im R_l^m) has the
// monomials idx[ptr[r] ..] with coefficients val; mono packs (a, b, c) of x^a y^b z^c.
struct HarmonicTable {
  const int *ptr, *idx, *cptr, *cidx, *mono;
  const double *val, *cval;
};

// Complex M_l^m for any m, from the stored m >= 0 (M^{-m} = (-1)^m conj M^m); zero outside.
__device__ __forceinline__ void moment(const double* M, int l, int m, double& re, double& im) {
  const int am = m < 0 ? -m : m;
  if (l < 0 || l > kDeg || am > l) {
    re = im = 0.0;
    return;
  }
  re = M[2 * lm_index(l, am)];
  im = M[2 * lm_index(l, am) + 1];
  if (m < 0) {
    if (am & 1)
      re = -re;
    else
      im = -im;
  }
}

// Moments of a tile and, from them, the coefficients A, B of Re E_m and Im E_m per (n, m) and
// quantity that the data kernel multiplies with h_{n,m}: gz; for gz + FTG gz, Uzz, Uxx - Uyy,
// 2 Uxy, Uxz, Uyz.  Also the tile's own corner weights for the near sum.  grid: x = tiles,
// y = models.
template <int MASK>
__global__ __launch_bounds__(kBlock) void k_tile_moments(TileGrid g, int ntiles,
                                                         const double* __restrict__ rho, long ld,
                                                         const double* __restrict__ ref,
                                                         HarmonicTable h,
                                                         double* __restrict__ coefs,
                                                         double* __restrict__ wt) {
  constexpr int NQ = MASK == kMaskScalar ? 1 : 6;
  __shared__ double ax[3][kT][kK];
  __shared__ double cell[kT * kT * kT];
  __shared__ double A[kK][kT * kT];
  __shared__ double B[kPairs][kT];
  __shared__ double mu[kMono];
  __shared__ double M[kRows];
  const int t = blockIdx.x;
  rho += blockIdx.y * ld;
  ref += blockIdx.y;
  coefs += (long)blockIdx.y * ntiles * kNM * 2 * NQ;
  wt += (long)blockIdx.y * ntiles * kTCorners;
  const Tile q = tile_of(g, t);
  axis_moments(g, q, ax);
  for (int e = threadIdx.x; e < kT * kT * kT; e += kBlock) {
    const int k = e % kT, j = e / kT % kT, i = e / (kT * kT);
    cell[e] = i < q.ni && j < q.nj && k < q.nk
                  ? rho[((long)(q.i0 + i) * g.ny + (q.j0 + j)) * g.nz + q.k0 + k] - ref[0]
                  : 0.0;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < kTCorners; e += kBlock) {
    const int K = e % kTC, J = e / kTC % kTC, I = e / (kTC * kTC);
    double w = 0.0;
    for (int a = 0; a < 2; ++a)
      for (int b = 0; b < 2; ++b)
        for (int c = 0; c < 2; ++c) {
          const int i = I - a, j = J - b, k = K - c;
          if (i < 0 || j < 0 || k < 0 || i >= kT || j >= kT || k >= kT) continue;
          const double v = cell[(i * kT + j) * kT + k];
          w += ((a + b + c) & 1) ? v : -v;
        }
    wt[(long)t * kTCorners + e] = w;
  }
  for (int e = threadIdx.x; e < kK * kT * kT; e += kBlock) {
    const int ij = e % (kT * kT), c = e / (kT * kT);
    double s = 0.0;
    for (int k = 0; k < kT; ++k) s = fma(cell[ij * kT + k], ax[2][k][c], s);
    A[c][ij] = s;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < kK * kK * kT; e += kBlock) {
    const int i = e % kT, b = e / kT % kK, c = e / (kT * kK);
    if (b + c > kDeg) continue;
    double s = 0.0;
    for (int j = 0; j < kT; ++j) s = fma(A[c][i * kT + j], ax[1][j][b], s);
    B[bc_index(b, c)][i] = s;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < kMono; e += kBlock) {
    const int p = h.mono[e], a = p & 255, bc = bc_index((p >> 8) & 255, p >> 16);
    double s = 0.0;
    for (int i = 0; i < kT; ++i) s = fma(B[bc][i], ax[0][i][a], s);
    mu[e] = s;
  }
  __syncthreads();
  for (int r = threadIdx.x; r < kRows; r += kBlock) {
    double s = 0.0;
    for (int e = h.ptr[r]; e < h.ptr[r + 1]; ++e) s = fma(h.val[e], mu[h.idx[e]], s);
    M[r] = (r & 1) ? -s : s;  // conj(R)
  }
  __syncthreads();
  double* out = coefs + (long)t * kNM * 2 * NQ;
  for (int e = threadIdx.x; e < kNM; e += kBlock) {
    int m = 0, first = 0;  // (n, m) of entry e
    for (; m < kOrders; ++m) {
      const int count = kOrders - (m < 1 ? 1 : m);
      if (e < first + count) break;
      first += count;
    }
    const int n = (m < 1 ? 1 : m) + e - first;
    const double two = m == 0 ? 1.0 : 2.0, sg = (m & 1) ? -1.0 : 1.0;
    const double scale = sg * odd_factorial(n);
    double* o = out + (long)e * 2 * NQ;
    double re, im;
    moment(M, n - 1, m, re, im);  // gz = -sum M_{n-1}^m I_n^m, times a
    o[0] = -two * re * scale * q.a;
    o[1] = two * im * scale * q.a;
    if constexpr (NQ == 6) {
      moment(M, n - 2, m, re, im);
      o[2] = two * re * scale;
      o[3] = -two * im * scale;
      for (int d = 2; d >= 1; --d) {  // W = sum M^{mu-2} I^mu, V = -sum M^{mu-1} I^mu
        const double f = d == 2 ? 1.0 : -1.0;
        double pr, pi, nr = 0.0, ni = 0.0;
        moment(M, n - 2, m - d, pr, pi);
        if (m > 0) {
          moment(M, n - 2, -m - d, nr, ni);
          nr *= sg;
          ni *= sg;
        }
        double* v = o + (d == 2 ? 4 : 8);
        v[0] = f * (pr + nr) * scale;
        v[1] = f * (ni - pi) * scale;
        v[2] = f * (pi + ni) * scale;
        v[3] = f * (pr - nr) * scale;
      }
    }
  }
}

// Data, far tiles: a lane has kSites sites (64 apart), a workgroup of four waves walks a chunk of
// tiles.  The tile's coefficients (26 KB, gz 4 KB) go through LDS, the next tile's on their way
// through 128 bytes of scratch a lane for gz + FTG: as scalar loads, which the scalar cache does
// not hold, their latency took twice the rest (2048 tiles and 4096 sites, gz + FTG, degree 16: 0.83
// ms, 1.90 ms with scalar loads, 0.62 ms is the VALU's; degree 20: 1.25 ms).  Orders m outermost,
// so a lane holds one h recurrence and the 2 NQ sums of the order per site: 3 FP64 operations per
// (n, m) for h and 12 (gz: 2) for the sums.  Sums in the corner sums' signs and components:
// partial[model ld + (chunk NC + m) S + s]; grid: z = models.
constexpr int kSites = 2;
// entry of (n, m) in a tile's coefficients
__host__ __device__ constexpr int entry_nm(int n, int m) {
  int e = 0;
  for (int k = 0; k < m; ++k) e += kOrders - (k < 1 ? 1 : k);
  return e + n - (m < 1 ? 1 : m);
}
// Sites of a lane: scaled offset terms, E_m and the sums.
template <int NQ>
struct FarSites {
  double u[kSites], zr[kSites], xu[kSites], yu[kSites], er[kSites], ei[kSites];
  double acc[kSites][NQ];
};
// degrees n = N .. of order M: sums of the coefficients times h_{n,M}
template <int NQ, int M, int N>
__device__ __forceinline__ void far_degrees(const double* __restrict__ cf, const FarSites<NQ>& f,
                                            double (&h)[kSites], double (&hp)[kSites],
                                            double (&sum)[kSites][2 * NQ]) {
  if constexpr (N < (NQ == 1 ? kOrders - 1 : kOrders)) {
    if constexpr (N >= 1) {
      constexpr int e = entry_nm(N, M) * 2 * NQ;
#pragma unroll
      for (int v = 0; v < 2 * NQ; ++v) {
        if (M == 0 && (v & 1)) continue;                 // Im E_0 = 0
        if (v < 2 ? N == kOrders - 1 : N < 2) continue;  // gz ends at kDeg + 1
        const double c = cf[e + v];
#pragma unroll
        for (int i = 0; i < kSites; ++i) sum[i][v] = fma(c, h[i], sum[i][v]);
      }
    }
    constexpr double gamma = gamma_nm(N, M);
#pragma unroll
    for (int i = 0; i < kSites; ++i) {
      const double hn = fma(f.zr[i], h[i], -(gamma * f.u[i]) * hp[i]);
      hp[i] = h[i];
      h[i] = hn;
    }
    far_degrees<NQ, M, N + 1>(cf, f, h, hp, sum);
  }
}
template <int NQ, int M>
__device__ __forceinline__ void far_orders(const double* __restrict__ cf, FarSites<NQ>& f) {
  if constexpr (M < (NQ == 1 ? kOrders - 1 : kOrders)) {
    double sum[kSites][2 * NQ], h[kSites], hp[kSites];  // h_{n,m}, h_{n-1,m}
#pragma unroll
    for (int i = 0; i < kSites; ++i) {
      h[i] = 1.0;
      hp[i] = 0.0;
#pragma unroll
      for (int v = 0; v < 2 * NQ; ++v) sum[i][v] = 0.0;
    }
    far_degrees<NQ, M, M>(cf, f, h, hp, sum);
#pragma unroll
    for (int i = 0; i < kSites; ++i) {
#pragma unroll
      for (int v = 0; v < NQ; ++v) {
        f.acc[i][v] = fma(f.er[i], sum[i][2 * v], f.acc[i][v]);
        if (M > 0) f.acc[i][v] = fma(f.ei[i], sum[i][2 * v + 1], f.acc[i][v]);
      }
      const double nr = fma(f.er[i], f.xu[i], -f.ei[i] * f.yu[i]);
      f.ei[i] = fma(f.er[i], f.yu[i], f.ei[i] * f.xu[i]);
      f.er[i] = nr;
    }
    far_orders<NQ, M + 1>(cf, f);
  }
}

template <int MASK>
__global__ __launch_bounds__(kBlock) void k_tile_far_forward(
    const double* __restrict__ sx, const double* __restrict__ sy, const double* __restrict__ sz,
    int S, const double4* __restrict__ geo, const double* __restrict__ coefs, int ntiles,
    int per, double* __restrict__ partial, long ld) {
  constexpr int NC = Ncomp<MASK>::value;
  constexpr int NQ = MASK == kMaskScalar ? 1 : 6;
  const int s0 = (blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6)) * 64 * kSites +
                 (int)(threadIdx.x & 63);
  coefs += (long)blockIdx.z * ntiles * kNM * 2 * NQ;
  partial += blockIdx.z * ld + (long)blockIdx.y * NC * S;
  constexpr int kPieces = kNM * NQ, kLoads = (kPieces + kBlock - 1) / kBlock;  // of 16 bytes
  __shared__ double2 tile[2][kPieces];
  const bool busy = s0 - (int)(threadIdx.x & 63) < S;  // the wave has sites
  double px[kSites], py[kSites], pz[kSites];
  FarSites<NQ> f;
#pragma unroll
  for (int i = 0; i < kSites; ++i) {
    const int s = min(s0 + 64 * i, S - 1);
    px[i] = sx[s];
    py[i] = sy[s];
    pz[i] = sz[s];
#pragma unroll
    for (int v = 0; v < NQ; ++v) f.acc[i][v] = 0.0;
  }
  const int t0 = blockIdx.y * per, t1 = min(t0 + per, ntiles);
  double2 next[kLoads];
  auto load = [&](int t) {
    const double2* from = reinterpret_cast<const double2*>(coefs) + (long)t * kPieces;
#pragma unroll
    for (int l = 0; l < kLoads; ++l)
      next[l] = from[min(l * kBlock + (int)threadIdx.x, kPieces - 1)];
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int l = 0; l < kLoads; ++l)
      if (l * kBlock + (int)threadIdx.x < kPieces) tile[buf][l * kBlock + threadIdx.x] = next[l];
  };
  load(t0);
  store(0);
  __syncthreads();
  for (int t = t0; t < t1; ++t) {
    const int buf = (t - t0) & 1;
    if (t + 1 < t1) load(t + 1);
    const double4 centre = geo[t];
    bool any = false;
#pragma unroll
    for (int i = 0; i < kSites; ++i) {
      const Offset o = offset_of(px[i], py[i], pz[i], centre);
      const bool far = o.far<MASK>();
      any = any || far;
      f.u[i] = far ? 1.0 / o.r2 : 0.0;  // near: every E is zero
      f.zr[i] = far ? o.z * f.u[i] : 0.0;
      f.xu[i] = far ? o.x * f.u[i] : 0.0;
      f.yu[i] = far ? o.y * f.u[i] : 0.0;
      f.er[i] = sqrt(f.u[i]);  // E_0
      f.ei[i] = 0.0;
    }
    if (busy && __any(any)) far_orders<NQ, 0>(reinterpret_cast<const double*>(tile[buf]), f);
    if (t + 1 < t1) store(buf ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < kSites; ++i) {
    const int s = s0 + 64 * i;
    if (s >= S) continue;
    double out[NC];
    out[0] = -f.acc[i][0];
    if constexpr (NQ == 6) {  // Uzz, Uxx - Uyy, 2 Uxy, Uxz, Uyz -> xx, yy, zz, -xy, -xz, -yz
      out[1] = 0.5 * (f.acc[i][2] - f.acc[i][1]);
      out[2] = -0.5 * (f.acc[i][2] + f.acc[i][1]);
      out[3] = f.acc[i][1];
      out[4] = -0.5 * f.acc[i][3];
      out[5] = -f.acc[i][4];
      out[6] = -f.acc[i][5];
    }
#pragma unroll
    for (int m = 0; m < NC; ++m) partial[(long)m * S + s] = out[m];
  }
}

// Data, near tiles: a workgroup per site (and split of the tiles); its waves test 64 tiles at a
// time and share the corners of each near one (tiles dealt to the waves instead left half of
// them idle: the near ones of a site lie in few runs of 64).  NB models share the corner terms.
// Sums to row `split` of partial.
template <int MASK, int NB>
__global__ __launch_bounds__(kBlock) void k_tile_near_forward(
    const double* __restrict__ sx, const double* __restrict__ sy, const double* __restrict__ sz,
    int S, TileGrid g, const double4* __restrict__ geo, const double* __restrict__ wt, int ntiles,
    double* __restrict__ partial, long ld) {
  constexpr int NC = Ncomp<MASK>::value;
  constexpr int W = kBlock / 64;
  __shared__ LogTableShared tab;
  __shared__ double red[NB * NC][W];
  const LogTable lg = tab.fill();
  const int s = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const double px = sx[s], py = sy[s], pz = sz[s];
  double acc[NB * NC];
#pragma unroll
  for (int m = 0; m < NB * NC; ++m) acc[m] = 0.0;
  for (int b = (int)blockIdx.y * 64; b < ntiles; b += (int)gridDim.y * 64) {
    bool near = false;
    if (b + lane < ntiles) near = !offset_of(px, py, pz, geo[b + lane]).far<MASK>();
    unsigned long long mask = __ballot(near);
    while (mask) {
      const int t = b + __builtin_ctzll(mask);
      mask &= mask - 1;
      const int k = t % g.tz, ij = t / g.tz, j = ij % g.ty, i = ij / g.ty;
      const double* w = wt + (long)t * kTCorners;
      for (int q = threadIdx.x; q < kTCorners; q += kBlock) {
        // corners past the mesh's end carry no weight
        const int K = min(k * kT + q % kTC, g.nz), J = min(j * kT + q / kTC % kTC, g.ny);
        const int I = min(i * kT + q / (kTC * kTC), g.nx);
        double v[NC];
        corner_terms_f64<MASK>(px - g.Xc[I], py - g.Yc[J], pz - g.Zc[K], v, lg);
#pragma unroll
        for (int n = 0; n < NB; ++n) {
          const double wn = w[(long)n * ntiles * kTCorners + q];
#pragma unroll
          for (int m = 0; m < NC; ++m) acc[n * NC + m] = fma(wn, v[m], acc[n * NC + m]);
        }
      }
    }
  }
#pragma unroll
  for (int m = 0; m < NB * NC; ++m) {
    double v = acc[m];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if (lane == 0) red[m][wave] = v;
  }
  __syncthreads();
  if (threadIdx.x < NB * NC) {
    const int m = threadIdx.x;
    double v = 0.0;
    for (int x = 0; x < W; ++x) v += red[m][x];
    partial[m / NC * ld + ((long)blockIdx.y * NC + m % NC) * S + s] = v;
  }
}

// Gradient, near tiles: thread = corner of the workgroup's tile; each wave tests 64 sites at a
// time and sums coef F over the near ones.  NB residual sets (coef[(set S + s) NC + m]) share the
// corner terms.  H[((split NB + set) ntiles + t) kTCorners + corner].
constexpr int kNearThreads = 768;
template <int MASK, int NB>
__global__ __launch_bounds__(kNearThreads) void k_tile_near_adjoint(
    const double* __restrict__ sx, const double* __restrict__ sy, const double* __restrict__ sz,
    int S, const double* __restrict__ coef, TileGrid g, const double4* __restrict__ geo,
    int ntiles, double* __restrict__ H) {
  constexpr int NC = Ncomp<MASK>::value;
  __shared__ LogTableShared tab;
  const LogTable lg = tab.fill();
  const int t = tile_of_block(g, blockIdx.x), lane = threadIdx.x & 63;
  const int q = min((int)threadIdx.x, kTCorners - 1);
  const int tk = t % g.tz, ij = t / g.tz, tj = ij % g.ty, ti = ij / g.ty;
  const double cx = g.Xc[min(ti * kT + q / (kTC * kTC), g.nx)];
  const double cy = g.Yc[min(tj * kT + q / kTC % kTC, g.ny)];
  const double cz = g.Zc[min(tk * kT + q % kTC, g.nz)];
  const double4 centre = geo[t];
  double h[NB];
#pragma unroll
  for (int n = 0; n < NB; ++n) h[n] = 0.0;
  for (int b = (int)blockIdx.y * 64; b < S; b += (int)gridDim.y * 64) {
    bool near = false;
    if (b + lane < S) near = !offset_of(sx[b + lane], sy[b + lane], sz[b + lane], centre).far<MASK>();
    unsigned long long mask = __ballot(near);
    while (mask) {
      const int s = __builtin_amdgcn_readfirstlane(b + __builtin_ctzll(mask));
      mask &= mask - 1;
      double v[NC];
      corner_terms_f64<MASK>(sx[s] - cx, sy[s] - cy, sz[s] - cz, v, lg);
#pragma unroll
      for (int n = 0; n < NB; ++n) {
        const double* cs = coef + ((long)n * S + s) * NC;
#pragma unroll
        for (int m = 0; m < NC; ++m) h[n] = fma(cs[m], v[m], h[n]);
      }
    }
  }
  if ((int)threadIdx.x < kTCorners)
#pragma unroll
    for (int n = 0; n < NB; ++n)
      H[(((long)blockIdx.y * NB + n) * ntiles + t) * kTCorners + threadIdx.x] = h[n];
}

// One h recurrence of order MU (none for MU < 0): value at the current n and at n - 1.
template <int MU>
struct Recur {
  double h = 1.0, hp = 0.0;
  template <int N>
  __device__ __forceinline__ void step(double zr, double u) {  // n = N -> N + 1
    const double hn = fma(zr, h, -(gamma_nm(N, MU) * u) * hp);
    hp = h;
    h = hn;
  }
  template <int FROM, int TO>
  __device__ __forceinline__ void advance(double zr, double u) {
    if constexpr (FROM < TO) {
      step<FROM>(zr, u);
      advance<FROM + 1, TO>(zr, u);
    }
  }
};

// The degrees l = L .. kDeg of order m = M of one site's local coefficients: G_l and T_l.
template <int MASK, int M, int L, class R0, class Rm2, class Rm1, class R, class Rp1, class Rp2>
__device__ __forceinline__ void local_degrees(const double* q0, const double (&tm)[5][2], double zr,
                                              double u, R0& g0, Rm2& m2, Rm1& m1, R& r0, Rp1& p1,
                                              Rp2& p2, double (&G)[kK][2], double (&T)[kK][2]) {
  if constexpr (L <= kDeg) {
    // g0 at n = L + 1, the others at n = L + 2
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      if (M == 0 && c == 1) continue;
      G[L - M][c] = fma(q0[c], g0.h, G[L - M][c]);
      if constexpr (MASK != kMaskScalar) {
        double v = T[L - M][c];
        if constexpr (M >= 2) v = fma(tm[0][c], m2.h, v);
        if constexpr (M >= 1) v = fma(tm[1][c], m1.h, v);
        v = fma(tm[2][c], r0.h, v);
        v = fma(tm[3][c], p1.h, v);
        T[L - M][c] = fma(tm[4][c], p2.h, v);
      }
    }
    if constexpr (L < kDeg) {
      g0.template step<L + 1>(zr, u);
      if constexpr (MASK != kMaskScalar) {
        if constexpr (M >= 2) m2.template step<L + 2>(zr, u);
        if constexpr (M >= 1) m1.template step<L + 2>(zr, u);
        r0.template step<L + 2>(zr, u);
        p1.template step<L + 2>(zr, u);
        p2.template step<L + 2>(zr, u);
      }
      local_degrees<MASK, M, L + 1>(q0, tm, zr, u, g0, m2, m1, r0, p1, p2, G, T);
    }
  }
}

// Sums of n values over the wave's 64 lanes, one or none to a lane: at each step a lane passes
// half of its values to its partner and adds the partner's to the other half (44 exchanges for
// the 42 values of order 0; each value by itself takes 252, and the far gradient of 2048 tiles and
// 256 sites, degree 16, 0.45 ms instead of 0.23).  The same additions as a butterfly of each value.
// The lane's sum ends in v[0]; returns its index, -1 for none.
template <int N, int OFF = 32>
__device__ __forceinline__ int sum_lanes(double* v, int lane) {
  constexpr int half = (N + 1) / 2;
  const bool upper = (lane & OFF) != 0;
#pragma unroll
  for (int i = 0; i < half; ++i) {
    const double a = v[i], b = i + half < N ? v[i + half] : 0.0;
    v[i] = (upper ? b : a) + __shfl_xor(upper ? a : b, OFF, 64);
  }
  int at = 0;
  if constexpr (OFF > 1) at = sum_lanes<half, OFF / 2>(v, lane);
  if (at >= 0 && upper) at = at + half < N ? at + half : -1;
  return at;
}

// Gradient, far tiles, order M: lane = site, the workgroup's four waves stride through the
// survey 64 sites at a time; the lane keeps the order's local coefficients (G for gz, T for the
// tensor) of the tile over its sites, and lanes and waves are added once at the end.
template <int MASK, int M>
__device__ inline void far_adjoint_order(const double* __restrict__ sx,
                                         const double* __restrict__ sy,
                                         const double* __restrict__ sz, int S,
                                         const double* __restrict__ coef, double4 centre,
                                         double (*red)[2 * kK], double* __restrict__ lam) {
  constexpr int NC = Ncomp<MASK>::value;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  double G[kK][2], T[kK][2];
#pragma unroll
  for (int l = 0; l < kK; ++l)
#pragma unroll
    for (int c = 0; c < 2; ++c) G[l][c] = T[l][c] = 0.0;
  const double a = 1.0 / centre.w;
  for (int b = wave * 64; b < S; b += kBlock) {
    const int s = min(b + lane, S - 1);
    Offset o = offset_of(sx[s], sy[s], sz[s], centre);
    const bool far = b + lane < S && o.far<MASK>();
    if (__ballot(far) == 0) continue;
    double c7[7];
#pragma unroll
    for (int m = 0; m < NC; ++m) c7[m] = far ? coef[(long)s * NC + m] : 0.0;
    if (!far) {  // any far offset: the coefficients are zero
      o.x = 0.0;
      o.y = 0.0;
      o.z = kRatio<MASK>;
      o.r2 = kRatio<MASK> * kRatio<MASK>;
    }
    const double u = 1.0 / o.r2, zr = o.z * u, xu = o.x * u, yu = o.y * u;
    double E[M + 3][2];  // E_0 .. E_{M+2}
    E[0][0] = sqrt(u);
    E[0][1] = 0.0;
#pragma unroll
    for (int k = 0; k < M + 2; ++k) {
      E[k + 1][0] = fma(E[k][0], xu, -E[k][1] * yu);
      E[k + 1][1] = fma(E[k][0], yu, E[k][1] * xu);
    }
    constexpr double two = M == 0 ? 1.0 : 2.0, sg = (M & 1) ? -1.0 : 1.0;
    const double cz = -a * c7[0];  // corner sum of gz: -a times the harmonic sum's gz
    const double q0[2] = {-two * sg * cz * E[M][0], -two * sg * cz * E[M][1]};
    double tm[5][2] = {};
    Recur<M> g0, r0;
    Recur<(M >= 2 ? M - 2 : 0)> m2;
    Recur<(M >= 1 ? M - 1 : 0)> m1;
    Recur<M + 1> p1;
    Recur<M + 2> p2;
    g0.template advance<M, M + 1>(zr, u);
    if constexpr (MASK != kMaskScalar) {
      // value = zeta Uzz + Re(lambda W) + Re(kappa V); the off-diagonal corner sums carry -1
      const double zeta = c7[3] - 0.5 * (c7[1] + c7[2]);
      const double lr = 0.5 * (c7[1] - c7[2]), li = 0.5 * c7[4];  // (xx - yy)/2 - i xy/2
      const double kr = -c7[5], ki = c7[6];                       // xz - i yz
      tm[2][0] = two * sg * zeta * E[M][0];
      tm[2][1] = two * sg * zeta * E[M][1];
      // -kappa I^{M+1}
      tm[3][0] = sg * fma(kr, E[M + 1][0], -ki * E[M + 1][1]);
      tm[3][1] = sg * fma(kr, E[M + 1][1], ki * E[M + 1][0]);
      // lambda I^{M+2}
      tm[4][0] = sg * fma(lr, E[M + 2][0], -li * E[M + 2][1]);
      tm[4][1] = sg * fma(lr, E[M + 2][1], li * E[M + 2][0]);
      if constexpr (M >= 1) {  // conj(kappa) I^{M-1}
        tm[1][0] = -sg * fma(kr, E[M - 1][0], ki * E[M - 1][1]);
        tm[1][1] = -sg * fma(kr, E[M - 1][1], -ki * E[M - 1][0]);
      }
      if constexpr (M == 1) {  // -conj(lambda I^1), on the same h as Uzz
        tm[2][0] += fma(lr, E[1][0], -li * E[1][1]);
        tm[2][1] -= fma(lr, E[1][1], li * E[1][0]);
      }
      if constexpr (M >= 2) {  // conj(lambda) I^{M-2}
        tm[0][0] = sg * fma(lr, E[M - 2][0], li * E[M - 2][1]);
        tm[0][1] = sg * fma(lr, E[M - 2][1], -li * E[M - 2][0]);
        m2.template advance<M - 2, M + 2>(zr, u);
      }
      if constexpr (M >= 1) m1.template advance<M - 1, M + 2>(zr, u);
      r0.template advance<M, M + 2>(zr, u);
      p1.template advance<M + 1, M + 2>(zr, u);
    }
    local_degrees<MASK, M, M>(q0, tm, zr, u, g0, m2, m1, r0, p1, p2, G, T);
  }
  constexpr int count = 2 * (kK - M);
  double v[count];
#pragma unroll
  for (int l = M; l < kK; ++l)
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      v[2 * (l - M) + c] = odd_factorial(l + 1) * G[l - M][c];
      if constexpr (MASK != kMaskScalar)
        v[2 * (l - M) + c] = fma(odd_factorial(l + 2), T[l - M][c], v[2 * (l - M) + c]);
    }
  if (wave * 64 < S) {
    const int e = sum_lanes<count>(v, lane);
    if (e >= 0) red[wave][e] = v[0];
  }
  __syncthreads();
  const int waves = min(kBlock / 64, (S + 63) / 64);  // the ones with sites
  for (int e = threadIdx.x; e < count; e += kBlock) {
    double sum = 0.0;
    for (int w = 0; w < waves; ++w) sum += red[w][e];
    lam[2 * lm_index(M + e / 2, M) + e % 2] = sum;
  }
}

template <int MASK, int M>
__device__ inline void far_adjoint_select(int m, const double* __restrict__ sx,
                                          const double* __restrict__ sy,
                                          const double* __restrict__ sz, int S,
                                          const double* __restrict__ coef, double4 centre,
                                          double (*red)[2 * kK], double* __restrict__ lam) {
  if (m == M) {
    far_adjoint_order<MASK, M>(sx, sy, sz, S, coef, centre, red, lam);
  } else if constexpr (M < kDeg) {
    far_adjoint_select<MASK, M + 1>(m, sx, sy, sz, S, coef, centre, red, lam);
  }
}

// grid: x = tiles, y = orders m, z = residual sets
template <int MASK>
__global__ __launch_bounds__(kBlock) void k_tile_far_adjoint(
    const double* __restrict__ sx, const double* __restrict__ sy, const double* __restrict__ sz,
    int S, const double* __restrict__ coef, TileGrid g, const double4* __restrict__ geo,
    double* __restrict__ lam) {
  __shared__ double red[kBlock / 64][2 * kK];
  const int t = tile_of_block(g, blockIdx.x);
  far_adjoint_select<MASK, 0>((int)blockIdx.y, sx, sy, sz, S,
                              coef + (long)blockIdx.z * S * Ncomp<MASK>::value, geo[t], red,
                              lam + ((long)blockIdx.z * gridDim.x + t) * kRows);
}

// Local coefficients -> monomials -> the cells' integrals, plus the near corner sums'
// differences: the tile's cells of the gradient.  grid: x = tiles, y = residual sets.
__global__ __launch_bounds__(kBlock) void k_tile_gradient(TileGrid g, const double* __restrict__ lam,
                                                          HarmonicTable h,
                                                          const double* __restrict__ H, int splits,
                                                          int ntiles, double* __restrict__ grad,
                                                          long ld) {
  __shared__ double ax[3][kT][kK];
  __shared__ double L[kRows];
  __shared__ double mu[kMono];
  __shared__ double A[kK][kT * kT];
  __shared__ double B[kPairs][kT];
  __shared__ double hs[kTCorners];
  const int t = blockIdx.x;
  lam += (long)blockIdx.y * ntiles * kRows;
  H += (long)blockIdx.y * ntiles * kTCorners;
  grad += blockIdx.y * ld;
  const Tile q = tile_of(g, t);
  axis_moments(g, q, ax);
  for (int r = threadIdx.x; r < kRows; r += kBlock) L[r] = lam[(long)t * kRows + r];
  for (int e = threadIdx.x; e < kTCorners; e += kBlock)
    hs[e] = sum_strided(0.0, H + (long)t * kTCorners + e, splits,
                        (long)gridDim.y * ntiles * kTCorners);
  __syncthreads();
  for (int e = threadIdx.x; e < kMono; e += kBlock) {
    double s = 0.0;
    for (int c = h.cptr[e]; c < h.cptr[e + 1]; ++c) s = fma(h.cval[c], L[h.cidx[c]], s);
    mu[h.mono[kMono + e]] = s;
  }
  __syncthreads();
  // mu is now ordered (c, b, a): the pair (b, c) starts at h.mono[2 kMono + bc]
  for (int e = threadIdx.x; e < kK * kK * kT; e += kBlock) {
    const int i = e % kT, b = e / kT % kK, c = e / (kT * kK);
    if (b + c > kDeg) continue;
    const int bc = bc_index(b, c), at = h.mono[2 * kMono + bc];
    double s = 0.0;
    for (int a = 0; a <= kDeg - b - c; ++a) s = fma(mu[at + a], ax[0][i][a], s);
    B[bc][i] = s;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < kK * kT * kT; e += kBlock) {
    const int j = e % kT, i = e / kT % kT, c = e / (kT * kT);
    double s = 0.0;
    for (int b = 0; b <= kDeg - c; ++b) s = fma(B[bc_index(b, c)][i], ax[1][j][b], s);
    A[c][i * kT + j] = s;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < kT * kT * kT; e += kBlock) {
    const int k = e % kT, j = e / kT % kT, i = e / (kT * kT);
    if (i >= q.ni || j >= q.nj || k >= q.nk) continue;
    double far = 0.0;
    for (int c = 0; c < kK; ++c) far = fma(A[c][i * kT + j], ax[2][k][c], far);
    double near = 0.0;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const double v = hs[((i + a) * kTC + j + b) * kTC + k + c];
          near += ((a + b + c) & 1) ? v : -v;
        }
    grad[((long)(q.i0 + i) * g.ny + (q.j0 + j)) * g.nz + q.k0 + k] = 2.0 * (near + far);
  }
}

// Harmonic polynomials Re R_l^m, Im R_l^m as sparse rows over the monomials, and the transpose.
struct HarmonicPolynomials {
  std::vector<int> ptr, idx, cptr, cidx, mono;
  std::vector<double> val, cval;
  HarmonicPolynomials() {
    typedef std::complex<long double> C;
    // monomial (a, b, c) of degree d = a + b + c: degrees in turn, then c, then b
    auto local = [](int d, int b, int c) { return c * (d + 1) - c * (c - 1) / 2 + b; };
    std::vector<int> base(kK + 1, 0);
    for (int d = 0; d <= kDeg; ++d) base[d + 1] = base[d] + (d + 1) * (d + 2) / 2;
    mono.assign(2 * kMono + kPairs, 0);
    std::vector<int> start(kPairs, 0);
    int at = 0;
    for (int c = 0; c <= kDeg; ++c)
      for (int b = 0; b + c <= kDeg; ++b) {
        start[c * kK - c * (c - 1) / 2 + b] = at;
        at += kDeg - b - c + 1;
      }
    for (int d = 0; d <= kDeg; ++d)
      for (int c = 0; c <= d; ++c)
        for (int b = 0; b + c <= d; ++b) {
          const int e = base[d] + local(d, b, c), a = d - b - c;
          mono[e] = a | b << 8 | c << 16;
          mono[kMono + e] = start[c * kK - c * (c - 1) / 2 + b] + a;  // (c, b, a) order
        }
    for (int p = 0; p < kPairs; ++p) mono[2 * kMono + p] = start[p];
    // to += f y^db z^dc x^(rest) from, a polynomial of degree fd raised to degree d
    auto add = [&](std::vector<C>& to, int d, const std::vector<C>& from, int fd, int db, int dc,
                   C f) {
      for (int c = 0; c <= fd; ++c)
        for (int b = 0; b + c <= fd; ++b)
          to[local(d, b + db, c + dc)] += f * from[local(fd, b, c)];
    };
    std::vector<std::vector<C>> R(kPairs);
    for (int m = 0; m <= kDeg; ++m) {
      for (int l = m; l <= kDeg; ++l) {
        std::vector<C>& r = R[lm_index(l, m)];
        r.assign((l + 1) * (l + 2) / 2, C(0));
        if (l == 0) {
          r[0] = C(1);
        } else if (l == m) {
          const C f = C(-1.0L / (2 * m));
          add(r, l, R[lm_index(m - 1, m - 1)], m - 1, 0, 0, f);
          add(r, l, R[lm_index(m - 1, m - 1)], m - 1, 1, 0, f * C(0, 1));
        } else {
          const long double den = (long double)(l + m) * (l - m);
          add(r, l, R[lm_index(l - 1, m)], l - 1, 0, 1, C((2 * l - 1) / den));
          if (l >= m + 2) {
            const std::vector<C>& q = R[lm_index(l - 2, m)];
            add(r, l, q, l - 2, 0, 0, C(-1 / den));
            add(r, l, q, l - 2, 2, 0, C(-1 / den));
            add(r, l, q, l - 2, 0, 2, C(-1 / den));
          }
        }
      }
    }
    std::vector<std::vector<std::pair<int, double>>> cols(kMono);
    ptr.push_back(0);
    for (int l = 0; l <= kDeg; ++l)
      for (int m = 0; m <= l; ++m)
        for (int part = 0; part < 2; ++part) {
          const std::vector<C>& r = R[lm_index(l, m)];
          const int row = 2 * lm_index(l, m) + part;
          for (size_t e = 0; e < r.size(); ++e) {
            const double v = (double)(part ? r[e].imag() : r[e].real());
            if (v == 0.0) continue;
            idx.push_back(base[l] + (int)e);
            val.push_back(v);
            cols[base[l] + e].push_back({row, v});
          }
          ptr.push_back((int)idx.size());
        }
    cptr.push_back(0);
    for (const auto& c : cols) {
      for (const auto& e : c) {
        cidx.push_back(e.first);
        cval.push_back(e.second);
      }
      cptr.push_back((int)cidx.size());
    }
  }
};

// The tables as one block: val, cval, then ptr, idx, cptr, cidx, mono.  They hold numbers of the
// method only, so a process makes them once (a new context of a small mesh, first data and
// gradient, at degree 16: 0.36 ms, 0.89 ms when each context made them, in seven buffers).
struct HarmonicBlock {
  size_t at[7];
  std::vector<char> bytes;
  HarmonicBlock() {
    const HarmonicPolynomials p;
    add(0, p.val);
    add(1, p.cval);
    add(2, p.ptr);
    add(3, p.idx);
    add(4, p.cptr);
    add(5, p.cidx);
    add(6, p.mono);
  }
  template <class V>
  void add(int which, const std::vector<V>& v) {
    at[which] = bytes.size();
    const char* from = reinterpret_cast<const char*>(v.data());
    bytes.insert(bytes.end(), from, from + sizeof(V) * v.size());
  }
};
const HarmonicBlock& harmonic_block() {
  static const HarmonicBlock b;
  return b;
}

TileGrid tile_grid(const jgm_context* ctx) {
  TileGrid g;
  g.Xc = ctx->d_Xc.as<const double>();
  g.Yc = ctx->d_Yc.as<const double>();
  g.Zc = ctx->d_Zc.as<const double>();
  g.nx = (int)ctx->nx;
  g.ny = (int)ctx->ny;
  g.nz = (int)ctx->nz;
  g.tx = (g.nx + kT - 1) / kT;
  g.ty = (g.ny + kT - 1) / kT;
  g.tz = (g.nz + kT - 1) / kT;
  return g;
}

// How a geometry's sums are split.  None of it depends on the number of models, whose sums must
// not either.
struct TilePlan {
  int ntiles, far_blocks, far_per, far_chunks;  // data, far: workgroups of sites, tiles a chunk
  int near_splits;                              // data, near: rows of a site's sum
  int adj_splits;                               // gradient, near: rows of a corner's sum
};
TilePlan tile_plan(const jgm_context* ctx) {
  const TileGrid g = tile_grid(ctx);
  const int S = (int)ctx->S;
  TilePlan p;
  p.ntiles = g.tx * g.ty * g.tz;
  // chunks of tiles for about 16 waves per SIMD
  p.far_blocks = (int)blocks_for((S + kSites - 1) / kSites);
  const int want = std::max(1, std::min(p.ntiles, 16 * ctx->cu_count / p.far_blocks));
  p.far_per = (p.ntiles + want - 1) / want;
  p.far_chunks = (p.ntiles + p.far_per - 1) / p.far_per;
  // a split per 1024 sites short of filling the CUs
  p.near_splits = std::max(1, std::min(8, 2048 / S));
  // for 8192 workgroups and more; beyond that a split only costs memory and the log tables again
  // (gz, 512 x 512 x 64 cells and 1024 sites: near gradient 1.47 ms in four, 0.97 in one)
  p.adj_splits = std::max(1, std::min(std::min(4, S / 256), 8192 / p.ntiles));
  return p;
}

// Bytes of the buffers of a model's data and gradient: coefficients, corner weights and partial
// sums; local expansions and corner sums.  (gz + FTG of 128 x 128 x 64 cells and 4096 sites: 54, 12
// and 118 MB, 8 and 48 MB.)
size_t tile_bytes(const jgm_context* ctx, const TilePlan& p, bool tensor) {
  const size_t tile = (size_t)kNM * (tensor ? 12 : 2) + kTCorners + kRows +
                      (size_t)p.adj_splits * kTCorners;
  const size_t row = (size_t)(tensor ? 7 : 1) * ctx->S;
  return sizeof(double) * (p.ntiles * tile + (p.far_chunks + p.near_splits + 1) * row);
}

HarmonicTable harmonic_table(const jgm_context* ctx) {
  const size_t* at = harmonic_block().at;
  const char* base = ctx->tile_far.table.as<const char>();
  auto ints = [&](int which) { return reinterpret_cast<const int*>(base + at[which]); };
  auto doubles = [&](int which) { return reinterpret_cast<const double*>(base + at[which]); };
  return {ints(2), ints(3), ints(4), ints(5), ints(6), doubles(0), doubles(1)};
}

// Whether the geometry takes the expansions.  A batch's results are the single call's bit for bit,
// so the choice must not depend on the batch; with more models the closed form gains, whose corner
// terms all share, where the expansions share only the near ones.  The line is where three models
// at a time, data and gradient, take the same: on it one takes 0.4 to 0.7 of the closed form's time
// and eight up to a third more (gz + FTG, 128 x 128 x 64 cells, 100 stations: 0.93 against 2.19 ms
// for one model, 1.63 and 2.28 for two, 2.94 and 2.68 for four, 5.43 and 4.18 for eight).
bool choose(const jgm_context* ctx, bool tensor) {
  const long N = (long)ncells(ctx), S = (long)ctx->S;
  // 48 x 48 x 24 cells, where most tiles are near, lose (gz of 625 sites, four models 0.68 ms,
  // closed form 0.55), 128 x 64 x 8 win (4096 sites 1.4 and 2.6 ms)
  if (N < 60000 || S < 64) return false;
  // increasing corner coordinates (the tiles' boxes)
  const std::vector<double>* C[3] = {&ctx->xc, &ctx->yc, &ctx->zc};
  for (const auto* c : C)
    for (size_t i = 1; i < c->size(); ++i)
      if (!((*c)[i] > (*c)[i - 1])) return false;
  // No station on or next to a mesh line.  Of the corners down a line at distance
  // rho, those at u < 0 along it have log(u + r), u + r = rho^2 / 2|u|, formed with an ulp of |u|:
  // guarded or a few ulps where rho is small, not the field but what the reference computes, and
  // tiles that are expanded would give the field instead.  At rho = 2^-18 of the farthest |u| (5 mm
  // for 1.3 km) the argument keeps 15 bits and the closed form is the field with some noise.
  // gz has the logarithms of the horizontal lines only, times the offset from the line, without
  // the guard: not a number on the line (as the reference's), 1e-8 of gz a micrometre beside it.
  const std::vector<double>* P[3] = {&ctx->hsx, &ctx->hsy, &ctx->hsz};
  auto plane = [&](int a, long s) {  // distance to the nearest corner plane
    const double v = (*P[a])[s];
    const auto up = std::lower_bound(C[a]->begin(), C[a]->end(), v);
    const double above = up != C[a]->end() ? *up - v : HUGE_VAL;
    return up != C[a]->begin() ? std::min(above, v - up[-1]) : above;
  };
  auto ahead = [&](int a, long s) { return std::max(0.0, C[a]->back() - (*P[a])[s]); };
  for (long s = 0; s < S; ++s) {
    const double ux = ahead(0, s), uy = ahead(1, s), dz = plane(2, s);
    if (!tensor && dz > 0x1p-18 * std::max(ux, uy)) continue;
    const double dx = plane(0, s), dy = plane(1, s);
    if (dy * dy + dz * dz <= 0x1p-36 * ux * ux || dx * dx + dz * dz <= 0x1p-36 * uy * uy)
      return false;
    const double uz = tensor ? ahead(2, s) : 0.0;
    if (tensor && dx * dx + dy * dy <= 0x1p-36 * uz * uz) return false;
  }
  // near tiles of a sample of stations
  std::vector<double> centre[3], half2[3];
  for (int a = 0; a < 3; ++a) {
    const long n = (long)C[a]->size() - 1;
    for (long i = 0; i < n; i += kT) {
      const double lo = (*C[a])[i], hi = (*C[a])[std::min(n, i + kT)];
      centre[a].push_back(0.5 * (lo + hi));
      half2[a].push_back(0.25 * (hi - lo) * (hi - lo));
    }
  }
  const double ratio = tensor ? kRatio<kMaskAll> : kRatio<kMaskScalar>;
  const double tiles = (double)centre[0].size() * centre[1].size() * centre[2].size();
  // a launch dimension ends at 2^32 threads: a workgroup per site, and one per tile
  if (S * kBlock >= 1L << 32 || tiles * kNearThreads >= 0x1p32) return false;
  const long samples = std::min<long>(S, 16);
  double near = 0.0;
  for (long f = 0; f < samples; ++f) {
    const long s = (2 * f + 1) * S / (2 * samples);
    for (size_t i = 0; i < centre[0].size(); ++i)
      for (size_t j = 0; j < centre[1].size(); ++j)
        for (size_t k = 0; k < centre[2].size(); ++k) {
          const double dx = ctx->hsx[s] - centre[0][i], dy = ctx->hsy[s] - centre[1][j],
                       dz = ctx->hsz[s] - centre[2][k];
          near += dx * dx + dy * dy + dz * dz <
                  ratio * ratio * (half2[0][i] + half2[1][j] + half2[2][k]);
        }
  }
  near /= samples;
  // In the closed form's FP64 operations per site, data and gradient averaged: corner terms 250
  // (gz 170) and three models' sums on them, 6950 (2750) per far tile and model.  The near kernels
  // take 1.9 times as long per operation, the far ones 1.8 (2.9) times; a tile of a model its
  // moments, the cells' gradients and the ends of its sums over the sites, as 2.45 (1.45) million
  // operations; the launches and the waves they leave idle 7 to 11 thousand million.  Fitted to
  // 26 geometries of 128 x 128 x 64 to 48 x 48 x 24 cells and 36 to 4096 sites (four models, gz +
  // FTG, tiles against the closed form: 128 x 128 x 64 cells and 1024 sites 7.9 and 17.3 ms, 256
  // sites 3.3 and 4.7, 64 sites 2.8 and 1.8; 64 x 64 x 32 cells and 4096 sites 7.7 and 9.1, 1024
  // sites 2.5 and 2.5, 256 sites 1.2 and 0.9).
  const double term = tensor ? 250.0 + 21.0 : 170.0 + 3.0;
  const double far_tile = tensor ? 1.8 * 6950.0 : 2.9 * 2750.0, ends = tensor ? 2.45e6 : 1.45e6;
  const double closed = (double)ncorners(ctx) * term + (tensor ? 6.6e9 : 11.5e9) / (double)S;
  const double split = 1.9 * near * kTCorners * term + 3.0 * (tiles - near) * far_tile +
                       (3.0 * tiles * ends + (tensor ? 8.2e9 : 11.0e9)) / (double)S;
  // (one model's buffers take 42 KB a tile with the tensor: 64 GiB is 800 million cells)
  return split < closed && tile_bytes(ctx, tile_plan(ctx), tensor) <= (size_t)64 << 30;
}

// The calls of a launch over nb in {1, 2, 4, 8} models, nb a template argument.
template <class F>
void with_models(int nb, F&& f) {
  switch (nb) {
    case 8: f(std::integral_constant<int, 8>()); break;
    case 4: f(std::integral_constant<int, 4>()); break;
    case 2: f(std::integral_constant<int, 2>()); break;
    default: f(std::integral_constant<int, 1>()); break;
  }
}

template <int MASK>
hipError_t forward_partials(jgm_context* ctx, int nb, const double* models, size_t model_ld,
                            double** partial, int* nchunks) {
  constexpr int NC = Ncomp<MASK>::value;
  constexpr int NQ = MASK == kMaskScalar ? 1 : 6;
  TileFar& f = ctx->tile_far;
  hipStream_t st = ctx->stream;
  const TileGrid g = tile_grid(ctx);
  const TilePlan p = tile_plan(ctx);
  const int ntiles = p.ntiles, S = (int)ctx->S, far_chunks = p.far_chunks, splits = p.near_splits;
  hipError_t e;
  if ((e = f.coefs.ensure(sizeof(double) * (size_t)nb * ntiles * kNM * 2 * NQ)) != hipSuccess ||
      (e = f.wt.ensure(sizeof(double) * (size_t)nb * ntiles * kTCorners)) != hipSuccess ||
      (e = f.ref.ensure(sizeof(double) * 8)) != hipSuccess ||
      (e = ctx->partial.ensure(sizeof(double) * (size_t)(far_chunks + splits + 1) * nb * NC * S)) !=
          hipSuccess)
    return e;
  const double *sx = ctx->d_sx.as<const double>(), *sy = ctx->d_sy.as<const double>(),
               *sz = ctx->d_sz.as<const double>();
  const long row = (long)NC * S, ld = (far_chunks + splits + 1) * row;  // of a model
  double* part = ctx->partial.as<double>();
  {
    ProfScope ps(ctx, "tile_moments_fp64");
    hipLaunchKernelGGL(k_reference_density, dim3(nb), dim3(1024), 0, st, models, (long)model_ld,
                       (long)ncells(ctx), f.ref.as<double>());
    hipLaunchKernelGGL((k_reference_box<MASK>), dim3(blocks_for(S)), dim3(kBlock), 0, st, sx, sy, sz,
                       S, g, f.ref.as<const double>(), nb, part + (far_chunks + splits) * row, ld);
    hipLaunchKernelGGL((k_tile_moments<MASK>), dim3(ntiles, nb), dim3(kBlock), 0, st, g, ntiles,
                       models, (long)model_ld, f.ref.as<const double>(), harmonic_table(ctx),
                       f.coefs.as<double>(), f.wt.as<double>());
  }
  {
    ProfScope ps(ctx, "tile_far_forward_fp64");
    hipLaunchKernelGGL((k_tile_far_forward<MASK>), dim3(p.far_blocks, far_chunks, nb), dim3(kBlock),
                       0, st, sx, sy, sz, S, f.geo.as<const double4>(),
                       f.coefs.as<const double>(), ntiles, p.far_per, part, ld);
  }
  {
    ProfScope ps(ctx, "tile_near_forward_fp64");
    with_models(nb, [&](auto n) {
      hipLaunchKernelGGL((k_tile_near_forward<MASK, decltype(n)::value>), dim3(S, splits),
                         dim3(kBlock), 0, st, sx, sy, sz, S, g, f.geo.as<const double4>(),
                         f.wt.as<const double>(), ntiles, part + far_chunks * row, ld);
    });
  }
  *partial = part;
  *nchunks = far_chunks + splits + 1;
  return hipGetLastError();
}

template <int MASK>
hipError_t adjoint_cells(jgm_context* ctx, int nb, const double* coef, double* grads,
                         size_t grad_ld) {
  TileFar& f = ctx->tile_far;
  hipStream_t st = ctx->stream;
  const TileGrid g = tile_grid(ctx);
  const TilePlan p = tile_plan(ctx);
  const int ntiles = p.ntiles, S = (int)ctx->S, splits = p.adj_splits;
  hipError_t e;
  if ((e = f.lam.ensure(sizeof(double) * (size_t)nb * ntiles * kRows)) != hipSuccess ||
      (e = ctx->hpart.ensure(sizeof(double) * (size_t)splits * nb * ntiles * kTCorners)) !=
          hipSuccess)
    return e;
  const double *sx = ctx->d_sx.as<const double>(), *sy = ctx->d_sy.as<const double>(),
               *sz = ctx->d_sz.as<const double>();
  {
    ProfScope ps(ctx, "tile_far_adjoint_fp64");
    hipLaunchKernelGGL((k_tile_far_adjoint<MASK>), dim3(ntiles, kK, nb), dim3(kBlock), 0, st, sx,
                       sy, sz, S, coef, g, f.geo.as<const double4>(), f.lam.as<double>());
  }
  {
    ProfScope ps(ctx, "tile_near_adjoint_fp64");
    with_models(nb, [&](auto n) {
      hipLaunchKernelGGL((k_tile_near_adjoint<MASK, decltype(n)::value>), dim3(ntiles, splits),
                         dim3(kNearThreads), 0, st, sx, sy, sz, S, coef, g,
                         f.geo.as<const double4>(), ntiles, ctx->hpart.as<double>());
    });
  }
  {
    ProfScope ps(ctx, "tile_gradient_fp64");
    hipLaunchKernelGGL(k_tile_gradient, dim3(ntiles, nb), dim3(kBlock), 0, st, g,
                       f.lam.as<const double>(), harmonic_table(ctx),
                       ctx->hpart.as<const double>(), splits, ntiles, grads, (long)grad_ld);
  }
  return hipGetLastError();
}

}  // namespace

// Makes the choice and, if the expansions are taken, the tables and tile centres, once per
// geometry.
hipError_t tile_far_prepare(jgm_context* ctx, int kind, bool* applies) {
  *applies = false;
  if (kind != JGM_KIND_SCALAR && kind != JGM_KIND_SCALAR_TENSOR) return hipSuccess;
  TileFar& f = ctx->tile_far;
  const int which = kind == JGM_KIND_SCALAR ? 0 : 1;
  if (f.gen[which] != ctx->geom_gen) {
    f.chosen[which] = choose(ctx, which == 1);
    f.gen[which] = ctx->geom_gen;
  }
  if (!f.chosen[which]) return hipSuccess;
  hipError_t e;
  if (!f.tables) {
    const HarmonicBlock& h = harmonic_block();
    if ((e = f.table.ensure(h.bytes.size())) != hipSuccess ||
        (e = hipMemcpyAsync(f.table.ptr, h.bytes.data(), h.bytes.size(), hipMemcpyHostToDevice,
                            ctx->stream)) != hipSuccess ||
        (e = hipStreamSynchronize(ctx->stream)) != hipSuccess)
      return e;
    f.tables = true;
  }
  if (f.geo_gen != ctx->geom_gen) {
    const TileGrid g = tile_grid(ctx);
    const int ntiles = g.tx * g.ty * g.tz;
    if ((e = f.geo.ensure(sizeof(double4) * (size_t)ntiles)) != hipSuccess) return e;
    hipLaunchKernelGGL(k_tile_centres, dim3(blocks_for(ntiles)), dim3(kBlock), 0, ctx->stream, g,
                       ntiles, f.geo.as<double4>());
    if ((e = hipGetLastError()) != hipSuccess) return e;
    f.geo_gen = ctx->geom_gen;
  }
  *applies = true;
  return hipSuccess;
}

// Models to a launch of the up to `left` that remain: as many as 2 GiB of their buffers hold.
int tile_far_models(const jgm_context* ctx, int kind, size_t left) {
  const size_t one = tile_bytes(ctx, tile_plan(ctx), kind != JGM_KIND_SCALAR);
  int nb = left >= 8 ? 8 : left >= 4 ? 4 : left >= 2 ? 2 : 1;
  while (nb > 1 && nb * one > (size_t)2 << 30) nb /= 2;
  return nb;
}

hipError_t tile_far_forward(jgm_context* ctx, int kind, int nb, const double* models,
                            size_t model_ld, double** partial, int* nchunks) {
  return kind == JGM_KIND_SCALAR
             ? forward_partials<kMaskScalar>(ctx, nb, models, model_ld, partial, nchunks)
             : forward_partials<kMaskAll>(ctx, nb, models, model_ld, partial, nchunks);
}

hipError_t tile_far_adjoint(jgm_context* ctx, int kind, int nb, const double* coef, double* grads,
                            size_t grad_ld) {
  return kind == JGM_KIND_SCALAR ? adjoint_cells<kMaskScalar>(ctx, nb, coef, grads, grad_ld)
                                 : adjoint_cells<kMaskAll>(ctx, nb, coef, grads, grad_ld);
}

}  // namespace jgm
