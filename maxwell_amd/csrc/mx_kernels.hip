// mx_kernels.hip -- gfx950 kernels for the Bloch-periodic Nedelec eigensolver.
//
// Every kernel works on a block of nv vectors (grid.y = vector) so that one
// launch covers all vectors of an eigenvector block or of a batch of Bloch
// problems.  Threads map to grid nodes (or patches, or coarse nodes) with the
// i index fastest, so consecutive lanes of a 64-wide wavefront touch
// consecutive complex values of a grid row.  Values outside the periodic cell
// are reached through the Bloch relation u(i+nx, j) = xf u(i, j),
// u(i, j+ny) = yf u(i, j).
//
// Reference behaviour restated here (file:line in the reference):
//   curl-curl + mass stencil ............ edge2d.c:1335-1650
//   AFW vertex-patch solve .............. edge2d.c:2029-2654
//   four-colour sweep order ............. edge2d.c:3043-3480
//   edge prolongation / restriction ..... edge2d.c:5583-5705
//   node Laplacian, GS, transfers ....... node2d.c:516-1273
//   gradient / adjoint gradient ......... node2d.c:1275-1350
//   Ritz Gram entries ................... exp_bloch2d.c:992-996
//   block update ........................ exp_bloch2d.c:1006-1010
#include <hip/hip_runtime.h>

#include <stdint.h>
#include <stdio.h>
#include <time.h>

#include "mxh.h"

#define MXH_DEV __device__ __forceinline__

static hipStream_t g_stream = nullptr;
static int g_device = -1;  // the device g_stream belongs to (current at mxh_init)

// Scratch of mxh_gram_static, the entry point that allocates nothing: the
// Gram kernel's partial-sum sets in a file-scope device array.  Every device
// the library runs on holds its own copy until the process ends; host code
// reaches it only through the address hipGetSymbolAddress returns for it on
// that device (g_scratch_ptr, set by mxh_init with the device current).
#define MXH_MAX_DEVICES 64
static __device__ __align__(256) double scratch[MXH_GRAM_SCRATCH_BYTES / sizeof(double)];
static void* g_scratch_ptr[MXH_MAX_DEVICES];

// ----------------------------------------------------------------- complex
template <typename T>
struct alignas(2 * sizeof(T)) C {
  T r, i;
};

template <typename T> MXH_DEV C<T> cmk(T r, T i) { C<T> z; z.r = r; z.i = i; return z; }
template <typename T> MXH_DEV C<T> operator+(C<T> a, C<T> b) { return cmk(a.r + b.r, a.i + b.i); }
template <typename T> MXH_DEV C<T> operator-(C<T> a, C<T> b) { return cmk(a.r - b.r, a.i - b.i); }
template <typename T> MXH_DEV C<T> operator*(C<T> a, C<T> b)
{
  return cmk(a.r * b.r - a.i * b.i, a.r * b.i + a.i * b.r);
}
template <typename T> MXH_DEV C<T> operator*(T s, C<T> a) { return cmk(s * a.r, s * a.i); }
template <typename T> MXH_DEV C<T> cconj(C<T> a) { return cmk(a.r, -a.i); }
// acc += conj(a) b as four fused multiply-adds
template <typename T> MXH_DEV void cmac_conj(C<T>& acc, C<T> a, C<T> b)
{
  acc.r = fma(a.r, b.r, acc.r);
  acc.r = fma(a.i, b.i, acc.r);
  acc.i = fma(a.r, b.i, acc.i);
  acc.i = fma(-a.i, b.r, acc.i);
}
template <typename T> MXH_DEV C<T> cdiv(C<T> a, C<T> b)
{
  const T d = T(1) / (b.r * b.r + b.i * b.i);
  return cmk((a.r * b.r + a.i * b.i) * d, (a.i * b.r - a.r * b.i) * d);
}
template <typename T> MXH_DEV C<T> czero() { return cmk(T(0), T(0)); }
template <typename T> MXH_DEV C<T>& operator+=(C<T>& a, C<T> b) { a.r += b.r; a.i += b.i; return a; }
template <typename T> MXH_DEV C<T>& operator-=(C<T>& a, C<T> b) { a.r -= b.r; a.i -= b.i; return a; }
template <typename T, typename S> MXH_DEV C<T> ccast(C<S> a) { return cmk(T(a.r), T(a.i)); }

// ----------------------------------------------------------------- geometry
template <typename T>
struct Geo {
  int nx, ny;
  C<T> xf, yf;

  // value at unwrapped (i, j) of a row-major nx x ny array, with Bloch phase
  MXH_DEV C<T> at(const C<T>* a, int i, int j) const
  {
    C<T> ph = cmk(T(1), T(0));
    bool w = false;
    if (i < 0) { i += nx; ph = cconj(xf); w = true; }
    else if (i >= nx) { i -= nx; ph = xf; w = true; }
    if (j < 0) { j += ny; ph = w ? ph * cconj(yf) : cconj(yf); w = true; }
    else if (j >= ny) { j -= ny; ph = w ? ph * yf : yf; w = true; }
    C<T> v = a[i + (size_t)j * nx];
    return w ? ph * v : v;
  }
  // stored value at wrapped (i, j) += conj(phase) * d  (inverse of `at`)
  MXH_DEV void add(C<T>* a, int i, int j, C<T> d) const
  {
    C<T> ph = cmk(T(1), T(0));
    bool w = false;
    if (i < 0) { i += nx; ph = xf; w = true; }
    else if (i >= nx) { i -= nx; ph = cconj(xf); w = true; }
    if (j < 0) { j += ny; ph = w ? ph * yf : yf; w = true; }
    else if (j >= ny) { j -= ny; ph = w ? ph * cconj(yf) : cconj(yf); w = true; }
    size_t k = i + (size_t)j * nx;
    a[k] += w ? ph * d : d;
  }
};

template <typename T>
MXH_DEV T eta_at(const T* eta, int nx, int ny, int i, int j)
{
  if (i < 0) i += nx; else if (i >= nx) i -= nx;
  if (j < 0) j += ny; else if (j >= ny) j -= ny;
  return eta[i + (size_t)j * nx];
}

template <typename T>
MXH_DEV Geo<T> make_geo(const mxh_level& lv, const mxh_bloch& bl, int v)
{
  Geo<T> g;
  g.nx = lv.nx;
  g.ny = lv.ny;
  if (bl.per_problem) {
    const int gv = bl.vmap ? bl.vmap[v] : v;
    const double* q = bl.per_problem + 4 * (gv / bl.vpp);
    g.xf = cmk(T(q[0]), T(q[1]));
    g.yf = cmk(T(q[2]), T(q[3]));
  } else {
    g.xf = cmk(T(bl.xr), T(bl.xi));
    g.yf = cmk(T(bl.yr), T(bl.yi));
  }
  return g;
}

// Edge vector view: x-edges at x, y-edges at x + nx*ny.
template <typename T>
struct EdgeV {
  const C<T>* x;
  const C<T>* y;
};

template <typename T>
MXH_DEV EdgeV<T> edge_view(const void* base, long long stride, int v, size_t N)
{
  EdgeV<T> e;
  e.x = (const C<T>*)base + (size_t)v * stride;
  e.y = e.x + N;
  return e;
}

// Curl of cell (i,j) in unwrapped coordinates (edge2d.c:1505-1514).
template <typename T>
MXH_DEV C<T> cell_curl(const Geo<T>& g, const EdgeV<T>& e, int i, int j)
{
  return g.at(e.x, i, j) - g.at(e.x, i, j + 1) - g.at(e.y, i, j) + g.at(e.y, i + 1, j);
}

// (alpha K + beta M) x at x-edge (i,j) and y-edge (i,j), unwrapped (i,j) allowed.
template <typename T>
MXH_DEV void apply_at(const Geo<T>& g, const EdgeV<T>& e, const T* eta, int i, int j,
                      C<T> axy, C<T> mx, C<T> my, C<T>& ox, C<T>& oy)
{
  C<T> x00 = g.at(e.x, i, j), x0m = g.at(e.x, i, j - 1), x0p = g.at(e.x, i, j + 1);
  C<T> xm0 = g.at(e.x, i - 1, j), xmp = g.at(e.x, i - 1, j + 1);
  C<T> y00 = g.at(e.y, i, j), ym0 = g.at(e.y, i - 1, j), yp0 = g.at(e.y, i + 1, j);
  C<T> y0m = g.at(e.y, i, j - 1), ypm = g.at(e.y, i + 1, j - 1);
  T e00 = eta_at(eta, g.nx, g.ny, i, j);
  T e0m = eta_at(eta, g.nx, g.ny, i, j - 1);
  T em0 = eta_at(eta, g.nx, g.ny, i - 1, j);
  C<T> c00 = x00 - x0p - y00 + yp0;  // cell (i,j)
  C<T> c0m = x0m - x00 - y0m + ypm;  // cell (i,j-1)
  C<T> cm0 = xm0 - xmp - ym0 + y00;  // cell (i-1,j)
  C<T> kx = e00 * c00 - e0m * c0m;
  C<T> ky = em0 * cm0 - e00 * c00;
  ox = axy * kx + mx * (T(4) * x00 + x0m + x0p);
  oy = axy * ky + my * (T(4) * y00 + ym0 + yp0);
}

template <typename T>
MXH_DEV void coefs(const mxh_level& lv, const mxh_coef& cf, int v, C<T>& axy, C<T>& mx, C<T>& my)
{
  double ar = cf.ar, ai = cf.ai, br = cf.br, bi = cf.bi;
  if (cf.per_vector) {
    const double* q = cf.per_vector + 4 * v;
    ar = q[0]; ai = q[1]; br = q[2]; bi = q[3];
  }
  double s = 1.0 / (lv.hx * lv.hy), sx = lv.hy / lv.hx / 6.0, sy = lv.hx / lv.hy / 6.0;
  axy = cmk(T(ar * s), T(ai * s));
  mx = cmk(T(br * sx), T(bi * sx));
  my = cmk(T(br * sy), T(bi * sy));
}

// the value of one lane (uniform), in all lanes
MXH_DEV C<double> lane_value(C<double> v, int lane)
{
  union { double d[2]; int i[4]; } u;
  u.d[0] = v.r;
  u.d[1] = v.i;
#pragma unroll
  for (int q = 0; q < 4; q++) u.i[q] = __builtin_amdgcn_readlane(u.i[q], lane);
  return cmk(u.d[0], u.d[1]);
}

// ----------------------------------------------------------------- reductions
MXH_DEV double wave_sum(double v)
{
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
MXH_DEV double wave_max(double v)
{
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  return v;
}

// Sum over a 256-thread block; result valid in thread 0.
MXH_DEV double block_sum256(double v, double* sh)
{
  v = wave_sum(v);
  int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  __syncthreads();
  if (l == 0) sh[w] = v;
  __syncthreads();
  double r = 0.0;
  if (threadIdx.x == 0) r = sh[0] + sh[1] + sh[2] + sh[3];
  return r;
}
MXH_DEV double block_max256(double v, double* sh)
{
  v = wave_max(v);
  int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  __syncthreads();
  if (l == 0) sh[w] = v;
  __syncthreads();
  double r = 0.0;
  if (threadIdx.x == 0) r = fmax(fmax(sh[0], sh[1]), fmax(sh[2], sh[3]));
  return r;
}

// out[w] = sum_b part[b * width + w] (mode 0) or the max (mode 1): one
// wavefront per output, lane l takes b = l, l + 64, ..., then a fixed
// butterfly -- a fixed order, so the result is deterministic, and 64 loads
// in flight per output instead of a serial chain.
__global__ void k_reduce_partials(const double* __restrict__ part, int nblk, int width,
                                  double* __restrict__ out, int mode)
{
  const int w = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6), l = threadIdx.x & 63;
  if (w >= width) return;  // wave-uniform
  double s = 0.0;
  if (mode == 0) {
    for (int b = l; b < nblk; b += 64) s += part[(size_t)b * width + w];
    s = wave_sum(s);
  } else {
    for (int b = l; b < nblk; b += 64) s = fmax(s, part[(size_t)b * width + w]);
    s = wave_max(s);
  }
  if (l == 0) out[w] = s;
}

static const int TPB = 256;

__global__ __launch_bounds__(256) void k_copy(size_t n, const uint4* src, uint4* dst)
{
  const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) dst[k] = src[k];
}

// the LDS of a compute unit, and bytes per complex value
#define LDS_MAX (160 * 1024)
static size_t csize(int prec) { return prec == MXH_F64 ? 16 : 8; }

static inline unsigned nblocks(long long n, int tpb = TPB) { return (unsigned)((n + tpb - 1) / tpb); }

// k_reduce_partials over `width` outputs: four outputs per 256-thread block
static inline unsigned reduce_blocks(long long width) { return nblocks(width, TPB / 64); }

// Blocks per vector of the row-mapped kernels.
static inline unsigned row_blocks(int ny) { return (unsigned)(ny < 128 ? (ny < 1 ? 1 : ny) : 128); }
// The lifting right-hand side walks columns down its band and reads two
// FP64 and two FP32 rows per band start: taller bands (16 rows at 512) pay
// that start less often (768 vectors at 512^2: 2.75 ms against 3.02 ms for
// 8-row bands, which were 10% faster than 4-row bands; short bands suit the
// defect and the lifting update better).
static inline unsigned lift_blocks(int ny) { return (unsigned)(ny < 32 ? (ny < 1 ? 1 : ny) : 32); }
// Rows of block blockIdx.x in a row-mapped kernel: a contiguous band, so the
// neighbouring rows a stencil reads were read by the same block just before.
MXH_DEV int row_first(int ny)
{
  const int rpb = (ny + (int)gridDim.x - 1) / (int)gridDim.x;
  return min(ny, (int)blockIdx.x * rpb);
}
MXH_DEV int row_end(int ny)
{
  const int rpb = (ny + (int)gridDim.x - 1) / (int)gridDim.x;
  return min(ny, ((int)blockIdx.x + 1) * rpb);
}

// The defect's map: a workgroup of 256 threads covers bands of rows of one
// vector, a thread walks its columns (i0, i0 + 256, ...) down rows j0 .. j1 - 1,
// so the neighbouring rows a stencil reads were read by the same thread or its
// neighbours just before.  Grids of at most 128 columns put 256 / nx bands side
// by side into a workgroup (84^2 in FP64, 194 vectors, defect: 41 -> 23 us).
template <bool NARROW>
struct Band {
  int i0, j0, j1;  // no rows: j0 = j1
  MXH_DEV Band(int nx, int ny)
  {
    const int groups = NARROW ? 256 / nx : 1, q = NARROW ? (int)threadIdx.x / nx : 0;
    const int bands = (int)gridDim.x * groups, rpb = (ny + bands - 1) / bands;
    i0 = (int)threadIdx.x - q * nx;
    const int b = q < groups ? (int)blockIdx.x * groups + q : bands;
    j0 = min(ny, b * rpb);
    j1 = min(ny, j0 + rpb);
  }
};
static inline bool narrow(const mxh_level* lv) { return lv->nx <= 128; }
// Its workgroups per vector: four rows a band, fewer where that leaves the chip
// short of workgroups (four per compute unit), BAND_MAX at most (the partial
// sums' places).
#define BAND_MAX 128
static inline unsigned band_blocks(const mxh_level* lv, int nv)
{
  const int groups = narrow(lv) ? 256 / lv->nx : 1;
  auto blocks = [&](int r) { return (lv->ny + groups * r - 1) / (groups * r); };
  int rows = 4;
  while (rows > 1 && (long long)nv * blocks(rows) < 1024) rows >>= 1;
  const int nb = blocks(rows);
  return (unsigned)(nb < 1 ? 1 : nb < BAND_MAX ? nb : BAND_MAX);
}

// The frame of an nx x ny grid (rows 0 and ny - 1, columns 0 and nx - 1):
// the points whose stencils wrap.  The row-mapped kernels run the interior
// with direct indexing and the frame in a second, small launch with the
// wrapped form, so the interior kernel carries no registers for the wrap.
__host__ __device__ inline long long frame_points(int nx, int ny)
{
  return ny > 2 ? 2LL * nx + 2LL * (ny - 2) : (long long)nx * ny;
}
MXH_DEV void frame_point(int k, int nx, int ny, int& i, int& j)
{
  if (ny <= 2) { i = k % nx; j = k / nx; }
  else if (k < nx) { i = k; j = 0; }
  else if (k < 2 * nx) { i = k - nx; j = ny - 1; }
  else { const int q = k - 2 * nx; i = (q & 1) ? nx - 1 : 0; j = 1 + (q >> 1); }
}
static inline unsigned frame_blocks(const mxh_level* lv)
{
  const long long b = (frame_points(lv->nx, lv->ny) + 255) / 256;
  return (unsigned)(b > 8 ? 8 : (b < 1 ? 1 : b));
}

// Number of blocks used for grid-stride reductions (partials per vector).
static inline unsigned red_blocks(long long n)
{
  long long b = (n + TPB - 1) / TPB;
  if (b > 512) b = 512;
  if (b < 1) b = 1;
  return (unsigned)b;
}

// ----------------------------------------------------------------- addeval
template <typename T>
__global__ __launch_bounds__(256) void k_addeval(mxh_level lv, mxh_bloch bl, const C<T>* X, long long xs,
                                                 C<T>* Y, long long ys, const T* eta, mxh_coef cf,
                                                 int accumulate)
{
  const int v = blockIdx.y;
  const size_t N = (size_t)lv.nx * lv.ny;
  size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= N) return;
  int i = (int)(idx % lv.nx), j = (int)(idx / lv.nx);
  Geo<T> g = make_geo<T>(lv, bl, v);
  C<T> axy, mx, my;
  coefs<T>(lv, cf, v, axy, mx, my);
  EdgeV<T> e = edge_view<T>(X, xs, v, N);
  C<T> ox, oy;
  apply_at(g, e, eta, i, j, axy, mx, my, ox, oy);
  C<T>* y = Y + (size_t)v * ys;
  if (accumulate) {
    y[idx] += ox;
    y[N + idx] += oy;
  } else {
    y[idx] = ox;
    y[N + idx] = oy;
  }
}

// PINVIT defect r = (K + (1 - lam) M) e in FP64, stored in precision R, plus
// per-block partial sums of |r|^2 and |M e|^2 over the block's band of rows.
//
// Each thread walks its columns down the band, keeping the values the next
// row's stencil shares with this one (half the loads per point).  Columns start
// at 0 (whole cache lines per wave); the Bloch factors are applied in the first
// and last column and row only.  192 vectors of 512^2 in mixed precision: 548 ->
// 482 us with its reduction (4.4 -> 5.0 TB/s).
template <typename R, bool NARROW>
__global__ __launch_bounds__(256) void k_defect(mxh_level lv, mxh_bloch bl, const C<double>* E, long long es,
                                                const int* emap, C<R>* Rv, long long rs, const double* eta,
                                                const double* lam, double* part)
{
  __shared__ double sh[4];
  const int v = blockIdx.y;
  const int gv = emap ? emap[v] : v;
  const int nx = lv.nx, ny = lv.ny;
  const size_t N = (size_t)nx * ny;
  const Geo<double> g = make_geo<double>(lv, bl, v);
  const double s = 1.0 / (lv.hx * lv.hy), sx = lv.hy / lv.hx / 6.0, sy = lv.hx / lv.hy / 6.0;
  const double be = 1.0 - lam[gv];
  const EdgeV<double> e = edge_view<double>(E, es, gv, N);
  C<R>* r = Rv + (size_t)v * rs;
  double rr = 0.0, mm = 0.0;
  const Band<NARROW> band(nx, ny);
  const int j0 = band.j0, j1 = band.j1;
  const C<double>* ex = e.x;
  const C<double>* ey = e.y;
  if (j0 < j1)
    for (int i = band.i0; i < nx; i += 256) {
      const bool wl = i == 0, wr = i == nx - 1;
      const int im = wl ? nx - 1 : i - 1, ip = wr ? 0 : i + 1;
      const size_t below = (size_t)(j0 ? j0 - 1 : ny - 1) * nx;
      size_t k = (size_t)j0 * nx;
      C<double> x0m = ex[below + i], x00 = ex[k + i], xm0 = ex[k + im];
      C<double> y0m = ey[below + i], ypm = ey[below + ip];
      double e0m = eta[below + i];
      if (wl) xm0 = cconj(g.xf) * xm0;
      if (wr) ypm = g.xf * ypm;
      if (j0 == 0) {
        x0m = cconj(g.yf) * x0m;
        y0m = cconj(g.yf) * y0m;
        ypm = cconj(g.yf) * ypm;
      }
      for (int j = j0; j < j1; j++, k += nx) {
        const size_t above = j + 1 < ny ? k + nx : 0;
        C<double> x0p = ex[above + i], xmp = ex[above + im];
        C<double> ym0 = ey[k + im], yp0 = ey[k + ip];
        const C<double> y00 = ey[k + i];
        const double e00 = eta[k + i], em0 = eta[k + im];
        if (wl) {
          xmp = cconj(g.xf) * xmp;
          ym0 = cconj(g.xf) * ym0;
        }
        if (wr) yp0 = g.xf * yp0;
        if (j + 1 == ny) {
          x0p = g.yf * x0p;
          xmp = g.yf * xmp;
        }
        const C<double> c00 = x00 - x0p - y00 + yp0;  // cell (i,j)
        const C<double> c0m = x0m - x00 - y0m + ypm;  // cell (i,j-1)
        const C<double> cm0 = xm0 - xmp - ym0 + y00;  // cell (i-1,j)
        const C<double> kx = e00 * c00 - e0m * c0m, ky = em0 * cm0 - e00 * c00;
        const C<double> mxv = sx * (4.0 * x00 + x0m + x0p), myv = sy * (4.0 * y00 + ym0 + yp0);
        const C<double> ox = s * kx + be * mxv, oy = s * ky + be * myv;
        r[k + i] = ccast<R>(ox);
        r[N + k + i] = ccast<R>(oy);
        rr += ox.r * ox.r + ox.i * ox.i + oy.r * oy.r + oy.i * oy.i;
        mm += mxv.r * mxv.r + mxv.i * mxv.i + myv.r * myv.r + myv.i * myv.i;
        x0m = x00;
        x00 = x0p;
        xm0 = xmp;
        y0m = y00;
        ypm = yp0;
        e0m = e00;
      }
    }
  double a = block_sum256(rr, sh);
  double b = block_sum256(mm, sh);
  if (threadIdx.x == 0) {
    size_t w = (size_t)blockIdx.x * (2 * gridDim.y) + 2 * v;
    part[w] = a;
    part[w + 1] = b;
  }
}

// ----------------------------------------------------------------- AFW local solve
// Exact solve of the 4x4 patch system
//   [[a0, 0, -eLL, eLU], [0, a1, eRL, -eRU], [-eLL, eRL, a2, 0], [eLU, -eRU, 0, a3]] z = r
// by eliminating z0, z1 (diagonal block) and solving the 2x2 Schur complement
// for z2, z3.  a0..a3 carry the reference's doubled mass diagonal.
// Reciprocals of the local solve's pivots, which only feed the multigrid
// preconditioner: in FP64 the hardware estimate refined by two Newton steps
// (within an ulp or two of IEEE division, at half its instructions); in FP32
// the hardware reciprocal (1 ulp).  The pivots are positive and of order
// 1 / (hx hy).
MXH_DEV double recip(double a)
{
  double r = __builtin_amdgcn_rcp(a);
  r = fma(fma(-a, r, 1.0), r, r);
  return fma(fma(-a, r, 1.0), r, r);
}
MXH_DEV float recip(float a) { return __builtin_amdgcn_rcpf(a); }

template <typename T>
MXH_DEV void afw_local_solve(T eLL, T eRL, T eLU, T eRU, T mx, T my, C<T> r0, C<T> r1, C<T> r2, C<T> r3, C<T>& z0,
                             C<T>& z1, C<T>& z2, C<T>& z3)
{
  const T a0 = eLL + eLU + T(8) * mx, a1 = eRL + eRU + T(8) * mx;
  const T a2 = eLL + eRL + T(8) * my, a3 = eLU + eRU + T(8) * my;
  const T p = recip(a0), q = recip(a1);
  const T c20 = eLL * p, c21 = eRL * q, c30 = eLU * p, c31 = eRU * q;
  const T s22 = a2 - eLL * c20 - eRL * c21;
  const T s33 = a3 - eLU * c30 - eRU * c31;
  const T s23 = eLL * c30 + eRL * c31;
  const T idet = recip(s22 * s33 - s23 * s23);
  const C<T> s2 = r2 + c20 * r0 - c21 * r1;
  const C<T> s3 = r3 - c30 * r0 + c31 * r1;
  z2 = idet * (s33 * s2 - s23 * s3);
  z3 = idet * (s22 * s3 - s23 * s2);
  z0 = p * r0 + c20 * z2 - c30 * z3;
  z1 = q * r1 - c21 * z2 + c31 * z3;
}

// ----------------------------------------------------------------- AFW smoother
// Exact solve on the star of node (i,j) with the reference's patch matrix
// alpha K_patch + 2 beta M_patch (edge2d.c:2038-2062) and the exact residual
// b - (alpha K + beta M) x.  Unknowns: u0 = x(i-1,j), u1 = x(i,j),
// u2 = y(i,j-1), u3 = y(i,j).
template <typename T>
__global__ __launch_bounds__(256) void k_afw_phase(mxh_level lv, mxh_bloch bl, const C<T>* B, long long bs,
                                                   C<T>* X, long long xs, const T* eta, double alpha,
                                                   double beta, int ci, int cj)
{
  const int v = blockIdx.y;
  const int hx2 = lv.nx >> 1;
  const size_t np = (size_t)hx2 * (lv.ny >> 1);
  size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  const int i = 2 * (int)(p % hx2) + ci, j = 2 * (int)(p / hx2) + cj;
  const size_t N = (size_t)lv.nx * lv.ny;
  Geo<T> g = make_geo<T>(lv, bl, v);
  C<T>* xx = X + (size_t)v * xs;
  C<T>* xy = xx + N;
  const C<T>* bx = B + (size_t)v * bs;
  const C<T>* by = bx + N;
  const T axy = T(alpha / (lv.hx * lv.hy));
  const T mx = T(beta * lv.hy / lv.hx / 6.0), my = T(beta * lv.hx / lv.hy / 6.0);

  C<T> xLm = g.at(xx, i - 1, j - 1), xL0 = g.at(xx, i - 1, j), xLp = g.at(xx, i - 1, j + 1);
  C<T> xRm = g.at(xx, i, j - 1), xR0 = g.at(xx, i, j), xRp = g.at(xx, i, j + 1);
  C<T> yLm = g.at(xy, i - 1, j - 1), yCm = g.at(xy, i, j - 1), yRm = g.at(xy, i + 1, j - 1);
  C<T> yL0 = g.at(xy, i - 1, j), yC0 = g.at(xy, i, j), yR0 = g.at(xy, i + 1, j);

  const T eLL = axy * eta_at(eta, lv.nx, lv.ny, i - 1, j - 1);
  const T eRL = axy * eta_at(eta, lv.nx, lv.ny, i, j - 1);
  const T eLU = axy * eta_at(eta, lv.nx, lv.ny, i - 1, j);
  const T eRU = axy * eta_at(eta, lv.nx, lv.ny, i, j);

  C<T> qLL = eLL * (xLm - xL0 - yLm + yCm);
  C<T> qRL = eRL * (xRm - xR0 - yCm + yRm);
  C<T> qLU = eLU * (xL0 - xLp - yL0 + yC0);
  C<T> qRU = eRU * (xR0 - xRp - yC0 + yR0);

  C<T> r0 = g.at(bx, i - 1, j) - (qLU - qLL) - mx * (T(4) * xL0 + xLm + xLp);
  C<T> r1 = g.at(bx, i, j) - (qRU - qRL) - mx * (T(4) * xR0 + xRm + xRp);
  C<T> r2 = g.at(by, i, j - 1) - (qLL - qRL) - my * (T(4) * yCm + yLm + yRm);
  C<T> r3 = g.at(by, i, j) - (qLU - qRU) - my * (T(4) * yC0 + yL0 + yR0);

  C<T> z0, z1, z2, z3;
  afw_local_solve(eLL, eRL, eLU, eRU, mx, my, r0, r1, r2, r3, z0, z1, z2, z3);

  g.add(xx, i - 1, j, z0);
  xx[i + (size_t)j * lv.nx] += z1;
  g.add(xy, i, j - 1, z2);
  xy[i + (size_t)j * lv.nx] += z3;
}

// ----------------------------------------------------------------- residual + restriction
template <typename T>
MXH_DEV void resid_at(const Geo<T>& g, const EdgeV<T>& b, const EdgeV<T>& x, const T* eta, int i, int j,
                      C<T> axy, C<T> mx, C<T> my, C<T>& rx, C<T>& ry)
{
  C<T> ax, ay;
  apply_at(g, x, eta, i, j, axy, mx, my, ax, ay);
  rx = g.at(b.x, i, j) - ax;
  ry = g.at(b.y, i, j) - ay;
}

template <typename T>
__global__ __launch_bounds__(256) void k_resid_restrict(mxh_level lf, mxh_bloch bl, const C<T>* BF, long long bfs,
                                                        const C<T>* XF, long long xfs, const T* eta,
                                                        C<T>* BC, long long bcs, C<T>* XC, long long xcs)
{
  const int v = blockIdx.y;
  const int cnx = lf.nx >> 1, cny = lf.ny >> 1;
  const size_t NC = (size_t)cnx * cny, NF = (size_t)lf.nx * lf.ny;
  size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= NC) return;
  const int I = (int)(idx % cnx), J = (int)(idx / cnx);
  Geo<T> g = make_geo<T>(lf, bl, v);
  EdgeV<T> b = edge_view<T>(BF, bfs, v, NF), x = edge_view<T>(XF, xfs, v, NF);
  const double s = 1.0 / (lf.hx * lf.hy);
  const C<T> axy = cmk(T(s), T(0));
  const C<T> mx = cmk(T(lf.hy / lf.hx / 6.0), T(0)), my = cmk(T(lf.hx / lf.hy / 6.0), T(0));
  C<T> rx, ry, sx = czero<T>(), sy = czero<T>();
  const int i0 = 2 * I, j0 = 2 * J;
  // x-edges: (i0,j0),(i0+1,j0) weight 1/2; rows j0-1 and j0+1 weight 1/4
  resid_at(g, b, x, eta, i0, j0, axy, mx, my, rx, ry);
  sx += T(0.5) * rx;
  sy += T(0.5) * ry;  // y(i0, j0)
  resid_at(g, b, x, eta, i0 + 1, j0, axy, mx, my, rx, ry);
  sx += T(0.5) * rx;
  sy += T(0.25) * ry;  // y(i0+1, j0)
  resid_at(g, b, x, eta, i0, j0 + 1, axy, mx, my, rx, ry);
  sx += T(0.25) * rx;
  sy += T(0.5) * ry;  // y(i0, j0+1)
  resid_at(g, b, x, eta, i0 + 1, j0 + 1, axy, mx, my, rx, ry);
  sx += T(0.25) * rx;
  sy += T(0.25) * ry;  // y(i0+1, j0+1)
  resid_at(g, b, x, eta, i0, j0 - 1, axy, mx, my, rx, ry);
  sx += T(0.25) * rx;
  resid_at(g, b, x, eta, i0 + 1, j0 - 1, axy, mx, my, rx, ry);
  sx += T(0.25) * rx;
  resid_at(g, b, x, eta, i0 - 1, j0, axy, mx, my, rx, ry);
  sy += T(0.25) * ry;
  resid_at(g, b, x, eta, i0 - 1, j0 + 1, axy, mx, my, rx, ry);
  sy += T(0.25) * ry;
  C<T>* bc = BC + (size_t)v * bcs;
  C<T>* xc = XC + (size_t)v * xcs;
  bc[idx] = sx;
  bc[NC + idx] = sy;
  xc[idx] = czero<T>();
  xc[NC + idx] = czero<T>();
}

// ----------------------------------------------------------------- transfers
template <typename T>
__global__ __launch_bounds__(256) void k_prolong(mxh_level lf, mxh_bloch bl, const C<T>* CV, long long cs,
                                                 C<T>* FV, long long fs, T alpha)
{
  const int v = blockIdx.y;
  const int cnx = lf.nx >> 1, cny = lf.ny >> 1;
  const size_t NC = (size_t)cnx * cny, NF = (size_t)lf.nx * lf.ny;
  size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= NC) return;
  const int I = (int)(idx % cnx), J = (int)(idx / cnx);
  Geo<T> gc = make_geo<T>(lf, bl, v);
  gc.nx = cnx;
  gc.ny = cny;
  const C<T>* cx = CV + (size_t)v * cs;
  const C<T>* cy = cx + NC;
  C<T>* fx = FV + (size_t)v * fs;
  C<T>* fy = fx + NF;
  C<T> a0 = cx[idx], a1 = gc.at(cx, I, J + 1);
  C<T> b0 = cy[idx], b1 = gc.at(cy, I + 1, J);
  const size_t r0 = (size_t)(2 * J) * lf.nx, r1 = r0 + lf.nx;
  const int i0 = 2 * I;
  C<T> h = (T(0.5) * alpha) * a0, q = (T(0.25) * alpha) * (a0 + a1);
  fx[r0 + i0] += h;
  fx[r0 + i0 + 1] += h;
  fx[r1 + i0] += q;
  fx[r1 + i0 + 1] += q;
  h = (T(0.5) * alpha) * b0;
  q = (T(0.25) * alpha) * (b0 + b1);
  fy[r0 + i0] += h;
  fy[r1 + i0] += h;
  fy[r0 + i0 + 1] += q;
  fy[r1 + i0 + 1] += q;
}

template <typename T>
__global__ __launch_bounds__(256) void k_restrict(mxh_level lf, mxh_bloch bl, const C<T>* FV, long long fs,
                                                  C<T>* CV, long long cs, T alpha)
{
  const int v = blockIdx.y;
  const int cnx = lf.nx >> 1, cny = lf.ny >> 1;
  const size_t NC = (size_t)cnx * cny, NF = (size_t)lf.nx * lf.ny;
  size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= NC) return;
  const int I = (int)(idx % cnx), J = (int)(idx / cnx);
  Geo<T> g = make_geo<T>(lf, bl, v);
  const C<T>* fx = FV + (size_t)v * fs;
  const C<T>* fy = fx + NF;
  const int i0 = 2 * I, j0 = 2 * J;
  C<T> sx = T(0.5) * (g.at(fx, i0, j0) + g.at(fx, i0 + 1, j0)) +
            T(0.25) * (g.at(fx, i0, j0 - 1) + g.at(fx, i0 + 1, j0 - 1) + g.at(fx, i0, j0 + 1) +
                       g.at(fx, i0 + 1, j0 + 1));
  C<T> sy = T(0.5) * (g.at(fy, i0, j0) + g.at(fy, i0, j0 + 1)) +
            T(0.25) * (g.at(fy, i0 - 1, j0) + g.at(fy, i0 - 1, j0 + 1) + g.at(fy, i0 + 1, j0) +
                       g.at(fy, i0 + 1, j0 + 1));
  C<T>* cx = CV + (size_t)v * cs;
  cx[idx] += alpha * sx;
  cx[NC + idx] += alpha * sy;
}

// ----------------------------------------------------------------- coarse dense solve
// x = L^{-H} L^{-1} b with L lower, column-major n x n (double complex).
// One block per vector, n <= blockDim.x; column-oriented substitution.
// Per-k coarse set-up on the device (exp_bloch2d.c:799-809): one workgroup per
// problem assembles the n0 x n0 coarse matrices from cell matrices -- the edge
// K + M with the reference's phases (edge2d.c:5870-6110) and the Q1 node
// Laplacian with the Gamma fill of node2d.c:1454-1458 -- in LDS, factors them
// (lower Cholesky, column by column) and writes the factors column-major.
// Each entry sums its cell contributions in the order of a serial assembly
// (cells row-major, element rows, element columns).  info[p] = 0, or the
// column (1-based) of a non-positive pivot.
MXH_DEV C<double> coarse_wrap(int nx, int ny, C<double> xf, C<double> yf, int& i, int& j)
{
  C<double> ph = cmk(1.0, 0.0);
  if (i >= nx) { i -= nx; ph = ph * xf; }
  if (j >= ny) { j -= ny; ph = ph * yf; }
  return ph;
}

MXH_DEV void coarse_cholesky(C<double>* a, int n, double* dsh, int* info)
{
  for (int c = 0; c < n; c++) {
    __syncthreads();
    if (threadIdx.x == 0) {
      double s = a[c + c * n].r;
      for (int k = 0; k < c; k++) {
        const C<double> v = a[c + k * n];
        s -= v.r * v.r + v.i * v.i;
      }
      if (!(s > 0.0) && *info == 0) *info = c + 1;
      const double d = s > 0.0 ? sqrt(s) : 1.0;
      dsh[0] = d;
      a[c + c * n] = cmk(d, 0.0);
    }
    __syncthreads();
    const double d = dsh[0];
    for (int r = c + 1 + (int)threadIdx.x; r < n; r += blockDim.x) {
      C<double> t = a[r + c * n];
      for (int k = 0; k < c; k++) t -= a[r + k * n] * cconj(a[c + k * n]);
      a[r + c * n] = cmk(t.r / d, t.i / d);
    }
    for (int r = threadIdx.x; r < c; r += blockDim.x) a[r + c * n] = czero<double>();
  }
  __syncthreads();
}

__global__ __launch_bounds__(256) void k_coarse_setup(int n0, const double* bloch, const double* eta, double* Ae,
                                                      double* An, int* info)
{
  extern __shared__ double smem[];
  const int p = blockIdx.x, nx = n0, ny = n0, N = n0 * n0, ne = 2 * N;
  C<double>* a = (C<double>*)smem;
  C<double>* b = a + ne * ne;
  double* dsh = (double*)(b + N * N);
  __shared__ int inf;
  if (threadIdx.x == 0) inf = 0;
  const double* q = bloch + 4 * p;
  const C<double> xf = cmk(q[0], q[1]), yf = cmk(q[2], q[3]);
  const double hx = 1.0 / n0, hy = 1.0 / n0;
  const double axy = 1.0 / hx / hy, mx = hy / hx / 6.0, my = hx / hy / 6.0;
  // edge matrix K + M
  for (int e = threadIdx.x; e < ne * ne; e += blockDim.x) {
    const int r = e % ne, c = e / ne;
    C<double> acc = czero<double>();
    for (int j = 0; j < ny; j++)
      for (int i = 0; i < nx; i++) {
        int gi[4];
        C<double> ph[4];
        const int di[4] = {0, 0, 0, 1}, dj[4] = {0, 1, 0, 0}, off[4] = {0, 0, N, N};
        bool hit = false;
        for (int k = 0; k < 4; k++) {
          int ii = i + di[k], jj = j + dj[k];
          ph[k] = coarse_wrap(nx, ny, xf, yf, ii, jj);
          gi[k] = off[k] + ii + jj * nx;
          hit |= gi[k] == r;
        }
        if (!hit) continue;
        const double sgn[4] = {1.0, -1.0, -1.0, 1.0};
        const double et = eta[i + j * nx];
        for (int kp = 0; kp < 4; kp++) {
          if (gi[kp] != r) continue;
          for (int kq = 0; kq < 4; kq++) {
            if (gi[kq] != c) continue;
            double ke = axy * et * sgn[kp] * sgn[kq];
            if (kp < 2 && kq < 2) ke += (kp == kq ? 2.0 : 1.0) * mx;
            if (kp >= 2 && kq >= 2) ke += (kp == kq ? 2.0 : 1.0) * my;
            acc += (cconj(ph[kp]) * cmk(ke, 0.0)) * ph[kq];
          }
        }
      }
    a[r + c * ne] = acc;
  }
  // node matrix: Q1 Laplacian, Gamma fill
  const bool gamma = hypot(xf.r - 1.0, xf.i) < 1e-8 && hypot(yf.r - 1.0, yf.i) < 1e-8;
  const double fill = gamma ? 0.1 / ((double)N * N) : 0.0;
  const double rx = hy / hx, ry = hx / hy;
  for (int e = threadIdx.x; e < N * N; e += blockDim.x) {
    const int r = e % N, c = e / N;
    C<double> acc = cmk(fill, 0.0);
    for (int j = 0; j < ny; j++)
      for (int i = 0; i < nx; i++) {
        int gi[4];
        C<double> ph[4];
        for (int k = 0; k < 4; k++) {
          int ii = i + (k & 1), jj = j + (k >> 1);
          ph[k] = coarse_wrap(nx, ny, xf, yf, ii, jj);
          gi[k] = ii + jj * nx;
        }
        for (int kp = 0; kp < 4; kp++) {
          if (gi[kp] != r) continue;
          for (int kq = 0; kq < 4; kq++) {
            if (gi[kq] != c) continue;
            const int px = kp & 1, py = kp >> 1, qx = kq & 1, qy = kq >> 1;
            const double S0 = px == qx ? 1.0 : -1.0, S1 = py == qy ? 1.0 : -1.0;
            const double T0 = px == qx ? 1.0 / 3.0 : 1.0 / 6.0, T1 = py == qy ? 1.0 / 3.0 : 1.0 / 6.0;
            const double ke = rx * S0 * T1 + ry * T0 * S1;
            acc += (cconj(ph[kp]) * cmk(ke, 0.0)) * ph[kq];
          }
        }
      }
    b[r + c * N] = acc;
  }
  __syncthreads();
  coarse_cholesky(a, ne, dsh, &inf);
  coarse_cholesky(b, N, dsh, &inf);
  C<double>* oa = (C<double>*)Ae + (size_t)p * ne * ne;
  C<double>* ob = (C<double>*)An + (size_t)p * N * N;
  for (int e = threadIdx.x; e < ne * ne; e += blockDim.x) oa[e] = a[e];
  for (int e = threadIdx.x; e < N * N; e += blockDim.x) ob[e] = b[e];
  if (threadIdx.x == 0) info[p] = inf;
}

template <typename T>
__global__ __launch_bounds__(256) void k_coarse_solve(int n, const double* Lm, const double* Lper, int vpp,
                                                      const int* vmap, const C<T>* B, long long bs, C<T>* X,
                                                      long long xs)
{
  extern __shared__ double smem[];
  C<double>* z = (C<double>*)smem;
  const int v = blockIdx.x;
  const int gv = vmap ? vmap[v] : v;
  const C<double>* L = (const C<double>*)(Lper ? Lper + (size_t)2 * n * n * (gv / vpp) : Lm);
  const int t = threadIdx.x;
  if (t < n) z[t] = ccast<double>(B[(size_t)v * bs + t]);
  __syncthreads();
  for (int c = 0; c < n; c++) {
    if (t == c) {
      C<double> d = L[c + (size_t)c * n];
      double inv = 1.0 / d.r;  // real positive diagonal
      z[c] = inv * z[c];
    }
    __syncthreads();
    if (t > c && t < n) z[t] -= L[t + (size_t)c * n] * z[c];
    __syncthreads();
  }
  for (int c = n - 1; c >= 0; c--) {
    if (t == c) {
      double inv = 1.0 / L[c + (size_t)c * n].r;
      z[c] = inv * z[c];
    }
    __syncthreads();
    if (t < c) z[t] -= cconj(L[c + (size_t)t * n]) * z[c];
    __syncthreads();
  }
  if (t < n) X[(size_t)v * xs + t] = ccast<T>(z[t]);
}

// ----------------------------------------------------------------- Gram products
// For each block j (problem q = pmap[j]) of m FP64 vectors, the lower
// triangles of gk[a,b] = sum_cells eta conj(c_a) c_b and gm[a,b] = u_a^H M u_b,
// c the cell curl.  The mass matrix couples an x-edge with its neighbours in
// j by the rows mx (1, 4, 1) (a y-edge with its neighbours in i by my (1, 4,
// 1)); with the Bloch shift S (x(j+1), unitary) that circulant factors as
//   4 + S + S^H = 6 (a + b S)^H (a + b S),  a, b = (1 +- 1/sqrt 3) / 2
// (a^2 + b^2 = 2/3, ab = 1/6), so x^H M y = ux^H uy + (y-edge analogue) with
// ux = sqrt(6 mx) (a x(i,j) + b x(i,j+1)): every cell contributes three
// features (c, ux, uy) of its own edges and their upper and right neighbours.
//
// The contraction runs on the FP64 matrix cores without LDS: eight vectors
// are the 16 real columns of a tile (real parts, then imaginary parts), and
// v_mfma_f64_16x16x4 wants both operands of P^T P in the same lane layout
// (column lane & 15, cell lane >> 4), so one register holds a feature of a
// tile as left and as right operand.  A lane loads (16 bytes) the complex
// values of vector lane & 7 at cell 2 (lane >> 4) + ((lane >> 3) & 1) of a
// strip of eight cells (128 bytes per vector) and trades one half with lane ^ 8
// to have the operands of the even and of the odd cells.  A wave walks a strip
// down its rows, carrying x(j + 1) over as the next row's x(j); the next row's
// loads are issued as soon as a tile's features are formed and land behind
// its products.  The waves share nothing until the end, where their sums meet
// in LDS.
//
// What bounds it: the FP64 pipe.  36 columns (5 tiles, one wave per SIMD: the
// sums of 15 tile pairs take 240 registers) spend 90 MFMAs of 64 cycles per
// strip row and wave and about a sixth of that on features, which the matrix
// core does not overlap.  512^2, against a register-blocked vector kernel fed
// from LDS (bound by its LDS reads and their latency): 36 columns of 64
// problems 10.8 -> 6.4 ms (60 TFLOP/s with the padded tiles' products, the
// matrix pipe busy 81% of the cycles), 32 columns of 16 2.62 -> 1.27, 12 columns
// of 64 2.2 -> 1.64 (3.9 TB/s).  The tile loop's MFMA and vector instructions interleaved by
// hand, and two waves per SIMD at 3 tiles, measured no better.
#define GRAM_MMAX 48
#define GRAM_STRIP 8

MXH_DEV void pair_ab(int p, int& a, int& b)
{
  int r = (int)((sqrtf(8.0f * (float)p + 1.0f) - 1.0f) * 0.5f);
  while ((r + 1) * (r + 2) / 2 <= p) r++;
  while (r * (r + 1) / 2 > p) r--;
  a = r;
  b = p - r * (r + 1) / 2;
}

typedef double v4d __attribute__((ext_vector_type(4)));

// the value of lane ^ 8 (a rotation by 8 in each row of 16 lanes) where the
// bank mask selects (banks of four lanes: 0xf all, 0x3 lanes 0-7 of a row,
// 0xc lanes 8-15), elsewhere old
template <int BANKS>
MXH_DEV double lane_xor8(double old, double v)
{
  union { double d; int i[2]; } u, o;
  u.d = v;
  o.d = old;
  o.i[0] = __builtin_amdgcn_update_dpp(o.i[0], u.i[0], 0x128, 0xf, BANKS, false);
  o.i[1] = __builtin_amdgcn_update_dpp(o.i[1], u.i[1], 0x128, 0xf, BANKS, false);
  return o.d;
}

struct gram_false { static constexpr bool value = false; };
struct gram_true { static constexpr bool value = true; };

struct GramArgs {
  const C<double>* U;  // the problem's first vector
  long long us;
  const int* cl;       // its column list (after the count), or null
  const double* eta;
  double* out;         // the workgroup's partial sums
  C<double> xf, yf;
  double xa, xb, ya, yb;
  int nx, ny, mq, j0, j1;
};

// The sums of one workgroup's rows over Q tiles (8 vectors each), or (LAST) of the
// last tile with itself and those before only: K (MATS & 1) and M (MATS & 2).
template <int Q, bool LAST = false, int MATS = 3>
MXH_DEV void gram_rows(const GramArgs& g, double* lds)
{
  constexpr int NP = LAST ? Q : Q * (Q + 1) / 2;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = (lane >> 3) & 1, k2 = 2 * (lane >> 4);
  const int nx = g.nx, ny = g.ny;
  const size_t N = (size_t)nx * ny;
  const C<double>* u[Q];
#pragma unroll
  for (int t = 0; t < Q; t++) {
    // columns past the list repeat the last one; their sums are not written
    const int a = min(8 * t + (lane & 7), g.mq - 1);
    u[t] = g.U + (size_t)(g.cl ? g.cl[a] : a) * g.us;
  }
  v4d K[NP], M[NP];
#pragma unroll
  for (int p = 0; p < NP; p++) K[p] = M[p] = v4d{0.0, 0.0, 0.0, 0.0};
  // the waves share the strips of a row, or the rows where there are few strips
  const int ns = (nx + GRAM_STRIP - 1) / GRAM_STRIP;
  int ja = g.j0, jb = g.j1, s0 = wave, sstep = 4;
  if (ns < 4) {
    const int sub = (g.j1 - g.j0 + 3) >> 2;
    ja = min(g.j1, g.j0 + wave * sub);
    jb = min(g.j1, ja + sub);
    s0 = 0;
    sstep = 1;
  }
  for (int s = s0; s < ns; s += sstep) {
    if (ja >= jb) break;
    const int cell = GRAM_STRIP * s + k2 + h, i = min(cell, nx - 1);
    const bool last = GRAM_STRIP * s + GRAM_STRIP >= nx;  // wraps in x (and may hold cells past the grid)
    const int ir = i + 1 < nx ? i + 1 : 0;
    const int ie = min(GRAM_STRIP * s + k2, nx - 1), io = min(GRAM_STRIP * s + k2 + 1, nx - 1);
    C<double> x0[Q], x1[Q], y0[Q], yr[Q];
    size_t row = (size_t)ja * nx, up = (size_t)(ja + 1 < ny ? ja + 1 : 0) * nx;
    double ee = g.eta[row + ie], eo = g.eta[row + io];
#pragma unroll
    for (int t = 0; t < Q; t++) {
      x0[t] = u[t][row + i];
      x1[t] = u[t][up + i];
      y0[t] = u[t][N + row + i];
      yr[t] = u[t][N + row + ir];
    }
    // Row j of the strip.  edge: the strip wraps in x, or the row in y; the
    // other rows run without the test, as a loop of one block, so that the
    // next row's loads stay where they are issued
    auto row_step = [&](int j, auto edge) {
      const double e0 = ee, e1 = eo;
      // the next row (the last one loads itself again)
      const int jn = j + 1 < jb ? j + 1 : j;
      row = (size_t)jn * nx;
      up = (size_t)(jn + 1 < ny ? jn + 1 : 0) * nx;
      ee = g.eta[row + ie];
      eo = g.eta[row + io];
      double F[Q][3][2];
#pragma unroll
      for (int t = 0; t < Q; t++) {
        if constexpr (decltype(edge)::value) {
          if (j + 1 == ny) x1[t] = g.yf * x1[t];
          if (i + 1 == nx) yr[t] = g.xf * yr[t];
          if (cell >= nx) x0[t] = x1[t] = y0[t] = yr[t] = czero<double>();
        }
        C<double> f[3];
        f[0] = x0[t] - x1[t] - y0[t] + yr[t];
        f[1] = g.xa * x0[t] + g.xb * x1[t];
        f[2] = g.ya * y0[t] + g.yb * yr[t];
        x0[t] = x1[t];
        x1[t] = u[t][up + i];
        y0[t] = u[t][N + row + i];
        yr[t] = u[t][N + row + ir];
#pragma unroll
        for (int q = 0; q < 3; q++) {
          // lanes 0-7 hold the even cell, lanes 8-15 the odd one: the even
          // cell's operand takes its imaginary parts to lanes 8-15, the odd
          // cell's its real parts to lanes 0-7
          F[t][q][0] = lane_xor8<0xc>(f[q].r, f[q].i);
          F[t][q][1] = lane_xor8<0x3>(f[q].i, f[q].r);
        }
        if (LAST && t + 1 < Q) continue;
        const double a0 = e0 * F[t][0][0], a1 = e1 * F[t][0][1];
        const int p0 = LAST ? 0 : t * (t + 1) / 2;
        auto mac = [&](v4d* acc, double l, int q, int cell2) {
#pragma unroll
          for (int c = 0; c <= t; c++)
            acc[p0 + c] = __builtin_amdgcn_mfma_f64_16x16x4f64(l, F[c][q][cell2], acc[p0 + c], 0, 0, 0);
        };
        if (MATS & 1) mac(K, a0, 0, 0);
        if (MATS & 2) mac(M, F[t][1][0], 1, 0);
        if (MATS & 1) mac(K, a1, 0, 1);
        if (MATS & 2) {
          mac(M, F[t][1][1], 1, 1);
          mac(M, F[t][2][0], 2, 0);
          mac(M, F[t][2][1], 2, 1);
        }
      }
    };
    int j = ja;
    if (!last)
      for (const int je = min(jb, ny - 1); j < je; j++) row_step(j, gram_false());
    for (; j < jb; j++) row_step(j, gram_true());
  }
  // Element e of a tile in lane (j = lane & 15, im = lane >> 4) is row 4 e +
  // im, column j.  With a = row & 7, b = column & 7 the complex sum is
  // rr + ii + i (ri - ir): lanes j < 8 form the real part of rows 4 e + im,
  // e < 2, lanes j >= 8 the imaginary part.  Summed over the waves in order.
  constexpr int NM = MATS == 3 ? 2 : 1, PER = NP * NM * 128;  // matrices; sums of a wave
#pragma unroll
  for (int p = 0; p < NP; p++)
#pragma unroll
    for (int mat = 0; mat < NM; mat++) {
      const v4d d = mat || MATS == 2 ? M[p] : K[p];
#pragma unroll
      for (int e = 0; e < 2; e++) {
        const double o = lane_xor8<0xf>(0.0, d[e + 2]);
        lds[wave * PER + ((p * NM + mat) * 2 + e) * 64 + lane] = h ? d[e] - o : d[e] + o;
      }
    }
  __syncthreads();
  for (int w = tid; w < PER; w += 256) {
    const int l = w & 63, e = (w >> 6) & 1, p = w / (NM * 128);
    const int mat = MATS == 3 ? (w >> 7) & 1 : MATS - 1;
    int T = Q - 1, S = p;
    if (!LAST) pair_ab(p, T, S);
    const int a = 8 * T + 4 * e + (l >> 4), b = 8 * S + (l & 7);
    if (a < g.mq && b <= a)
      g.out[4 * (a * (a + 1) / 2 + b) + 2 * mat + ((l >> 3) & 1)] =
          ((lds[w] + lds[PER + w]) + lds[2 * PER + w]) + lds[3 * PER + w];
  }
}

// A workgroup covers a band of rows of one problem; bands are summed by
// k_reduce_partials in a fixed order.  NT: tiles of the widest block.  With a
// column list (cmap: per problem q, cmap[q (m+1)] = mq columns, then their
// indices in the block, increasing) a problem's sums run over those mq
// columns only and land at the pair indices of the list (pair a (a+1)/2 + b
// of list positions a >= b); the rest of its output is left unwritten.
// Workgroups z = 0 take the first FIRST tiles and all their pairs, z > 0 tile
// FIRST + z - 1 with itself and those before.  All six tiles in one workgroup go over
// their rows twice, for K and for M: the sums of 21 pairs of both would not fit in
// registers.
template <int NT, int FIRST>
__global__ __launch_bounds__(256, NT <= 2 ? 2 : 1) void k_gram(mxh_level lv, mxh_bloch bl, int m, const int* pmap,
                                                               const int* cmap, const C<double>* U0, long long us,
                                                               const double* eta, double* part, int rpb)
{
  extern __shared__ double smem[];
  const int jb = blockIdx.y;
  const int prob = pmap ? pmap[jb] : jb;
  const int* cl = cmap ? cmap + (size_t)prob * (m + 1) : nullptr;
  const int mq = cl ? cl[0] : m;  // columns summed (block-uniform)
  if (mq < 1 || mq > m) return;   // (the whole block: before any barrier)
  const Geo<double> gg = make_geo<double>(lv, bl, prob * m);
  GramArgs g;
  g.U = U0 + (size_t)prob * m * us;
  g.us = us;
  g.cl = cl ? cl + 1 : nullptr;
  g.eta = eta;
  g.out = part + ((size_t)blockIdx.x * gridDim.y + jb) * 4 * (m * (m + 1) / 2);
  g.xf = gg.xf;
  g.yf = gg.yf;
  // the mass factors' weights: sqrt(6 mx) a, sqrt(6 mx) b (x-edges), sqrt(6 my) a, sqrt(6 my) b
  const double fa = 0.5 * (1.0 + 1.0 / sqrt(3.0)), fb = 0.5 * (1.0 - 1.0 / sqrt(3.0));
  const double sxm = sqrt(lv.hy / lv.hx), sym = sqrt(lv.hx / lv.hy);
  g.xa = sxm * fa;
  g.xb = sxm * fb;
  g.ya = sym * fa;
  g.yb = sym * fb;
  g.nx = lv.nx;
  g.ny = lv.ny;
  g.mq = mq;
  g.j0 = min(lv.ny, (int)blockIdx.x * rpb);
  g.j1 = min(lv.ny, g.j0 + rpb);
  // the tiles this problem's columns fill (uniform)
  const int nt = min((mq + 7) / 8, NT), z = (int)blockIdx.z;
  if (z == 0) {
    switch (min(nt, FIRST)) {
    case 1: gram_rows<1>(g, smem); break;
    case 2: if constexpr (FIRST >= 2) gram_rows<2>(g, smem); break;
    case 3: if constexpr (FIRST >= 3) gram_rows<3>(g, smem); break;
    case 4: if constexpr (FIRST >= 4) gram_rows<4>(g, smem); break;
    case 5: if constexpr (FIRST >= 5) gram_rows<5>(g, smem); break;
    case 6:
      if constexpr (FIRST >= 6) {
        gram_rows<6, false, 1>(g, smem);
        __syncthreads();
        gram_rows<6, false, 2>(g, smem);
      }
      break;
    }
  } else if (FIRST + z <= nt) {
    switch (FIRST + z) {
    case 4: if constexpr (NT >= 4 && FIRST < 4) gram_rows<4, true>(g, smem); break;
    case 5: if constexpr (NT >= 5 && FIRST < 5) gram_rows<5, true>(g, smem); break;
    case 6: if constexpr (NT >= 6 && FIRST < 6) gram_rows<6, true>(g, smem); break;
    }
  }
}

// ----------------------------------------------------------------- Ritz problems
// The small generalised eigenproblems of the Rayleigh-Ritz step, one workgroup
// per problem, from the Gram sums of k_gram: A = sk K + M and B = M over the
// problem's n columns (at most 48).  The columns are scaled to unit M-norm and
// taken in order, each kept only if its pivot in the Cholesky factorisation of
// the scaled B (the squared sine of its angle to the columns kept before it)
// exceeds pivot; then C = L^-1 A L^-H, cyclic Jacobi with the rotations of a
// round-robin round (n / 2 disjoint pairs) applied together, and X = L^-H Y.
// The lowest m pairs give lam and the coefficient block, with basis > 0 (the
// LOBPCG basis of `basis` columns) basis x 2m: the Ritz vectors and once more
// without their first m rows.  status: 0, 1 a sum is not finite, 2 fewer than
// m columns kept; the coefficients are then 0.
//
// A rotation is (c, -f; conj(f), c) with c real (and exactly 1 for an angle whose
// square is lost against 1), not one that turns a column by a phase: a pair that
// has converged keeps the coefficient 1 and its vector every bit.  Multiplied by
// a new phase in each step it is rounded anew, and where rounding is all its
// residual holds (eps |K| / lambda: 1e-8 on 512^2 at |k| = 0.12) the pair leaves
// the tolerance again: of 64 LOBPCG start blocks 14 stalled that way, 0 do now.
//
// Everything stays in LDS in FP64; a step of a factorisation or substitution
// has one barrier, a Jacobi round two.  What bounds it is that chain (per round
// a rotation's square roots, a barrier, the LDS reads and writes of A and V, a
// barrier): 51 us a step of a solve with 64 problems of 12 columns, all of which
// run at once; random dense pencils, which need more sweeps, 73 us for 16 of 9
// columns and 945 us for 64 of 36.  On the host the same problems took 0.5 to
// 1 ms between device steps that wait for them (64^2 grids in FP64, 16 problems:
// a solve of 80 ms against 56) and needed two transfers.  LOBPCG's bases of three
// blocks stay on the host, where they run beside the device (bloch_solver.c).
#define RITZ_MAX 48

MXH_DEV double rsqrt64(double a)
{
  double r = __builtin_amdgcn_rsq(a);
  r = r * fma(-0.5 * a * r, r, 1.5);
  return r * fma(-0.5 * a * r, r, 1.5);
}

__global__ __launch_bounds__(1024) void k_ritz(int m, int basis, const int* pmap, const int* cmap, const double* gram,
                                              double sk, double pivot, double* Cout, double* lam,
                                              int vpp, int* status)
{
  extern __shared__ double smem[];
  const int jb = blockIdx.x, prob = pmap ? pmap[jb] : jb, tid = threadIdx.x, bd = blockDim.x;
  const int k = basis ? basis : m, np = k * (k + 1) / 2;
  const int* cl = cmap ? cmap + (size_t)prob * (k + 1) : nullptr;
  const int n = cl ? min(cl[0], k) : k;
  C<double>*A = (C<double>*)smem, *B = A + n * n, *Vv = B + n * n;
  __shared__ double dsc[RITZ_MAX], w[RITZ_MAX], rc[RITZ_MAX / 2], red[16];
  __shared__ C<double> rs[RITZ_MAX / 2];
  __shared__ int keep[RITZ_MAX], ord[RITZ_MAX], bad;
  const double* g = gram + 4 * (size_t)np * jb;
  const int csz = basis ? basis * 2 * m : m * m;
  C<double>* Cj = (C<double>*)Cout + (size_t)jb * csz;
  if (tid == 0) bad = 0;
  for (int e = tid; e < csz; e += bd) Cj[e] = czero<double>();
  __syncthreads();
  // column-major A and B, lower triangle of the sums mirrored
  for (int e = tid; e < n * n; e += bd) {
    const int c = e / n, a = e - c * n, hi = max(a, c), lo = min(a, c);
    const double* q = g + 4 * (hi * (hi + 1) / 2 + lo);
    const double q0 = q[0], q1 = q[1], q2 = q[2], q3 = q[3];
    if (!(isfinite(q0) && isfinite(q1) && isfinite(q2) && isfinite(q3))) bad = 1;
    const double s = a >= c ? 1.0 : -1.0;
    B[e] = cmk(q2, a == c ? 0.0 : s * q3);
    A[e] = cmk(sk * q0 + q2, a == c ? 0.0 : s * (sk * q1 + q3));
  }
  __syncthreads();
  if (bad) {
    if (tid == 0) status[jb] = 1;
    return;
  }
  if (tid < n) {
    const double b = B[tid + tid * n].r;
    dsc[tid] = b > 0.0 ? 1.0 / sqrt(b) : 0.0;  // 0: never kept
  }
  __syncthreads();
  for (int e = tid; e < n * n; e += bd) {
    const int c = e / n, a = e - c * n;
    const double s = dsc[a] * dsc[c];
    A[e] = s * A[e];
    B[e] = s * B[e];
  }
  // pivots in order; a kept column's multiples leave the rest (right-looking)
  const int ti = tid & 15, tj = tid >> 4, sj = bd >> 4;
  int kk = 0;
  for (int c = 0; c < n; c++) {
    __syncthreads();
    const double piv = B[c + c * n].r;
    if (!(piv > pivot)) continue;  // uniform
    if (tid == 0) keep[kk] = c;
    kk++;
    const double inv = 1.0 / piv;
    for (int j = c + 1 + tj; j < n; j += sj) {
      const C<double> f = inv * cconj(B[j + c * n]);
      for (int i = j + ti; i < n; i += 16) B[i + j * n] -= B[i + c * n] * f;
    }
  }
  __syncthreads();
  if (kk < m) {
    if (tid == 0) status[jb] = 2;
    return;
  }
  // the kept rows and columns, with leading dimension kk: the factor L (lower)
  // and the matrix
  for (int e = tid; e < kk * kk; e += bd) {
    const int u = e / kk, t = e - u * kk, ku = keep[u], kt = keep[t];
    Vv[e] = t > u ? (1.0 / sqrt(B[ku + ku * n].r)) * B[kt + ku * n]
                  : (t == u ? cmk(sqrt(B[ku + ku * n].r), 0.0) : czero<double>());
  }
  __syncthreads();
  for (int e = tid; e < kk * kk; e += bd) B[e] = Vv[e];
  __syncthreads();
  for (int e = tid; e < kk * kk; e += bd) {
    const int u = e / kk, t = e - u * kk;
    Vv[e] = A[keep[t] + keep[u] * n];
  }
  __syncthreads();
  for (int e = tid; e < kk * kk; e += bd) A[e] = Vv[e];
  // A <- L^-1 A (rows, divided by the diagonal at the end), then A L^-H
  for (int r = 0; r < kk; r++) {
    __syncthreads();
    const double inv = 1.0 / B[r + r * kk].r;
    for (int j = tj; j < kk; j += sj) {
      const C<double> f = inv * A[r + j * kk];
      for (int i = r + 1 + ti; i < kk; i += 16) A[i + j * kk] -= B[i + r * kk] * f;
    }
  }
  for (int r = 0; r < kk; r++) {
    __syncthreads();
    const double inv = 1.0 / B[r + r * kk].r;
    for (int j = r + 1 + tj; j < kk; j += sj) {
      const C<double> f = inv * cconj(B[j + r * kk]);
      for (int i = ti; i < kk; i += 16) A[i + j * kk] -= A[i + r * kk] * f;
    }
  }
  __syncthreads();
  for (int e = tid; e < kk * kk; e += bd) {
    const int j = e / kk, i = e - j * kk;
    const C<double> a = A[i + j * kk], b = cconj(A[j + i * kk]);
    Vv[e] = (0.5 / (B[i + i * kk].r * B[j + j * kk].r)) * (a + b);
  }
  __syncthreads();
  for (int e = tid; e < kk * kk; e += bd) {
    const int j = e / kk, i = e - j * kk;
    A[e] = i == j ? cmk(Vv[e].r, 0.0) : Vv[e];
    Vv[e] = cmk(i == j ? 1.0 : 0.0, 0.0);
  }
  // Jacobi
  const int h = (kk + 1) / 2, ne = 2 * h;
  // this thread's items of a round: 2 x 2 blocks (slots P, K), then rows i of V
  // for slot K (P = -1 - i); none: K < 0.  At most two (mxh_ritz)
  int itP[2], itK[2];
#pragma unroll
  for (int u = 0; u < 2; u++) {
    const int x = tid + u * bd, y = x - h * h;
    itK[u] = x >= h * h + kk * h ? -1 : (y < 0 ? x / h : y / kk);
    itP[u] = y < 0 ? x % h : -1 - y % kk;
  }
  for (int sweep = 0; sweep < 64; sweep++) {
    __syncthreads();
    double off = 0.0, dia = 0.0;
    for (int e = tid; e < kk * kk; e += bd) {
      const double t = A[e].r * A[e].r + A[e].i * A[e].i;
      if (e / kk == e % kk) dia += t;
      else off += t;
    }
    off = wave_sum(off);
    dia = wave_sum(dia);
    if ((tid & 63) == 0) {
      // one slot pair per wave (at most 16 waves)
      w[tid >> 6] = off;
      red[tid >> 6] = dia;
    }
    __syncthreads();
    off = dia = 0.0;
    for (int q = 0; q < bd >> 6; q++) {
      off += w[q];
      dia += red[q];
    }
    if (off <= 1e-32 * dia) break;  // uniform
    for (int round = 0; round < ne - 1; round++) {
      // round-robin pairs: index ne - 1 stays, the others rotate (slot 0 holds
      // it); an index >= kk is the dummy of an odd count
      auto first = [&](int slot) {
        const int a = round + slot;
        return slot == 0 ? ne - 1 : (a >= ne - 1 ? a - (ne - 1) : a);
      };
      auto second = [&](int slot) {
        const int a = round - slot;
        return slot == 0 ? round : (a < 0 ? a + ne - 1 : a);
      };
      if (tid < h) {
        const int p = first(tid), q = second(tid);
        double cs = 1.0;
        C<double> f = czero<double>();
        if (p < kk) {
          const C<double> z = A[p + q * kk];
          const double z2 = z.r * z.r + z.i * z.i;
          if (z2 > 1e-290) {
            const double ri = rsqrt64(z2), r = z2 * ri, d = A[q + q * kk].r - A[p + p * kk].r;
            const double s2 = d * d + 4.0 * z2;
            const double t = copysign(2.0 * r, d) * recip(fabs(d) + s2 * rsqrt64(s2));
            // exactly 1 for the angles that leave a column as it is
            if (t * t > 0x1p-53) cs = rsqrt64(1.0 + t * t);
            f = (t * cs * ri) * cconj(z);
          }
        }
        rc[tid] = cs;
        rs[tid] = f;
      }
      __syncthreads();
      // A <- J^H A J on the 2 x 2 blocks of pairs, V <- V J: an item's slots
      // are fixed, its rows and columns follow from the round
#pragma unroll
      for (int u = 0; u < 2; u++) {
        if (itK[u] < 0) continue;
        const int K = itK[u], s = first(K), t = second(K);
        const double cK = rc[K];
        const C<double> fK = rs[K], gK = cconj(fK), z0 = czero<double>();
        const bool ok_s = s < kk;
        if (itP[u] >= 0) {
          const int P = itP[u], p = first(P), q = second(P);
          const bool ok_p = p < kk;
          C<double> a = ok_p && ok_s ? A[p + s * kk] : z0, b = ok_p ? A[p + t * kk] : z0;
          C<double> c = ok_s ? A[q + s * kk] : z0, d = A[q + t * kk];
          // columns: s' = c s - f t, t' = conj(f) s + c t
          const double cP = rc[P];
          const C<double> fP = rs[P], gP = cconj(fP);
          const C<double> a1 = cK * a - fK * b, b1 = gK * a + cK * b, c1 = cK * c - fK * d, d1 = gK * c + cK * d;
          // rows: p' = c p - conj(f) q, q' = f p + c q
          a = cP * a1 - gP * c1;
          c = fP * a1 + cP * c1;
          b = cP * b1 - gP * d1;
          d = fP * b1 + cP * d1;
          if (P == K) {
            a.i = d.i = 0.0;
            b = c = z0;
          }
          if (ok_p && ok_s) A[p + s * kk] = a;
          if (ok_p) A[p + t * kk] = b;
          if (ok_s) A[q + s * kk] = c;
          A[q + t * kk] = d;
        } else if (ok_s) {
          const int i = -1 - itP[u];
          const C<double> a = Vv[i + s * kk], b = Vv[i + t * kk];
          Vv[i + s * kk] = cK * a - fK * b;
          Vv[i + t * kk] = gK * a + cK * b;
        }
      }
      __syncthreads();
    }
  }
  __syncthreads();
  if (tid < kk) {
    const double v = A[tid + tid * kk].r;
    int r = 0;
    for (int j = 0; j < kk; j++) {
      const double u = A[j + j * kk].r;
      r += u < v || (u == v && j < tid);
    }
    ord[r] = tid;
    w[r] = v;
  }
  __syncthreads();
  for (int i = tid; i < m; i += bd) lam[(size_t)prob * vpp + i] = w[i];
  // X = L^-H Y for the lowest m (rows divided by the diagonal at the end)
  for (int r = kk - 1; r >= 0; r--) {
    __syncthreads();
    const double inv = 1.0 / B[r + r * kk].r;
    for (int j = tj; j < m; j += sj) {
      C<double>* y = Vv + ord[j] * kk;
      const C<double> f = inv * y[r];
      for (int i = ti; i < r; i += 16) y[i] -= cconj(B[r + i * kk]) * f;
    }
  }
  __syncthreads();
  for (int e = tid; e < kk * m; e += bd) {
    const int i = e / kk, t = e - i * kk, pos = keep[t], c = cl ? cl[1 + pos] : pos;
    const C<double> z = (dsc[pos] / B[t + t * kk].r) * Vv[t + ord[i] * kk];
    Cj[c + (size_t)i * k] = z;
    if (basis && c >= m) Cj[c + (size_t)(m + i) * k] = z;
  }
  if (tid == 0) status[jb] = 0;
}

// ----------------------------------------------------------------- block combine
// Per problem: out_j = sum_a C[a + j nin] in_a over nin input vectors, for
// nout outputs, every input read once.  Output j goes to slot j of the
// problem's output block, or to slot j + gap from j = nsplit on (the LOBPCG
// layout [E | W | P] writes E and P and skips W).  A thread owns one complex
// entry of every output; NOUT (16 or 32) is the accumulator count.
#define COMBX_NIN_MAX 48
template <int NOUT>
__global__ __launch_bounds__(256) void k_combine_x(long long n, int nin, int nout, int nsplit, int gap,
                                                   const int* pmap, const C<double>* X0, long long xs, int xvpp,
                                                   C<double>* Y0, long long ys, int yvpp, const double* Cm0)
{
  __shared__ C<double> sC[COMBX_NIN_MAX * NOUT];
  const int jb = blockIdx.y;
  const int prob = pmap ? pmap[jb] : jb;
  const C<double>* X = X0 + (size_t)prob * xvpp * xs;
  C<double>* Y = Y0 + (size_t)prob * yvpp * ys;
  const C<double>* Cm = (const C<double>*)Cm0 + (size_t)jb * nin * nout;
  // coefficients as [a][j] with a row of NOUT (zero beyond nout)
  for (int w = threadIdx.x; w < nin * NOUT; w += blockDim.x) {
    const int a = w / NOUT, j = w - a * NOUT;
    sC[w] = j < nout ? Cm[a + (size_t)j * nin] : czero<double>();
  }
  __syncthreads();
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)n) return;
  C<double> acc[NOUT];
#pragma unroll
  for (int q = 0; q < NOUT; q++) acc[q] = czero<double>();
  int a = 0;
  for (; a + 2 <= nin; a += 2) {
    const C<double> u0 = X[(size_t)a * xs + idx], u1 = X[(size_t)(a + 1) * xs + idx];
    const C<double>* c0 = sC + a * NOUT;
#pragma unroll
    for (int q = 0; q < NOUT; q++) acc[q] += c0[q] * u0 + c0[NOUT + q] * u1;
  }
  if (a < nin) {
    const C<double> u0 = X[(size_t)a * xs + idx];
    const C<double>* c0 = sC + a * NOUT;
#pragma unroll
    for (int q = 0; q < NOUT; q++) acc[q] += c0[q] * u0;
  }
#pragma unroll
  for (int q = 0; q < NOUT; q++)
    if (q < nout) Y[(size_t)(q < nsplit ? q : q + gap) * ys + idx] = acc[q];
}

// LOBPCG block update of one problem's basis X = [E | W | P] (3m vectors)
// with the Ritz coefficients c (3m x m, column-major: c[a + q 3m] for output
// q): P_new_q = sum_{a >= m} c[a, q] x_a (the W and P part), then
// E_new_q = P_new_q + sum_{a < m} c[a, q] e_a, written to the E and P slots
// of Y.  Every input is read once and the shared part is summed once (3 m^2
// complex multiply-adds per entry instead of 6 m^2); NM >= m accumulators.
template <int NM>
__global__ __launch_bounds__(256) void k_lobpcg_combine(long long n, int m, const int* pmap, const C<double>* X0,
                                                        long long xs, C<double>* Y0, long long ys, const double* Cm0)
{
  __shared__ C<double> sC[48 * NM];
  // bit a: input a has a non-zero coefficient.  The Ritz step zeroes the
  // rows of the columns it drops (no P at the first step, the W of locked
  // vectors, dependent directions), and those inputs are not read at all.
  __shared__ unsigned long long rows_nz;
  const int jb = blockIdx.y;
  const int prob = pmap ? pmap[jb] : jb;
  const int k = 3 * m;
  const C<double>* X = X0 + (size_t)prob * k * xs;
  C<double>* Y = Y0 + (size_t)prob * k * ys;
  const C<double>* Cm = (const C<double>*)Cm0 + (size_t)jb * k * 2 * m;  // the E_new block of the 3m x 2m matrix
  if (threadIdx.x == 0) rows_nz = 0ull;
  for (int w = threadIdx.x; w < k * NM; w += blockDim.x) {
    const int a = w / NM, q = w - a * NM;
    sC[w] = q < m ? Cm[a + (size_t)q * k] : czero<double>();
  }
  __syncthreads();
  if ((int)threadIdx.x < k) {
    bool nz = false;
    for (int q = 0; q < m; q++) {
      const C<double> c = sC[threadIdx.x * NM + q];
      nz = nz || c.r != 0.0 || c.i != 0.0;
    }
    if (nz) atomicOr(&rows_nz, 1ull << threadIdx.x);
  }
  __syncthreads();
  const unsigned long long nzm = rows_nz;
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)n) return;
  C<double> acc[NM];
#pragma unroll
  for (int q = 0; q < NM; q++) acc[q] = czero<double>();
  // W and P part (2m inputs, m even), by pairs; an input whose row is zero
  // is not read (its slot may hold anything: the W of a locked vector, a P
  // before the first direction)
  for (int a = m; a < k; a += 2) {
    const bool n0 = (nzm >> a) & 1ull, n1 = (nzm >> (a + 1)) & 1ull;
    if (!n0 && !n1) continue;
    const C<double> u0 = n0 ? X[(size_t)a * xs + idx] : czero<double>();
    const C<double> u1 = n1 ? X[(size_t)(a + 1) * xs + idx] : czero<double>();
    const C<double>* c0 = sC + a * NM;
#pragma unroll
    for (int q = 0; q < NM; q++) acc[q] += c0[q] * u0 + c0[NM + q] * u1;
  }
#pragma unroll
  for (int q = 0; q < NM; q++)
    if (q < m) Y[(size_t)(2 * m + q) * ys + idx] = acc[q];
  for (int a = 0; a < m; a += 2) {
    const bool n0 = (nzm >> a) & 1ull, n1 = (nzm >> (a + 1)) & 1ull;
    if (!n0 && !n1) continue;
    const C<double> u0 = n0 ? X[(size_t)a * xs + idx] : czero<double>();
    const C<double> u1 = n1 ? X[(size_t)(a + 1) * xs + idx] : czero<double>();
    const C<double>* c0 = sC + a * NM;
#pragma unroll
    for (int q = 0; q < NM; q++) acc[q] += c0[q] * u0 + c0[NM + q] * u1;
  }
#pragma unroll
  for (int q = 0; q < NM; q++)
    if (q < m) Y[(size_t)q * ys + idx] = acc[q];
}

#define COMB_MMAX 48
__global__ __launch_bounds__(256) void k_block_combine(long long n, int m, const int* pmap, const C<double>* U0,
                                                       long long us, C<double>* E0, long long es, const double* Cm0)
{
  __shared__ C<double> sC[COMB_MMAX * COMB_MMAX];
  const int jb = blockIdx.y;
  const int prob = pmap ? pmap[jb] : jb;
  const C<double>* U = U0 + (size_t)prob * m * us;
  C<double>* E = E0 + (size_t)prob * m * es;
  const C<double>* Cm = (const C<double>*)Cm0 + (size_t)jb * m * m;
  for (int w = threadIdx.x; w < m * m; w += blockDim.x) sC[w] = Cm[w];
  __syncthreads();
  size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)n) return;
  for (int j0 = 0; j0 < m; j0 += 16) {
    C<double> acc[16];
#pragma unroll
    for (int q = 0; q < 16; q++) acc[q] = czero<double>();
    for (int a = 0; a < m; a++) {
      const C<double> u = U[(size_t)a * us + idx];
#pragma unroll
      for (int q = 0; q < 16; q++)
        if (j0 + q < m) acc[q] += sC[a + (j0 + q) * m] * u;
    }
#pragma unroll
    for (int q = 0; q < 16; q++)
      if (j0 + q < m) E[(size_t)(j0 + q) * es + idx] = acc[q];
  }
}

// ----------------------------------------------- Householder M-orthonormalisation
// The reference's unit vectors (edge2d.c:6154-6210): vector idx is the
// x-edge (i, j) with j = 1, 3, 5, ... taking idx row by row, scaled to unit
// M-norm, s = sqrt(0.25 / mx), mx = hy / (6 hx); they are M-orthonormal (M
// couples an x-edge only to the x-edges of the rows above and below).
MXH_DEV void unit_ij(int idx, int nx, int& i, int& j)
{
  i = idx % nx;
  j = 1 + 2 * (idx / nx);
}

// unit(i,j)^H M y = sqrt(0.25 mx) (4 y(i,j) + y(i,j-1) + y(i,j+1)), the row
// above the last one through the Bloch factor yf
MXH_DEV C<double> unit_mprod(const C<double>* y, int i, int j, int nx, int ny, double mx, C<double> yf)
{
  const C<double> up = j + 1 < ny ? y[i + (size_t)(j + 1) * nx] : yf * y[i];
  return sqrt(0.25 * mx) * (4.0 * y[i + (size_t)j * nx] + y[i + (size_t)(j - 1) * nx] + up);
}

// Forward pass, two launches a reflection.  k_hh_row(i) sums x_i^H M x_j over
// every later vector and x_i^H M v_j over every finished one, and p_j = unit_i^H M
// of each; k_hh_update(i) turns the sums into reflection i (edge2d.c:6238-6262):
// alpha = |x_i|_M with the sign of Re(beta), beta = p_i, v_i = x_i + alpha
// unit_i, tau = 1 / (alpha^2 + beta alpha) (0 when x_i = 0), and applies it to the
// later vectors, whose component along unit_i then goes (edge2d.c:6273-6285).
// Every workgroup finishes the sums it needs itself, so that nothing but the
// end of a launch orders the two; v_i stays x_i in memory until the next
// k_hh_row adds alpha unit_i to its one entry.
//
// The outputs V_i = H_0 ... H_i unit_i (H_j = I - conj(tau_j) v_j v_j^H M) all at
// once: with S_jl = v_j^H M v_l (j < l) and w = (v_j^H M unit_i)_j, V_i = unit_i
// - sum_j v_j c_j where c_j = conj(tau_j) (w_j - sum_{l > j} S_jl c_l), l <= i.
//
// Bound by the chain of 2 k launches on the drivers' grids: 24 vectors of 128^2
// 1.28 -> 0.42 ms against one launch per product, update and fix of both passes.
#define HH_NB 64  // partial sums per vector at most (one wave's lanes)
struct HhVecs {
  C<double>* base;  // vector j at base + j stride, or, with a table, table[j]
  long long stride;
  C<double>* const* table;
  MXH_DEV C<double>* at(int j) const { return table ? table[j] : base + (size_t)j * stride; }
};
// work: [hh: alpha, tau, unused per vector | p | partial sums | S | W -> c]
struct HhWork {
  double *hh, *p, *part, *S, *W;
};
static HhWork hh_work(double* w, int k)
{
  HhWork h;
  h.hh = w;
  h.p = h.hh + 4 * (size_t)k;
  h.part = h.p + 2 * (size_t)k;
  h.S = h.part + 2 * HH_NB * (size_t)k;
  h.W = h.S + 2 * (size_t)k * k;
  return h;
}

__global__ __launch_bounds__(256) void k_hh_row(mxh_level lv, C<double> xf, C<double> yf, int idx, HhVecs X,
                                                HhWork wk)
{
  __shared__ double sh[4];
  const int nx = lv.nx, ny = lv.ny, j = blockIdx.y, tid = threadIdx.x;
  const size_t N = (size_t)nx * ny;
  const double mx = lv.hy / lv.hx / 6.0, my = lv.hx / lv.hy / 6.0;
  const C<double>*x = X.at(idx), *y = x + N;
  C<double>* u = X.at(j);
  int i0, j0;
  size_t fix = ~(size_t)0;  // v_{idx - 1}: alpha unit still to be added
  double add = 0.0;
  if (idx > 0 && j == idx - 1) {
    unit_ij(j, nx, i0, j0);
    fix = i0 + (size_t)j0 * nx;
    add = wk.hh[4 * j] * sqrt(0.25 / mx);
  }
  double sr = 0.0, si = 0.0;
  for (size_t e = (size_t)blockIdx.x * blockDim.x + tid; e < N; e += (size_t)gridDim.x * blockDim.x) {
    const int r = (int)((unsigned)e / (unsigned)nx), c = (int)e - r * nx;
    const C<double> dn = r ? x[e - nx] : cconj(yf) * x[e + N - nx], up = r + 1 < ny ? x[e + nx] : yf * x[c];
    const C<double> lf = c ? y[e - 1] : cconj(xf) * y[e + nx - 1], rt = c + 1 < nx ? y[e + 1] : xf * y[e - c];
    const C<double> a = mx * (4.0 * x[e] + dn + up), b = my * (4.0 * y[e] + lf + rt);
    C<double> p = u[e];
    const C<double> q = u[N + e];
    if (e == fix) {
      p.r += add;
      u[e] = p;
    }
    sr += a.r * p.r + a.i * p.i + b.r * q.r + b.i * q.i;
    si += a.r * p.i - a.i * p.r + b.r * q.i - b.i * q.r;
  }
  sr = block_sum256(sr, sh);
  si = block_sum256(si, sh);
  if (tid == 0) {
    double* o = wk.part + 2 * ((size_t)j * HH_NB + blockIdx.x);
    o[0] = sr;
    o[1] = si;
    if (blockIdx.x == 0) {
      unit_ij(idx, nx, i0, j0);
      const C<double> p = unit_mprod(u, i0, j0, nx, ny, mx, yf);
      wk.p[2 * j] = p.r;
      wk.p[2 * j + 1] = p.i;
    }
  }
}

// the sum of vector j's nb partial sums (whole waves)
MXH_DEV C<double> hh_sum(const HhWork& wk, int j, int nb)
{
  const int l = threadIdx.x & 63;
  const double* q = wk.part + 2 * ((size_t)j * HH_NB + l);
  return cmk(wave_sum(l < nb ? q[0] : 0.0), wave_sum(l < nb ? q[1] : 0.0));
}

// grid (blocks, k - idx): vector idx + blockIdx.y; nb: blocks of k_hh_row.  The
// workgroups of vector idx share the products with the finished vectors, a wave's
// sum each (64^2, 300 vectors: 40 us a launch where one workgroup formed them all).
__global__ __launch_bounds__(256) void k_hh_update(mxh_level lv, int idx, int k, int nb, HhVecs X, HhWork wk)
{
  const int nx = lv.nx, tid = threadIdx.x, j = idx + blockIdx.y;
  const size_t E = 2 * (size_t)nx * lv.ny;
  const double sc = sqrt(0.25 / (lv.hy / lv.hx / 6.0));
  const C<double> beta = cmk(wk.p[2 * idx], wk.p[2 * idx + 1]);
  double alpha = sqrt(hh_sum(wk, idx, nb).r);
  C<double> tau = czero<double>();
  if (alpha != 0.0) {
    if (beta.r < 0.0) alpha = -alpha;
    const C<double> den = cmk(alpha * alpha + beta.r * alpha, beta.i * alpha);
    const double dd = den.r * den.r + den.i * den.i;
    tau = cmk(den.r / dd, -den.i / dd);
  }
  const C<double> uv = cmk(beta.r + alpha, beta.i);  // unit^H M v
  C<double>*S = (C<double>*)wk.S, *W = (C<double>*)wk.W;
  if (j == idx) {
    for (int l = 4 * (int)blockIdx.x + (tid >> 6); l < idx; l += 4 * (int)gridDim.x) {
      const C<double> d = hh_sum(wk, l, nb), p = cmk(wk.p[2 * l], -wk.p[2 * l + 1]);
      if ((tid & 63) == 0) {
        S[(size_t)l * k + idx] = cconj(d) + alpha * p;
        W[(size_t)l * k + idx] = p;
      }
    }
    if (tid == 0 && blockIdx.x == 0) {
      W[(size_t)idx * k + idx] = cconj(uv);
      wk.hh[4 * idx] = alpha;
      wk.hh[4 * idx + 1] = tau.r;
      wk.hh[4 * idx + 2] = tau.i;
    }
    return;
  }
  const C<double> pj = cmk(wk.p[2 * j], wk.p[2 * j + 1]);
  const C<double> c = -1.0 * (tau * (hh_sum(wk, j, nb) + alpha * pj));
  int i0, j0;
  unit_ij(idx, nx, i0, j0);
  const size_t at = i0 + (size_t)j0 * nx;
  const C<double>* x = X.at(idx);
  C<double>* y = X.at(j);
  for (size_t e = (size_t)blockIdx.x * blockDim.x + tid; e < E; e += (size_t)gridDim.x * blockDim.x) {
    C<double> v = x[e], u = y[e];
    if (e == at) {
      v.r += alpha * sc;
      u -= sc * (pj + c * uv);
    }
    y[e] = u + c * v;
  }
}

// the coefficients c (in W) by back substitution and what the last k_hh_row would
// have finished: v_{k - 1}; tau to both outputs.  Up to HH_LDS vectors one workgroup
// in LDS; more: HH_COLS columns, which do not depend on each other, to a workgroup
// (300 vectors: 2.2 ms in one workgroup)
#define HH_LDS 48
#define HH_COLS 16
__global__ __launch_bounds__(1024) void k_hh_coef(mxh_level lv, int k, HhVecs X, HhWork wk, double* tau, double* host)
{
  extern __shared__ double smem[];
  const int tid = threadIdx.x, bd = blockDim.x;
  C<double>*S = (C<double>*)wk.S, *W = (C<double>*)wk.W;
  C<double>*s = S, *w = W;
  const int ia = k <= HH_LDS ? 0 : (int)blockIdx.x * HH_COLS, ib = k <= HH_LDS ? k : min(k, ia + HH_COLS);
  if (k <= HH_LDS) {  // 73 KB
    s = (C<double>*)smem;
    w = s + k * k;
    for (int e = tid; e < k * k; e += bd) {
      s[e] = S[e];
      w[e] = W[e];
    }
  }
  for (int j = ib - 1; j >= 0; j--) {
    __syncthreads();
    const C<double> t = cmk(wk.hh[4 * j + 1], -wk.hh[4 * j + 2]);
    const int first = max(ia, j), cols = ib - first;
    for (int e = tid; e < j * cols; e += bd) {
      const int r = e / cols, i = first + e - r * cols;
      w[(size_t)r * k + i] -= s[(size_t)r * k + j] * (t * w[(size_t)j * k + i]);
    }
  }
  __syncthreads();
  for (int e = tid; e < ib * (ib - ia); e += bd) {
    const int j = e / (ib - ia), i = ia + e - j * (ib - ia);
    if (i >= j) W[(size_t)j * k + i] = cmk(wk.hh[4 * j + 1], -wk.hh[4 * j + 2]) * w[(size_t)j * k + i];
  }
  if (blockIdx.x) return;
  for (int j = tid; j < k; j += bd) {
    const double r = wk.hh[4 * j + 1], i = wk.hh[4 * j + 2];
    if (tau) {
      tau[2 * j] = r;
      tau[2 * j + 1] = i;
    }
    if (host) {
      host[2 * j] = r;
      host[2 * j + 1] = i;
    }
  }
  if (tid == 0) {
    int i0, j0;
    unit_ij(k - 1, lv.nx, i0, j0);
    X.at(k - 1)[i0 + (size_t)j0 * lv.nx].r += wk.hh[4 * (k - 1)] * sqrt(0.25 / (lv.hy / lv.hx / 6.0));
  }
}

// V_i = unit_i - sum_{j <= i} v_j c_ji, eight outputs at a time from the last
// ones down: V may be X.  Eight vectors' entries and the 8 x 8 coefficients (one
// a lane, handed round by v_readlane) are loaded while the eight before are used;
// with a scalar load per coefficient and no load ahead the step took 5 us (300
// vectors of 64^2 3.5 ms, 24 of 128^2 33 us).
__global__ __launch_bounds__(64) void k_hh_out(mxh_level lv, int k, HhVecs X, HhVecs V,
                                               const C<double>* __restrict__ cf)
{
  const size_t N = (size_t)lv.nx * lv.ny, at = (size_t)blockIdx.x * 64 + threadIdx.x, e = at < 2 * N ? at : 0;
  const int lj = threadIdx.x >> 3, lq = threadIdx.x & 7;
  // the unit vector whose entry e is
  const unsigned row = (unsigned)(e < N ? e : 0) / (unsigned)lv.nx;
  const long long unit = e < N && (row & 1) ? (long long)(row >> 1) * lv.nx + (long long)(e - (size_t)row * lv.nx) : -1;
  const double sc = sqrt(0.25 / (lv.hy / lv.hx / 6.0));
  for (int i0 = (k - 1) & ~7; i0 >= 0; i0 -= 8) {
    const int m = min(8, k - i0);
    C<double> acc[8], v[8], c;
    auto load = [&](int j0) {
#pragma unroll
      for (int j = 0; j < 8; j++) v[j] = X.at(min(j0 + j, k - 1))[e];
      c = cf[(size_t)min(j0 + lj, k - 1) * k + min(i0 + lq, k - 1)];
    };
    // (vectors past the last one only reach outputs that are not written)
    auto step = [&](const C<double>* u, C<double> d, bool diag) {
#pragma unroll
      for (int j = 0; j < 8; j++)
#pragma unroll
        for (int q = 0; q < 8; q++)
          if (!diag || q >= j) acc[q] -= lane_value(d, 8 * j + q) * u[j];
    };
#pragma unroll
    for (int q = 0; q < 8; q++) acc[q] = cmk(unit == i0 + q ? sc : 0.0, 0.0);
    load(0);
    for (int j0 = 0; j0 < i0; j0 += 8) {
      C<double> u[8], d = c;
#pragma unroll
      for (int j = 0; j < 8; j++) u[j] = v[j];
      load(j0 + 8);
      step(u, d, false);
    }
    step(v, c, true);
    if (at < 2 * N) {
#pragma unroll
      for (int q = 0; q < 8; q++)
        if (q < m) V.at(i0 + q)[e] = acc[q];
    }
  }
}

template <typename T>
__global__ __launch_bounds__(256) void k_gather(long long n, C<T>* D, long long ds, const C<T>* S, long long ss,
                                                const int* smap)
{
  const int v = blockIdx.y;
  size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)n) return;
  D[(size_t)v * ds + idx] = S[(size_t)smap[v] * ss + idx];
}

// ------------------------------------------------ pointwise edge Gauss-Seidel
// One colour of the pointwise (one edge at a time) Gauss-Seidel smoother for
// alpha K + beta M (edge2d.c:3892-5600, the smoother of the Hiptmair cycle):
// x_e += (b - A x)_e / A_ee.  An x-edge couples to x-edges only in the rows
// above and below, a y-edge to y-edges only in the columns left and right,
// so colours 0 / 1 (x-edges of even / odd rows) and 2 / 3 (y-edges of even /
// odd columns) are independent sets on grids with even nx and ny.
template <typename T>
__global__ __launch_bounds__(256) void k_edge_gs_phase(mxh_level lv, mxh_bloch bl, const C<T>* B, long long bs,
                                                       C<T>* X, long long xs, const T* eta, mxh_coef cf,
                                                       int colour)
{
  const int v = blockIdx.y;
  const size_t N = (size_t)lv.nx * lv.ny;
  size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= N / 2) return;
  Geo<T> g = make_geo<T>(lv, bl, v);
  C<T> axy, mx, my;
  coefs<T>(lv, cf, v, axy, mx, my);
  C<T>* xv = X + (size_t)v * xs;
  const C<T>* ex = xv;
  const C<T>* ey = xv + N;
  const C<T>* b = B + (size_t)v * bs;
  if (colour < 2) {  // x-edge (i, j), j of parity colour
    const int i = (int)(p % lv.nx), j = 2 * (int)(p / lv.nx) + colour;
    const C<T> x00 = g.at(ex, i, j);
    const C<T> c00 = x00 - g.at(ex, i, j + 1) - g.at(ey, i, j) + g.at(ey, i + 1, j);          // cell (i, j)
    const C<T> c0m = g.at(ex, i, j - 1) - x00 - g.at(ey, i, j - 1) + g.at(ey, i + 1, j - 1);  // cell (i, j-1)
    const T e00 = eta_at(eta, g.nx, g.ny, i, j), e0m = eta_at(eta, g.nx, g.ny, i, j - 1);
    const C<T> ax = axy * (e00 * c00 - e0m * c0m) + mx * (T(4) * x00 + g.at(ex, i, j - 1) + g.at(ex, i, j + 1));
    const C<T> diag = (e00 + e0m) * axy + T(4) * mx;
    const size_t k = i + (size_t)j * lv.nx;
    xv[k] = x00 + cdiv(b[k] - ax, diag);
  } else {  // y-edge (i, j), i of parity colour - 2
    const int hx2 = lv.nx >> 1;
    const int i = 2 * (int)(p % hx2) + (colour - 2), j = (int)(p / hx2);
    const C<T> y00 = g.at(ey, i, j);
    const C<T> c00 = g.at(ex, i, j) - g.at(ex, i, j + 1) - y00 + g.at(ey, i + 1, j);          // cell (i, j)
    const C<T> cm0 = g.at(ex, i - 1, j) - g.at(ex, i - 1, j + 1) - g.at(ey, i - 1, j) + y00;  // cell (i-1, j)
    const T e00 = eta_at(eta, g.nx, g.ny, i, j), em0 = eta_at(eta, g.nx, g.ny, i - 1, j);
    const C<T> ay = axy * (em0 * cm0 - e00 * c00) + my * (T(4) * y00 + g.at(ey, i - 1, j) + g.at(ey, i + 1, j));
    const C<T> diag = (e00 + em0) * axy + T(4) * my;
    const size_t k = N + i + (size_t)j * lv.nx;
    xv[k] = y00 + cdiv(b[k] - ay, diag);
  }
}

// ----------------------------------------------------------------- node space
template <typename T>
struct NodeCoef {
  T ac, ax, ay, ad;
};

template <typename T>
MXH_DEV NodeCoef<T> node_coef(const mxh_level& lv, double alpha)
{
  const double hx = lv.hx, hy = lv.hy;
  NodeCoef<T> c;
  c.ac = T(4.0 * alpha * (hx / hy + hy / hx) / 3.0);
  c.ax = T(alpha * (hx / hy - 2.0 * hy / hx) / 3.0);
  c.ay = T(alpha * (hy / hx - 2.0 * hx / hy) / 3.0);
  c.ad = T(-alpha * (hx / hy + hy / hx) / 6.0);
  return c;
}

// A x at node (i,j) without the diagonal term
template <typename T>
MXH_DEV C<T> node_offdiag(const Geo<T>& g, const C<T>* x, int i, int j, const NodeCoef<T>& c)
{
  return c.ax * (g.at(x, i - 1, j) + g.at(x, i + 1, j)) + c.ay * (g.at(x, i, j - 1) + g.at(x, i, j + 1)) +
         c.ad * (g.at(x, i - 1, j - 1) + g.at(x, i + 1, j - 1) + g.at(x, i - 1, j + 1) + g.at(x, i + 1, j + 1));
}

template <typename T>
__global__ __launch_bounds__(256) void k_node_addeval(mxh_level lv, mxh_bloch bl, const C<T>* X, long long xs,
                                                      C<T>* Y, long long ys, double ar, double ai,
                                                      int accumulate)
{
  const int v = blockIdx.y;
  const size_t N = (size_t)lv.nx * lv.ny;
  size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= N) return;
  const int i = (int)(idx % lv.nx), j = (int)(idx / lv.nx);
  Geo<T> g = make_geo<T>(lv, bl, v);
  NodeCoef<T> c = node_coef<T>(lv, 1.0);
  const C<T>* x = X + (size_t)v * xs;
  C<T> a = c.ac * x[idx] + node_offdiag(g, x, i, j, c);
  C<T> al = cmk(T(ar), T(ai));
  C<T>* y = Y + (size_t)v * ys;
  if (accumulate) y[idx] += al * a;
  else y[idx] = al * a;
}

template <typename T>
__global__ __launch_bounds__(256) void k_node_gs_phase(mxh_level lv, mxh_bloch bl, const C<T>* B, long long bs,
                                                       C<T>* X, long long xs, double alpha, int ci, int cj)
{
  const int v = blockIdx.y;
  const int hx2 = lv.nx >> 1;
  const size_t np = (size_t)hx2 * (lv.ny >> 1);
  size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  const int i = 2 * (int)(p % hx2) + ci, j = 2 * (int)(p / hx2) + cj;
  Geo<T> g = make_geo<T>(lv, bl, v);
  NodeCoef<T> c = node_coef<T>(lv, alpha);
  C<T>* x = X + (size_t)v * xs;
  const C<T>* b = B + (size_t)v * bs;
  const size_t k = i + (size_t)j * lv.nx;
  x[k] = (T(1) / c.ac) * (b[k] - node_offdiag(g, (const C<T>*)x, i, j, c));
}

template <typename T>
__global__ __launch_bounds__(256) void k_node_resid_restrict(mxh_level lf, mxh_bloch bl, const C<T>* BF,
                                                             long long bfs, const C<T>* XF, long long xfs,
                                                             C<T>* BC, long long bcs, C<T>* XC, long long xcs)
{
  const int v = blockIdx.y;
  const int cnx = lf.nx >> 1, cny = lf.ny >> 1;
  const size_t NC = (size_t)cnx * cny;
  size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= NC) return;
  const int I = (int)(idx % cnx), J = (int)(idx / cnx);
  Geo<T> g = make_geo<T>(lf, bl, v);
  NodeCoef<T> c = node_coef<T>(lf, 1.0);
  const C<T>* b = BF + (size_t)v * bfs;
  const C<T>* x = XF + (size_t)v * xfs;
  C<T> s = czero<T>();
  for (int dj = -1; dj <= 1; dj++)
    for (int di = -1; di <= 1; di++) {
      const int i = 2 * I + di, j = 2 * J + dj;
      const T w = T((di == 0 ? 1.0 : 0.5) * (dj == 0 ? 1.0 : 0.5));
      C<T> r = g.at(b, i, j) - c.ac * g.at(x, i, j) - node_offdiag(g, x, i, j, c);
      s += w * r;
    }
  BC[(size_t)v * bcs + idx] = s;
  XC[(size_t)v * xcs + idx] = czero<T>();
}

template <typename T>
__global__ __launch_bounds__(256) void k_node_prolong(mxh_level lf, mxh_bloch bl, const C<T>* CV, long long cs,
                                                      C<T>* FV, long long fs, double ar, double ai)
{
  const int v = blockIdx.y;
  const int cnx = lf.nx >> 1, cny = lf.ny >> 1;
  const size_t NC = (size_t)cnx * cny;
  size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= NC) return;
  const int I = (int)(idx % cnx), J = (int)(idx / cnx);
  Geo<T> gc = make_geo<T>(lf, bl, v);
  gc.nx = cnx;
  gc.ny = cny;
  const C<T>* c = CV + (size_t)v * cs;
  C<T>* f = FV + (size_t)v * fs;
  const C<T> al = cmk(T(ar), T(ai));
  C<T> c00 = c[idx], c10 = gc.at(c, I + 1, J), c01 = gc.at(c, I, J + 1), c11 = gc.at(c, I + 1, J + 1);
  const size_t r0 = (size_t)(2 * J) * lf.nx + 2 * I, r1 = r0 + lf.nx;
  f[r0] += al * c00;
  f[r0 + 1] += al * (T(0.5) * (c00 + c10));
  f[r1] += al * (T(0.5) * (c00 + c01));
  f[r1 + 1] += al * (T(0.25) * (c00 + c10 + c01 + c11));
}

template <typename T>
__global__ __launch_bounds__(256) void k_node_restrict(mxh_level lf, mxh_bloch bl, const C<T>* FV, long long fs,
                                                       C<T>* CV, long long cs, double ar, double ai)
{
  const int v = blockIdx.y;
  const int cnx = lf.nx >> 1, cny = lf.ny >> 1;
  const size_t NC = (size_t)cnx * cny;
  size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= NC) return;
  const int I = (int)(idx % cnx), J = (int)(idx / cnx);
  Geo<T> g = make_geo<T>(lf, bl, v);
  const C<T>* f = FV + (size_t)v * fs;
  C<T> s = czero<T>();
  for (int dj = -1; dj <= 1; dj++)
    for (int di = -1; di <= 1; di++) {
      const T w = T((di == 0 ? 1.0 : 0.5) * (dj == 0 ? 1.0 : 0.5));
      s += w * g.at(f, 2 * I + di, 2 * J + dj);
    }
  CV[(size_t)v * cs + idx] += cmk(T(ar), T(ai)) * s;
}

// ----------------------------------------------------------------- gradient lifting
// Lowest Bloch plane wave of the node space, phi(i,j) = exp(i (tx i + ty j)),
// tx = arg(xf) / nx: an exact eigenvector of the constant-coefficient Q1
// Laplacian.  Its eigenvalue mu ~ (k / n)^2 is below FP32 resolution near the
// Gamma point, so the FP32 node solve handles it separately (see k_lift_rhs).
// The kernels below walk rows (block-uniform j) with thread columns
// i = tid, tid + blockDim, ...: phi = row(j) col(i), col advanced by a fixed
// complex step, so a thread evaluates one sincos per row and one per column
// start.
struct PlaneWave {
  double tx, ty;
  C<double> c0, step;  // col(tid), exp(i tx blockDim)
  MXH_DEV PlaneWave(const Geo<double>& g)
  {
    tx = atan2(g.xf.i, g.xf.r) / g.nx;
    ty = atan2(g.yf.i, g.yf.r) / g.ny;
    double s, c;
    sincos(tx * (double)threadIdx.x, &s, &c);
    c0 = cmk(c, s);
    sincos(tx * (double)blockDim.x, &s, &c);
    step = cmk(c, s);
  }
  MXH_DEV C<double> row(int j) const
  {
    double s, c;
    sincos(ty * (double)j, &s, &c);
    return cmk(c, s);
  }
  MXH_DEV C<double> col(int i) const
  {
    double s, c;
    sincos(tx * (double)i, &s, &c);
    return cmk(c, s);
  }
};

// u = e - x (u, e FP64; x of precision T, optional); bg (T) = G^H M u; xg = 0
// (xg optional).
// u must not alias e when x is given: threads read e at neighbouring nodes.
// With phi non-null, per-block partial sums of conj(phi) . (G^H M u) (FP64)
// go to phi (2 doubles per vector and block).
template <typename T>
MXH_DEV C<double> lift_point(const Geo<double>& g, const Geo<T>& gt, const C<double>* ex, const C<double>* ey,
                             const C<T>* xx, const C<T>* xy, int i, int j, double mx, double my, C<double>* u,
                             size_t N)
{
  // u at the 12 edges needed: x(i-1, j-1..j+1), x(i, j-1..j+1),
  // y(i-1..i+1, j-1), y(i-1..i+1, j)
  C<double> X[2][3], Y[3][2];
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int b = 0; b < 3; b++) X[a][b] = g.at(ex, i - 1 + a, j - 1 + b);
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 2; b++) Y[a][b] = g.at(ey, i - 1 + a, j - 1 + b);
  if (xx) {
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
      for (int b = 0; b < 3; b++) X[a][b] -= ccast<double>(gt.at(xx, i - 1 + a, j - 1 + b));
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int b = 0; b < 2; b++) Y[a][b] -= ccast<double>(gt.at(xy, i - 1 + a, j - 1 + b));
  }
  const C<double> mxl = mx * (4.0 * X[0][1] + X[0][0] + X[0][2]);  // (M u) at x(i-1, j)
  const C<double> mxr = mx * (4.0 * X[1][1] + X[1][0] + X[1][2]);  // x(i, j)
  const C<double> myb = my * (4.0 * Y[1][0] + Y[0][0] + Y[2][0]);  // y(i, j-1)
  const C<double> myt = my * (4.0 * Y[1][1] + Y[0][1] + Y[2][1]);  // y(i, j)
  if (u) {
    const size_t k = i + (size_t)j * g.nx;
    u[k] = X[1][1];
    u[N + k] = Y[1][1];
  }
  // G^H: node += incoming - outgoing edges (node2d.c:1312-1350)
  return mxl - mxr + myb - myt;
}

template <typename T, bool FRAME>
__global__ __launch_bounds__(256) void k_lift_rhs(mxh_level lv, mxh_bloch bl, const C<double>* E, long long es,
                                                  const int* emap, const C<T>* XV, long long xs, C<double>* U,
                                                  long long us, const int* umap, C<T>* BG, long long bgs, C<T>* XG,
                                                  long long xgs, double* phi, int slot0)
{
  __shared__ double sh[4];
  const int v = blockIdx.y;
  const int nx = lv.nx, ny = lv.ny;
  const size_t N = (size_t)nx * ny;
  const Geo<double> g = make_geo<double>(lv, bl, v);
  const Geo<T> gt = make_geo<T>(lv, bl, v);
  const C<double>* ex = E + (size_t)(emap ? emap[v] : v) * es;
  const C<double>* ey = ex + N;
  const C<T>* xx = XV ? XV + (size_t)v * xs : nullptr;
  const C<T>* xy = XV ? xx + N : nullptr;
  C<double>* u = U ? U + (size_t)(umap ? umap[v] : v) * us : nullptr;
  C<T>* bg = BG + (size_t)v * bgs;
  C<T>* xg = XG ? XG + (size_t)v * xgs : nullptr;
  const double mx = lv.hy / lv.hx / 6.0, my = lv.hx / lv.hy / 6.0;
  double pr = 0.0, pi = 0.0;
  PlaneWave pw(g);
  if (FRAME) {
    const int nf = (int)frame_points(nx, ny);
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < nf; k += gridDim.x * blockDim.x) {
      int i, j;
      frame_point(k, nx, ny, i, j);
      const C<double> d = lift_point<T>(g, gt, ex, ey, xx, xy, i, j, mx, my, u, N);
      const size_t q = i + (size_t)j * nx;
      bg[q] = ccast<T>(d);
      if (xg) xg[q] = czero<T>();
      if (phi) {
        const C<double> ph = pw.row(j) * pw.col(i);
        pr += ph.r * d.r + ph.i * d.i;  // conj(phi) d
        pi += ph.r * d.i - ph.i * d.r;
      }
    }
  } else {
    // each thread walks its columns down a band of rows and keeps the values
    // of u = e - x that the next row's stencil shares with this one (five
    // new values of each of e and x per point instead of twelve)
    const int j0 = max(1, row_first(ny)), j1 = min(ny - 1, row_end(ny));
    auto ux = [&](size_t q) {
      C<double> w = ex[q];
      if (xx) w -= ccast<double>(xx[q]);
      return w;
    };
    auto uy = [&](size_t q) {
      C<double> w = ey[q];
      if (xy) w -= ccast<double>(xy[q]);
      return w;
    };
    const C<double> rstep = phi ? pw.row(1) : czero<double>();
    if (j0 < j1)
      for (int i = 1 + (int)threadIdx.x; i < nx - 1; i += blockDim.x) {
        size_t k = i + (size_t)j0 * nx;
        // Xab = u_x(i - 1 + a, j - 1 + b), Yab = u_y(i - 1 + a, j - 1 + b)
        C<double> X00 = ux(k - nx - 1), X01 = ux(k - 1), X10 = ux(k - nx), X11 = ux(k);
        C<double> Y00 = uy(k - nx - 1), Y10 = uy(k - nx), Y20 = uy(k - nx + 1);
        C<double> rowf = phi ? pw.row(j0) : czero<double>();
        const C<double> cfi = phi ? pw.col(i) : czero<double>();
        for (int j = j0; j < j1; j++, k += nx) {
          const C<double> X02 = ux(k + nx - 1), X12 = ux(k + nx);
          const C<double> Y01 = uy(k - 1), Y11 = uy(k), Y21 = uy(k + 1);
          const C<double> mxl = mx * (4.0 * X01 + X00 + X02);  // (M u) at x(i-1, j)
          const C<double> mxr = mx * (4.0 * X11 + X10 + X12);  // x(i, j)
          const C<double> myb = my * (4.0 * Y10 + Y00 + Y20);  // y(i, j-1)
          const C<double> myt = my * (4.0 * Y11 + Y01 + Y21);  // y(i, j)
          if (u) {
            u[k] = X11;
            u[N + k] = Y11;
          }
          // G^H: node += incoming - outgoing edges (node2d.c:1312-1350)
          const C<double> d = mxl - mxr + myb - myt;
          bg[k] = ccast<T>(d);
          if (xg) xg[k] = czero<T>();
          if (phi) {
            const C<double> ph = rowf * cfi;
            pr += ph.r * d.r + ph.i * d.i;  // conj(phi) d
            pi += ph.r * d.i - ph.i * d.r;
            rowf = rowf * rstep;
          }
          X00 = X01;
          X01 = X02;
          X10 = X11;
          X11 = X12;
          Y00 = Y01;
          Y10 = Y11;
          Y20 = Y21;
        }
      }
  }
  if (phi) {
    double a = block_sum256(pr, sh);
    double b = block_sum256(pi, sh);
    if (threadIdx.x == 0) {
      size_t w = (size_t)(slot0 + blockIdx.x) * (2 * gridDim.y) + 2 * v;
      phi[w] = a;
      phi[w + 1] = b;
    }
  }
}

// Laplacian eigenvalue of the plane wave: ac + 2 ax cos tx + 2 ay cos ty +
// 4 ad cos tx cos ty, written with s = 1 - cos = 2 sin^2(t/2) (no cancellation)
MXH_DEV double plane_wave_mu(const mxh_level& lv, double tx, double ty)
{
  const NodeCoef<double> nc = node_coef<double>(lv, 1.0);
  const double sx = 2.0 * sin(0.5 * tx) * sin(0.5 * tx), sy = 2.0 * sin(0.5 * ty) * sin(0.5 * ty);
  return -2.0 * nc.ax * sx - 2.0 * nc.ay * sy - 4.0 * nc.ad * (sx + sy) + 4.0 * nc.ad * sx * sy;
}

// bg -= (c / N) phi with c = phi^H d from k_lift_rhs; coef[v] = c / (N mu)
// (zero at the Gamma point, where the coarse node matrix carries the
// regularisation of the constant mode instead).
template <typename T>
__global__ __launch_bounds__(256) void k_lift_deflate(mxh_level lv, mxh_bloch bl, C<T>* BG, long long bgs,
                                                      const double* csum, double* coef)
{
  const int v = blockIdx.y;
  const int nx = lv.nx, ny = lv.ny;
  const size_t N = (size_t)nx * ny;
  const Geo<double> g = make_geo<double>(lv, bl, v);
  const double cr = csum[2 * v] / N, ci = csum[2 * v + 1] / N;
  const bool gamma = g.xf.r == 1.0 && g.xf.i == 0.0 && g.yf.r == 1.0 && g.yf.i == 0.0;
  PlaneWave pw(g);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    const double mu = plane_wave_mu(lv, pw.tx, pw.ty);
    coef[2 * v] = gamma ? 0.0 : cr / mu;
    coef[2 * v + 1] = gamma ? 0.0 : ci / mu;
  }
  if (gamma) return;
  C<T>* bg = BG + (size_t)v * bgs;
  const C<double> cc = cmk(cr, ci);
  for (int j = row_first(ny), je = row_end(ny); j < je; j++) {
    const C<double> rowf = cc * pw.row(j);
    C<double> cf = pw.c0;
    for (int i = threadIdx.x; i < nx; i += blockDim.x) {
      const size_t k = i + (size_t)j * nx;
      bg[k] = ccast<T>(ccast<double>(bg[k]) - rowf * cf);
      cf = cf * pw.step;
    }
  }
}

// Per-block partial sums of phi^H xg (FP64; 2 doubles per vector and block).
template <typename T>
__global__ __launch_bounds__(256) void k_phi_dot(mxh_level lv, mxh_bloch bl, const C<T>* XG, long long xgs,
                                                 double* part)
{
  __shared__ double sh[4];
  const int v = blockIdx.y;
  const int nx = lv.nx, ny = lv.ny;
  const Geo<double> g = make_geo<double>(lv, bl, v);
  const C<T>* xg = XG + (size_t)v * xgs;
  PlaneWave pw(g);
  double pr = 0.0, pi = 0.0;
  for (int j = row_first(ny), je = row_end(ny); j < je; j++) {
    const C<double> rowf = pw.row(j);
    C<double> cf = pw.c0;
    for (int i = threadIdx.x; i < nx; i += blockDim.x) {
      const C<double> ph = rowf * cf, d = ccast<double>(xg[i + (size_t)j * nx]);
      pr += ph.r * d.r + ph.i * d.i;
      pi += ph.r * d.i - ph.i * d.r;
      cf = cf * pw.step;
    }
  }
  double a = block_sum256(pr, sh);
  double b = block_sum256(pi, sh);
  if (threadIdx.x == 0) {
    size_t w = (size_t)blockIdx.x * (2 * gridDim.y) + 2 * v;
    part[w] = a;
    part[w + 1] = b;
  }
}

// e (FP64) = u - x + alpha G (xg + a_v phi) with a_v = coef_v - phi^H xg / N
// (x of precision T, optional; u may be e itself: each thread reads and
// writes only its own edges): the plane-wave component of the node correction is replaced by the exact one
// (coef from k_lift_deflate; xg has none in exact arithmetic since its right
// hand side was deflated, so what phi^H xg finds is rounding).  pdot null: xg
// holds no plane wave (the direct solve leaves its mode out).
template <typename T>
__global__ __launch_bounds__(256) void k_lift_apply(mxh_level lv, mxh_bloch bl, const C<T>* XG, long long xgs,
                                                    const C<double>* U, long long us, const int* umap,
                                                    const C<T>* XV, long long xs, C<double>* E, long long es,
                                                    const int* emap, double alpha, const double* coef,
                                                    const double* pdot)
{
  const int v = blockIdx.y;
  const int nx = lv.nx, ny = lv.ny;
  const size_t N = (size_t)nx * ny;
  const Geo<T> gt = make_geo<T>(lv, bl, v);
  const C<T>* xg = XG + (size_t)v * xgs;
  const C<double>* u = U ? U + (size_t)(umap ? umap[v] : v) * us : nullptr;  // null: u = 0
  const C<T>* xv = XV ? XV + (size_t)v * xs : nullptr;
  C<double>* e = E + (size_t)(emap ? emap[v] : v) * es;
  const Geo<double> g = make_geo<double>(lv, bl, v);
  PlaneWave pw(g);
  C<double> a = czero<double>(), ex1 = czero<double>(), ey1 = czero<double>();
  if (coef) {
    a = cmk(coef[2 * v], coef[2 * v + 1]);
    if (pdot) a -= cmk(pdot[2 * v] / N, pdot[2 * v + 1] / N);
    double s, c;
    sincos(pw.tx, &s, &c);
    ex1 = cmk(c - 1.0, s);  // phi(i+1,j) / phi(i,j) - 1
    sincos(pw.ty, &s, &c);
    ey1 = cmk(c - 1.0, s);
  }
  for (int j = row_first(ny), je = row_end(ny); j < je; j++) {
    const bool jin = j <= ny - 2;
    const C<double> rowf = coef ? a * pw.row(j) : czero<double>();
    C<double> cf = pw.c0;
    for (int i = threadIdx.x; i < nx; i += blockDim.x) {
      const size_t k = i + (size_t)j * nx;
      const C<double> x0 = ccast<double>(xg[k]);
      C<double> gx, gy;
      if (jin && i <= nx - 2) {
        gx = ccast<double>(xg[k + 1]) - x0;
        gy = ccast<double>(xg[k + nx]) - x0;
      } else {
        gx = ccast<double>(gt.at(xg, i + 1, j)) - x0;
        gy = ccast<double>(gt.at(xg, i, j + 1)) - x0;
      }
      if (coef) {
        const C<double> ph = rowf * cf;
        gx += ph * ex1;
        gy += ph * ey1;
        cf = cf * pw.step;
      }
      C<double> u0 = u ? u[k] : czero<double>(), u1 = u ? u[N + k] : czero<double>();
      if (xv) {
        u0 -= ccast<double>(xv[k]);
        u1 -= ccast<double>(xv[N + k]);
      }
      e[k] = u0 + alpha * gx;
      e[N + k] = u1 + alpha * gy;
    }
  }
}

// ----------------------------------------------------------------- direct node solve
// The node operator of the lifting (the Q1 Laplacian on a uniform periodic
// grid) has constant coefficients, so with the Bloch phase taken out
// (g(i,j) = e^{-i(tx i + ty j)} b(i,j)) it is diagonal in the discrete Fourier
// basis, with eigenvalue
//   mu(p,q) = rx S(thx) T(thy) + ry T(thx) S(thy),  S = 2s, T = 1 - s / 3,
//   s = 1 - cos th = 2 sin^2(th / 2),  thx = (2 pi p + kx) / nx.
// One transform pair replaces the node V-cycles of the lifting: three read +
// write passes over the node vectors (one where a vector fits in LDS) against
// the forty-odd of five V(2,2) cycles.  Measured over the liftings of the
// 512^2 64-k mixed solve: row passes 3.1 TB/s, column pass 1.7 TB/s (its 128
// byte row segments and six LDS stages), 53 ms where the cycles took 363.
//
// The forward transform decimates in frequency in place, so mode p ends at
// the digit-reversed place; the eigenvalue is looked up by place and the
// inverse (decimation in time, the same stages backwards) restores the order:
// nothing is ever permuted.  Lines (rows or columns) of a workgroup sit in
// LDS; consecutive lanes take consecutive lines, which an odd row pitch keeps
// on different banks at every stage.
#define FFT_MAXS 12
struct FftPlan {
  int n, ns;          // length and number of stages
  int r[FFT_MAXS];    // radix of each stage: 3 or 5 (if any) first, then 8, 4, 2
  int lm[FFT_MAXS];   // log2 of the stage's span (a power of two)
};

// multiply by -i (DIR < 0) or i (DIR > 0)
template <int DIR, typename T> MXH_DEV C<T> mul_i(C<T> a)
{
  return DIR < 0 ? cmk(a.i, -a.r) : cmk(-a.i, a.r);
}

template <int R, int DIR, typename T> struct Dft;
template <int DIR, typename T> struct Dft<2, DIR, T> {
  static MXH_DEV void run(C<T>* a)
  {
    const C<T> t = a[0] - a[1];
    a[0] = a[0] + a[1];
    a[1] = t;
  }
};
template <int DIR, typename T> struct Dft<4, DIR, T> {
  static MXH_DEV void run(C<T>* a)
  {
    const C<T> s0 = a[0] + a[2], d0 = a[0] - a[2], s1 = a[1] + a[3], d1 = mul_i<DIR>(a[1] - a[3]);
    a[0] = s0 + s1;
    a[1] = d0 + d1;
    a[2] = s0 - s1;
    a[3] = d0 - d1;
  }
};
template <int DIR, typename T> struct Dft<8, DIR, T> {
  static MXH_DEV void run(C<T>* a)
  {
    C<T> e[4] = {a[0], a[2], a[4], a[6]}, o[4] = {a[1], a[3], a[5], a[7]};
    Dft<4, DIR, T>::run(e);
    Dft<4, DIR, T>::run(o);
    const T h = T(0.70710678118654752440);
    const C<T> i1 = mul_i<DIR>(o[1]), i3 = mul_i<DIR>(o[3]);
    o[1] = h * (o[1] + i1);  // e^{DIR i pi / 4}
    o[2] = mul_i<DIR>(o[2]);
    o[3] = h * (i3 - o[3]);  // e^{DIR 3 i pi / 4}
#pragma unroll
    for (int k = 0; k < 4; k++) {
      a[k] = e[k] + o[k];
      a[k + 4] = e[k] - o[k];
    }
  }
};
template <int DIR, typename T> struct Dft<3, DIR, T> {
  static MXH_DEV void run(C<T>* a)
  {
    const C<T> s = a[1] + a[2], d = mul_i<DIR>(a[1] - a[2]);
    const C<T> m = a[0] - T(0.5) * s, w = T(0.86602540378443864676) * d;
    a[0] = a[0] + s;
    a[1] = m + w;
    a[2] = m - w;
  }
};
template <int DIR, typename T> struct Dft<5, DIR, T> {
  static MXH_DEV void run(C<T>* a)
  {
    // cos and sin of 2 pi / 5 and 4 pi / 5
    const T c1 = T(0.30901699437494742410), c2 = T(-0.80901699437494742410);
    const T s1 = T(0.95105651629515357212), s2 = T(0.58778525229247312917);
    const C<T> p1 = a[1] + a[4], m1 = mul_i<DIR>(a[1] - a[4]), p2 = a[2] + a[3], m2 = mul_i<DIR>(a[2] - a[3]);
    const C<T> u1 = a[0] + c1 * p1 + c2 * p2, u2 = a[0] + c2 * p1 + c1 * p2;
    const C<T> v1 = s1 * m1 + s2 * m2, v2 = s2 * m1 - s1 * m2;
    a[0] = a[0] + p1 + p2;
    a[1] = u1 + v1;
    a[2] = u2 + v2;
    a[3] = u2 - v2;
    a[4] = u1 - v1;
  }
};

// frequency of the value at place pos after the forward stages
MXH_DEV int fft_freq(const FftPlan& pl, int pos)
{
  int f = 0, mul = 1;
  for (int s = 0; s < pl.ns; s++) {
    f += (pos >> pl.lm[s]) * mul;
    pos &= (1 << pl.lm[s]) - 1;
    mul *= pl.r[s];
  }
  return f;
}

// One stage over nl lines in LDS (value k of line l at d[l ls + k ps]): a
// thread takes line l0 + multiples of lstep and butterflies q0 + multiples of
// qstep.  Forward (DIR < 0): transform, then the twiddles; inverse: the
// conjugate twiddles, then the transform.  LAST (span 1, no twiddles): with
// SCALE, forward and inverse butterfly in one go with the factor fac(line,
// place) between them.
template <int R, int DIR, bool SCALE, typename T, typename F>
MXH_DEV void fft_stage(C<T>* d, int nl, int ls, int ps, int n, int lm, const C<T>* tw, int l0, int lstep,
                       int q0, int qstep, F fac)
{
  const int m = 1 << lm, nq = n / R, tstep = nq >> lm;  // tstep = n / (R m)
  for (int l = l0; l < nl; l += lstep)
    for (int q = q0; q < nq; q += qstep) {
      const int pos = q & (m - 1), base = ((q >> lm) << lm) * R + pos;
      C<T>* p = d + l * ls + base * ps;
      C<T> a[R];
#pragma unroll
      for (int k = 0; k < R; k++) a[k] = p[(k << lm) * ps];
      if (SCALE) {
        Dft<R, -1, T>::run(a);
#pragma unroll
        for (int k = 0; k < R; k++) a[k] = fac(l, base + k) * a[k];  // span 1: place base + k
        Dft<R, 1, T>::run(a);
      } else {
        if (DIR > 0 && lm > 0) {
#pragma unroll
          for (int k = 1; k < R; k++) a[k] = cconj(tw[k * pos * tstep]) * a[k];
        }
        Dft<R, DIR, T>::run(a);
        if (DIR < 0 && lm > 0) {
#pragma unroll
          for (int k = 1; k < R; k++) a[k] = tw[k * pos * tstep] * a[k];
        }
      }
#pragma unroll
      for (int k = 0; k < R; k++) p[(k << lm) * ps] = a[k];
    }
}

template <int DIR, bool SCALE, typename T, typename F>
MXH_DEV void fft_any_stage(const FftPlan& pl, int s, C<T>* d, int nl, int ls, int ps, const C<T>* tw, int l0,
                           int lstep, int q0, int qstep, F fac)
{
  switch (pl.r[s]) {  // uniform
  case 8: fft_stage<8, DIR, SCALE>(d, nl, ls, ps, pl.n, pl.lm[s], tw, l0, lstep, q0, qstep, fac); break;
  case 4: fft_stage<4, DIR, SCALE>(d, nl, ls, ps, pl.n, pl.lm[s], tw, l0, lstep, q0, qstep, fac); break;
  case 2: fft_stage<2, DIR, SCALE>(d, nl, ls, ps, pl.n, pl.lm[s], tw, l0, lstep, q0, qstep, fac); break;
  case 3: fft_stage<3, DIR, SCALE>(d, nl, ls, ps, pl.n, pl.lm[s], tw, l0, lstep, q0, qstep, fac); break;
  case 5: fft_stage<5, DIR, SCALE>(d, nl, ls, ps, pl.n, pl.lm[s], tw, l0, lstep, q0, qstep, fac); break;
  }
  __syncthreads();
}

// all stages of one direction over the lines of a workgroup
template <int DIR, typename T>
MXH_DEV void fft_lines(const FftPlan& pl, C<T>* d, int nl, int ls, int ps, const C<T>* tw, int l0, int lstep, int q0,
                       int qstep)
{
  auto one = [](int, int) { return T(1); };
  for (int t = 0; t < pl.ns; t++)
    fft_any_stage<DIR, false>(pl, DIR < 0 ? t : pl.ns - 1 - t, d, nl, ls, ps, tw, l0, lstep, q0, qstep, one);
}

// the column transforms with the division by nx ny mu between them: the last
// forward and the first inverse stage are one
template <typename T, typename F>
MXH_DEV void fft_solve_lines(const FftPlan& pl, C<T>* d, int nl, int ls, int ps, const C<T>* tw, int l0, int lstep,
                             int q0, int qstep, F fac)
{
  auto one = [](int, int) { return T(1); };
  for (int t = 0; t + 1 < pl.ns; t++)
    fft_any_stage<-1, false>(pl, t, d, nl, ls, ps, tw, l0, lstep, q0, qstep, one);
  fft_any_stage<-1, true>(pl, pl.ns - 1, d, nl, ls, ps, tw, l0, lstep, q0, qstep, fac);
  for (int t = pl.ns - 2; t >= 0; t--)
    fft_any_stage<1, false>(pl, t, d, nl, ls, ps, tw, l0, lstep, q0, qstep, one);
}

// s = 1 - cos th of the mode at place pos of a line of length n with Bloch
// angle k: th in [-pi, pi], so small angles keep their relative accuracy
MXH_DEV double mode_s(const FftPlan& pl, int pos, double k)
{
  int f = fft_freq(pl, pos);
  if (2 * f > pl.n) f -= pl.n;
  const double h = sin(0.5 * (6.283185307179586476925 * f + k) / pl.n);
  return 2.0 * h * h;
}

// 1 / (nx ny mu); the lowest wave (place 0, 0) is left out: its coefficient
// is formed in FP64 by the lifting (k_lift_coef)
template <typename T>
MXH_DEV T mode_factor(T sx, T sy, T rx, T ry, T cnt, bool lowest)
{
  const T mu = rx * (T(2) * sx) * (T(1) - sy / T(3)) + ry * (T(2) * sy) * (T(1) - sx / T(3));
  return lowest ? T(0) : T(1) / (cnt * mu);
}

// Row transforms of RB rows per workgroup.  Forward: the Bloch phase is taken
// out at load; inverse: put back at the store.
template <typename T, int DIR>
__global__ __launch_bounds__(256) void k_fft_rows(mxh_level lv, mxh_bloch bl, FftPlan pl, const C<T>* tw,
                                                  const C<T>* IN, long long is, C<T>* OUT, long long os, int RB)
{
  extern __shared__ double smem[];
  const int nx = lv.nx, ny = lv.ny, pitch = nx | 1, tid = threadIdx.x, bd = blockDim.x;
  C<T>* d = (C<T>*)smem;                   // [RB][pitch]
  C<T>* colf = d + (size_t)RB * pitch;     // [nx]: e^{-DIR' i tx i}
  C<T>* rowf = colf + nx;                  // [RB]
  const int v = blockIdx.y, j0 = blockIdx.x * RB, nr = min(RB, ny - j0);
  const Geo<double> g = make_geo<double>(lv, bl, v);
  const double tx = atan2(g.xf.i, g.xf.r) / nx, ty = atan2(g.yf.i, g.yf.r) / ny;
  for (int w = tid; w < nx + nr; w += bd) {
    double s, c;
    sincos(DIR * (w < nx ? tx * w : ty * (j0 + w - nx)), &s, &c);
    colf[w] = cmk(T(c), T(s));  // rowf follows colf
  }
  __syncthreads();
  const C<T>* in = IN + (size_t)v * is + (size_t)j0 * nx;
  C<T>* out = OUT + (size_t)v * os + (size_t)j0 * nx;
  const int tot = nr * nx, dr = bd / nx, di = bd - dr * nx;
  for (int w = tid, r = tid / nx, i = tid - r * nx; w < tot; w += bd) {
    d[r * pitch + i] = DIR < 0 ? (colf[i] * rowf[r]) * in[w] : in[w];
    r += dr;
    i += di;
    if (i >= nx) { i -= nx; r++; }
  }
  __syncthreads();
  fft_lines<DIR>(pl, d, nr, pitch, 1, tw, tid & (RB - 1), RB, tid / RB, bd / RB);
  for (int w = tid, r = tid / nx, i = tid - r * nx; w < tot; w += bd) {
    out[w] = DIR > 0 ? (colf[i] * rowf[r]) * d[r * pitch + i] : d[r * pitch + i];
    r += dr;
    i += di;
    if (i >= nx) { i -= nx; r++; }
  }
}

// Column transforms, division by the eigenvalues and back, in place: CB
// columns (128-byte row segments) of one vector per workgroup.
template <typename T>
__global__ __launch_bounds__(1024) void k_fft_cols(mxh_level lv, mxh_bloch bl, FftPlan px, FftPlan py, const C<T>* tw,
                                                   C<T>* X, long long xs, int CB)
{
  extern __shared__ double smem[];
  const int nx = lv.nx, ny = lv.ny, tid = threadIdx.x, bd = blockDim.x;
  C<T>* d = (C<T>*)smem;            // [ny][CB]
  T* sy = (T*)(d + (size_t)ny * CB);
  T* sx = sy + ny;
  const int v = blockIdx.y, c0 = blockIdx.x * CB, nc = min(CB, nx - c0);
  const Geo<double> g = make_geo<double>(lv, bl, v);
  const double kx = atan2(g.xf.i, g.xf.r), ky = atan2(g.yf.i, g.yf.r);
  C<T>* x = X + (size_t)v * xs + c0;
  const int l = tid & (CB - 1), q0 = tid / CB, qstep = bd / CB;
  if (l < nc)
    for (int j = q0; j < ny; j += qstep) d[j * CB + l] = x[l + (size_t)j * nx];
  for (int w = tid; w < ny + nc; w += bd) {
    if (w < ny) sy[w] = T(mode_s(py, w, ky));
    else sx[w - ny] = T(mode_s(px, c0 + w - ny, kx));
  }
  __syncthreads();
  const T rx = T(lv.hy / lv.hx), ry = T(lv.hx / lv.hy), cnt = T((double)nx * ny);
  auto fac = [&](int li, int pos) { return mode_factor(sx[li], sy[pos], rx, ry, cnt, c0 + li == 0 && pos == 0); };
  fft_solve_lines(py, d, nc, 1, CB, tw, l, CB, q0, qstep, fac);
  if (l < nc)
    for (int j = q0; j < ny; j += qstep) x[l + (size_t)j * nx] = d[j * CB + l];
}

// The whole solve of one vector in LDS (small grids): one launch, one read
// and one write.
template <typename T>
__global__ __launch_bounds__(1024) void k_fft_solve(mxh_level lv, mxh_bloch bl, FftPlan px, FftPlan py,
                                                    const C<T>* twx, const C<T>* twy, const C<T>* IN, long long is,
                                                    C<T>* OUT, long long os)
{
  extern __shared__ double smem[];
  const int nx = lv.nx, ny = lv.ny, pitch = nx | 1, tid = threadIdx.x, bd = blockDim.x, v = blockIdx.x;
  C<T>* d = (C<T>*)smem;                  // [ny][pitch]
  C<T>* colf = d + (size_t)ny * pitch;    // [nx]
  C<T>* rowf = colf + nx;                 // [ny]
  T* sx = (T*)(rowf + ny);                // [nx]
  T* sy = sx + nx;                        // [ny]
  const Geo<double> g = make_geo<double>(lv, bl, v);
  const double kx = atan2(g.xf.i, g.xf.r), ky = atan2(g.yf.i, g.yf.r);
  for (int w = tid; w < nx + ny; w += bd) {
    const bool isx = w < nx;
    const int k = isx ? w : w - nx;
    double s, c;
    sincos((isx ? kx / nx : ky / ny) * k, &s, &c);
    colf[w] = cmk(T(c), T(s));
    sx[w] = T(isx ? mode_s(px, k, kx) : mode_s(py, k, ky));
  }
  __syncthreads();
  const C<T>* in = IN + (size_t)v * is;
  C<T>* out = OUT + (size_t)v * os;
  const int tot = nx * ny, dr = bd / nx, di = bd - dr * nx;
  for (int w = tid, r = tid / nx, i = tid - r * nx; w < tot; w += bd) {
    d[r * pitch + i] = cconj(colf[i] * rowf[r]) * in[w];
    r += dr;
    i += di;
    if (i >= nx) { i -= nx; r++; }
  }
  __syncthreads();
  const int l = tid & 31, q0 = tid >> 5, qstep = bd >> 5;
  const T rx = T(lv.hy / lv.hx), ry = T(lv.hx / lv.hy), cnt = T((double)nx * ny);
  auto fac = [&](int li, int pos) { return mode_factor(sx[li], sy[pos], rx, ry, cnt, li == 0 && pos == 0); };
  fft_lines<-1>(px, d, ny, pitch, 1, twx, l, 32, q0, qstep);
  fft_solve_lines(py, d, nx, 1, pitch, twy, l, 32, q0, qstep, fac);
  fft_lines<1>(px, d, ny, pitch, 1, twx, l, 32, q0, qstep);
  for (int w = tid, r = tid / nx, i = tid - r * nx; w < tot; w += bd) {
    out[w] = (colf[i] * rowf[r]) * d[r * pitch + i];
    r += dr;
    i += di;
    if (i >= nx) { i -= nx; r++; }
  }
}

// e^{-2 pi i k / n}, k < n
template <typename T>
__global__ void k_fft_table(int n, C<T>* tw)
{
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  double s, c;
  sincospi(-2.0 * k / n, &s, &c);
  tw[k] = cmk(T(c), T(s));
}

// coef[v] = (phi^H d / N) / mu of the lowest Bloch wave (zero at the Gamma
// point) from the sums of k_lift_rhs
__global__ void k_lift_coef(mxh_level lv, mxh_bloch bl, int nv, const double* csum, double* coef)
{
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= nv) return;
  const Geo<double> g = make_geo<double>(lv, bl, v);
  const double N = (double)lv.nx * lv.ny;
  const bool gamma = g.xf.r == 1.0 && g.xf.i == 0.0 && g.yf.r == 1.0 && g.yf.i == 0.0;
  const double mu = plane_wave_mu(lv, atan2(g.xf.i, g.xf.r) / lv.nx, atan2(g.yf.i, g.yf.r) / lv.ny);
  coef[2 * v] = gamma ? 0.0 : csum[2 * v] / N / mu;
  coef[2 * v + 1] = gamma ? 0.0 : csum[2 * v + 1] / N / mu;
}

template <typename T>
__global__ __launch_bounds__(256) void k_gradient(mxh_level lv, mxh_bloch bl, const C<T>* VV, long long vs,
                                                  C<T>* EV_, long long es, double ar, double ai)
{
  const int v = blockIdx.y;
  const size_t N = (size_t)lv.nx * lv.ny;
  size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= N) return;
  const int i = (int)(idx % lv.nx), j = (int)(idx / lv.nx);
  Geo<T> g = make_geo<T>(lv, bl, v);
  const C<T>* x = VV + (size_t)v * vs;
  C<T>* e = EV_ + (size_t)v * es;
  const C<T> al = cmk(T(ar), T(ai));
  C<T> x0 = x[idx];
  e[idx] += al * (g.at(x, i + 1, j) - x0);
  e[N + idx] += al * (g.at(x, i, j + 1) - x0);
}

template <typename T>
__global__ __launch_bounds__(256) void k_adjgradient(mxh_level lv, mxh_bloch bl, const C<T>* EV_, long long es,
                                                     C<T>* VV, long long vs, double ar, double ai)
{
  const int v = blockIdx.y;
  const size_t N = (size_t)lv.nx * lv.ny;
  size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= N) return;
  const int i = (int)(idx % lv.nx), j = (int)(idx / lv.nx);
  Geo<T> g = make_geo<T>(lv, bl, v);
  const C<T>* ex = EV_ + (size_t)v * es;
  const C<T>* ey = ex + N;
  C<T> d = g.at(ex, i - 1, j) - ex[idx] + g.at(ey, i, j - 1) - ey[idx];
  VV[(size_t)v * vs + idx] += cmk(T(ar), T(ai)) * d;
}

// ----------------------------------------------------------------- BLAS-1
template <typename T>
__global__ __launch_bounds__(256) void k_scale(long long n, C<T>* X, long long xs, double ar, double ai)
{
  const int v = blockIdx.y;
  size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)n) return;
  C<T>* x = X + (size_t)v * xs;
  x[idx] = cmk(T(ar), T(ai)) * x[idx];
}

template <typename T>
__global__ __launch_bounds__(256) void k_axpy(long long n, const C<T>* X, long long xs, C<T>* Y, long long ys,
                                              double ar, double ai)
{
  const int v = blockIdx.y;
  size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)n) return;
  Y[(size_t)v * ys + idx] += cmk(T(ar), T(ai)) * X[(size_t)v * xs + idx];
}

template <typename T>
__global__ __launch_bounds__(256) void k_dot(long long n, const C<T>* X, long long xs, const C<T>* Y,
                                             long long ys, double* part)
{
  __shared__ double sh[4];
  const int v = blockIdx.y;
  double sr = 0.0, si = 0.0;
  const C<T>* x = X + (size_t)v * xs;
  const C<T>* y = Y + (size_t)v * ys;
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < (size_t)n;
       idx += (size_t)gridDim.x * blockDim.x) {
    C<double> a = ccast<double>(x[idx]), b = ccast<double>(y[idx]);
    sr += a.r * b.r + a.i * b.i;
    si += a.r * b.i - a.i * b.r;
  }
  double a = block_sum256(sr, sh);
  double b = block_sum256(si, sh);
  if (threadIdx.x == 0) {
    size_t w = (size_t)blockIdx.x * (2 * gridDim.y) + 2 * v;
    part[w] = a;
    part[w + 1] = b;
  }
}

// conj(y)^T x (EDGE 0) or y^H (alpha K + beta M) x (EDGE 1) in FP64 in one launch:
// a workgroup's sum, or the last one to finish adds all partial sums in their
// order, written where the host reads it.  What bounds it is the launch and the
// wait of the host: a 32^2 grid's product 28 -> 12 us against operator,
// product, sum and copy.  work: a counter (0 between launches), then the sums.
#define PRODUCT_TB 1024
#define PRODUCT_BLOCKS 256
template <int EDGE>
__global__ __launch_bounds__(PRODUCT_TB) void k_product(mxh_level lv, mxh_bloch bl, long long n, const C<double>* X,
                                                       const C<double>* Y, const double* eta, mxh_coef cf,
                                                       double* work, double* out, double mark)
{
  __shared__ double sh[2 * PRODUCT_TB / 64];
  __shared__ int last;
  const int tid = threadIdx.x, w = tid >> 6, nw = PRODUCT_TB / 64;
  double sr = 0.0, si = 0.0;
  auto add = [&](C<double> a, C<double> b) {
    sr += a.r * b.r + a.i * b.i;
    si += a.r * b.i - a.i * b.r;
  };
  if (EDGE) {
    const size_t N = (size_t)lv.nx * lv.ny;
    const Geo<double> g = make_geo<double>(lv, bl, 0);
    C<double> axy, mx, my, ox, oy;
    coefs<double>(lv, cf, 0, axy, mx, my);
    const EdgeV<double> e = edge_view<double>(X, 0, 0, N);
    for (size_t k = (size_t)blockIdx.x * PRODUCT_TB + tid; k < N; k += (size_t)gridDim.x * PRODUCT_TB) {
      const int j = (int)((unsigned)k / (unsigned)lv.nx);
      apply_at(g, e, eta, (int)k - j * lv.nx, j, axy, mx, my, ox, oy);
      add(Y[k], ox);
      add(Y[N + k], oy);
    }
  } else {
    for (size_t k = (size_t)blockIdx.x * PRODUCT_TB + tid; k < (size_t)n; k += (size_t)gridDim.x * PRODUCT_TB)
      add(Y[k], X[k]);
  }
  auto total = [&]() {  // over the workgroup, in thread 0
    sr = wave_sum(sr);
    si = wave_sum(si);
    if ((tid & 63) == 0) {
      sh[w] = sr;
      sh[nw + w] = si;
    }
    __syncthreads();
    sr = si = 0.0;
    if (tid == 0)
      for (int q = 0; q < nw; q++) {
        sr += sh[q];
        si += sh[nw + q];
      }
  };
  total();
  unsigned* count = (unsigned*)work;
  double* part = work + 8;
  if (gridDim.x > 1) {
    if (tid == 0) {
      part[2 * blockIdx.x] = sr;
      part[2 * blockIdx.x + 1] = si;
      __threadfence();
      last = atomicAdd(count, 1u) == gridDim.x - 1;
    }
    __syncthreads();
    if (!last) return;
    __threadfence();
    sr = si = 0.0;
    for (int q = tid; q < (int)gridDim.x; q += PRODUCT_TB) {
      sr += part[2 * q];
      si += part[2 * q + 1];
    }
    total();
    if (tid == 0) *count = 0;
  }
  if (tid == 0) {
    out[0] = sr;
    out[1] = si;
    __threadfence_system();
    __hip_atomic_store(out + 2, mark, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

template <typename T>
__global__ __launch_bounds__(256) void k_norm(long long n, const C<T>* X, long long xs, int kind, double* part)
{
  __shared__ double sh[4];
  const int v = blockIdx.y;
  double s = 0.0;
  const C<T>* x = X + (size_t)v * xs;
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < (size_t)n;
       idx += (size_t)gridDim.x * blockDim.x) {
    C<double> a = ccast<double>(x[idx]);
    double q = a.r * a.r + a.i * a.i;
    if (kind == 0) s += q;
    else s = fmax(s, sqrt(q));
  }
  double r = kind == 0 ? block_sum256(s, sh) : block_max256(s, sh);
  if (threadIdx.x == 0) part[(size_t)blockIdx.x * gridDim.y + v] = r;
}

// Sums of the x half and of the y half of each vector (per block partials)
template <typename T>
__global__ __launch_bounds__(256) void k_halfsums(long long half, const C<T>* X, long long xs, double* part)
{
  __shared__ double sh[4];
  const int v = blockIdx.y;
  const C<T>* x = X + (size_t)v * xs;
  double a = 0, b = 0, c = 0, d = 0;
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < (size_t)half;
       idx += (size_t)gridDim.x * blockDim.x) {
    C<double> p = ccast<double>(x[idx]), q = ccast<double>(x[half + idx]);
    a += p.r; b += p.i; c += q.r; d += q.i;
  }
  a = block_sum256(a, sh);
  b = block_sum256(b, sh);
  c = block_sum256(c, sh);
  d = block_sum256(d, sh);
  if (threadIdx.x == 0) {
    double* o = part + ((size_t)blockIdx.x * gridDim.y + v) * 4;
    o[0] = a; o[1] = b; o[2] = c; o[3] = d;
  }
}

template <typename T>
__global__ __launch_bounds__(256) void k_center_apply(long long half, C<T>* X, long long xs, const double* sums)
{
  const int v = blockIdx.y;
  size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)half) return;
  const double* s = sums + 4 * v;
  C<T>* x = X + (size_t)v * xs;
  x[idx] -= cmk(T(s[0] / half), T(s[1] / half));
  x[half + idx] -= cmk(T(s[2] / half), T(s[3] / half));
}

template <typename D, typename S>
__global__ __launch_bounds__(256) void k_convert(long long n, C<D>* Dv, long long ds, const C<S>* Sv, long long ss)
{
  const int v = blockIdx.y;
  size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)n) return;
  Dv[(size_t)v * ds + idx] = ccast<D>(Sv[(size_t)v * ss + idx]);
}

MXH_DEV uint64_t splitmix64(uint64_t z)
{
  z += 0x9E3779B97F4A7C15ULL;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
  return z ^ (z >> 31);
}

// Complex Gaussian entries by Box-Muller from a counter-based hash.
template <typename T>
__global__ __launch_bounds__(256) void k_random(long long n, C<T>* X, long long xs, unsigned long long seed,
                                                int first)
{
  const int v = blockIdx.y;
  size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)n) return;
  uint64_t key = splitmix64(seed ^ splitmix64((uint64_t)(v + first) * 0x100000001B3ULL + idx));
  uint64_t k2 = splitmix64(key);
  double u1 = ((key >> 11) + 0.5) * (1.0 / 9007199254740992.0);
  double u2 = ((k2 >> 11) + 0.5) * (1.0 / 9007199254740992.0);
  double rad = sqrt(-2.0 * log(u1));
  double s, c;
  sincos(6.283185307179586 * u2, &s, &c);
  X[(size_t)v * xs + idx] = cmk(T(rad * c), T(rad * s));
}

// ----------------------------------------------------------------- adjoint
// sum_v w_v |curl e_v|_c^2 / (hx hy) per cell: ADD, with the weights w, added to
// out; else with w_v = 1 / (e_v^H M e_v) from the vectors' Gram sums w (pair
// (v, v)), written to out, which may be host memory.
template <bool ADD>
__global__ __launch_bounds__(256) void k_eta_grad(mxh_level lv, mxh_bloch bl, int nv, const C<double>* E,
                                                 long long es, const double* w, double* out)
{
  const size_t N = (size_t)lv.nx * lv.ny;
  size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= N) return;
  const int j = (int)((unsigned)idx / (unsigned)lv.nx), i = (int)idx - j * lv.nx;
  const double s = 1.0 / (lv.hx * lv.hy);
  double acc = 0.0;
  for (int v = 0; v < nv; v++) {
    Geo<double> g = make_geo<double>(lv, bl, v);
    EdgeV<double> e = edge_view<double>(E, es, v, N);
    C<double> c = cell_curl(g, e, i, j);
    acc += (ADD ? w[v] : 1.0 / w[4 * (v * (v + 1) / 2 + v) + 2]) * (c.r * c.r + c.i * c.i) * s;
  }
  out[idx] = ADD ? out[idx] + acc : acc;
}

// ----------------------------------------------------------------- tile-fused AFW sweeps
// One workgroup smooths a T x T block of nodes of one vector (T = R - 20).  It
// loads the surrounding R x R region (halo TILE_H) into LDS in the
// unwrapped Bloch frame, runs whole colour sweeps there (patches of one colour
// are independent; a sweep moves the region of exact values inward by 4 nodes
// forward and 5 backward), and writes the owned block back.  Per sweep the
// vector is read and written once instead of once per colour.  One thread
// owns one 2x2 node block, i.e. one patch of every colour.  LDS is split by
// node parity so that a
// colour phase reads consecutive addresses across a wavefront.  x, y and the
// right-hand side live in LDS (4 R^2 complex values); eta in registers.
// Region side R (FP32: 64, 1024 threads, owned 44; FP64: 48, 576 threads,
// owned 28), halo 10: two forward sweeps with the residual and its
// restriction (4 + 4 + 2) or two backward sweeps (5 + 5) stay exact on the
// owned block, so a launch does both sweeps of a V(2,2) half-cycle.  The four
// LDS arrays take 128 KB (FP32) / 144 KB (FP64).  Measured alternative: FP32
// R = 48 with two workgroups per CU was slower (more halo work and register
// spills).
#define TILE_H 10
// Rows by which the exact region shrinks: per forward / backward AFW sweep,
// per nodal sweep, and for a residual with its restriction.
#define TILE_SHRINK_FWD 4
#define TILE_SHRINK_BWD 5
#define TILE_SHRINK_RES 2

template <int R>
MXH_DEV int lidx(int i, int j)
{
  return ((((j & 1) << 1) | (i & 1)) * ((R / 2) * (R / 2))) + (j >> 1) * (R / 2) + (i >> 1);
}

template <typename T> struct TileCfg;
#ifndef MXH_TILE_R_F32
#define MXH_TILE_R_F32 64
#endif
#ifndef MXH_TILE_WAVES_F32
#define MXH_TILE_WAVES_F32 1
#endif
template <> struct TileCfg<float> { static const int R = MXH_TILE_R_F32; };
template <> struct TileCfg<double> { static const int R = 48; };

// wrap (i,j) into the grid for any number of periods; returns the phase
template <typename T>
MXH_DEV C<T> wrap_any(int& i, int& j, int nx, int ny, C<T> xf, C<T> yf)
{
  C<T> ph = cmk(T(1), T(0));
  while (i < 0) { i += nx; ph = ph * cconj(xf); }
  while (i >= nx) { i -= nx; ph = ph * xf; }
  while (j < 0) { j += ny; ph = ph * cconj(yf); }
  while (j >= ny) { j -= ny; ph = ph * yf; }
  return ph;
}

template <typename T>
MXH_DEV C<T> load_any(const C<T>* a, int i, int j, int nx, int ny, C<T> xf, C<T> yf)
{
  C<T> ph = wrap_any(i, j, nx, ny, xf, yf);
  return ph * a[i + (size_t)j * nx];
}

template <typename T>
MXH_DEV T eta_any(const T* e, int i, int j, int nx, int ny)
{
  while (i < 0) i += nx;
  while (i >= nx) i -= nx;
  while (j < 0) j += ny;
  while (j >= ny) j -= ny;
  return e[i + (size_t)j * nx];
}

// The AFW patch update of k_afw_phase on LDS values (unwrapped frame).
template <int R, typename T>
MXH_DEV void tile_patch(C<T>* sx, C<T>* sy, int i, int j, C<T> b0, C<T> b1, C<T> b2, C<T> b3, T eLL, T eRL,
                        T eLU, T eRU, T mx, T my)
{
  const int iL0 = lidx<R>(i - 1, j), iR0 = lidx<R>(i, j), iCm = lidx<R>(i, j - 1), iC0 = iR0;
  C<T> xLm = sx[lidx<R>(i - 1, j - 1)], xL0 = sx[iL0], xLp = sx[lidx<R>(i - 1, j + 1)];
  C<T> xRm = sx[iCm], xR0 = sx[iR0], xRp = sx[lidx<R>(i, j + 1)];
  C<T> yLm = sy[lidx<R>(i - 1, j - 1)], yCm = sy[iCm], yRm = sy[lidx<R>(i + 1, j - 1)];
  C<T> yL0 = sy[iL0], yC0 = sy[iC0], yR0 = sy[lidx<R>(i + 1, j)];
  C<T> qLL = eLL * (xLm - xL0 - yLm + yCm);
  C<T> qRL = eRL * (xRm - xR0 - yCm + yRm);
  C<T> qLU = eLU * (xL0 - xLp - yL0 + yC0);
  C<T> qRU = eRU * (xR0 - xRp - yC0 + yR0);
  C<T> r0 = b0 - (qLU - qLL) - mx * (T(4) * xL0 + xLm + xLp);
  C<T> r1 = b1 - (qRU - qRL) - mx * (T(4) * xR0 + xRm + xRp);
  C<T> r2 = b2 - (qLL - qRL) - my * (T(4) * yCm + yLm + yRm);
  C<T> r3 = b3 - (qLU - qRU) - my * (T(4) * yC0 + yL0 + yR0);
  C<T> z0, z1, z2, z3;
  afw_local_solve(eLL, eRL, eLU, eRU, mx, my, r0, r1, r2, r3, z0, z1, z2, z3);
  sx[iL0] = xL0 + z0;
  sx[iR0] = xR0 + z1;
  sy[iCm] = yCm + z2;
  sy[iC0] = yC0 + z3;
}

// mode bits: 1 = backward colour order, 2 = x starts at zero, 4 = add the
// prolongation of the coarse vector XC at load, 8 = after the sweeps form the
// residual and write its restriction to BC (and zero XC).
template <typename T, int MODE, int R = TileCfg<T>::R>
__global__ __launch_bounds__((R / 2) * (R / 2)) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? MXH_TILE_WAVES_F32 : 1))) void k_afw_tile(mxh_level lv, mxh_bloch bl, const C<T>* B, long long bs,
                                                   const C<T>* Xin, C<T>* Xout, long long xs, const T* eta, int nsweep,
                                                   const C<T>* XCin,
                                                   C<T>* BC, C<T>* XC, long long cs, int ntx)
{
  __shared__ C<T> sx[R * R];
  __shared__ C<T> sy[R * R];
  __shared__ C<T> sbx[R * R];
  __shared__ C<T> sby[R * R];
  const int v = blockIdx.y;
  const int nx = lv.nx, ny = lv.ny;
  const size_t N = (size_t)nx * ny;
  const int tileX = blockIdx.x % ntx, tileY = blockIdx.x / ntx;
  const int ox = tileX * (R - 2 * TILE_H) - TILE_H, oy = tileY * (R - 2 * TILE_H) - TILE_H;  // global node of local (0,0)
  const int bx = threadIdx.x % (R / 2), by = threadIdx.x / (R / 2);
  Geo<T> g = make_geo<T>(lv, bl, v);
  const C<T>* gbx = B + (size_t)v * bs;
  const C<T>* gby = gbx + N;
  const C<T>* gx = Xin + (size_t)v * xs;
  const C<T>* gy = gx + N;
  C<T>* ox_ = Xout + (size_t)v * xs;
  C<T>* oy_ = ox_ + N;
  const T axy = T(1.0 / (lv.hx * lv.hy));
  const T mx = T(lv.hy / lv.hx / 6.0), my = T(lv.hx / lv.hy / 6.0);

  // ---- load x (optionally + P xc) for the thread's 2x2 nodes
  const int cnx = nx >> 1, cny = ny >> 1;
  const size_t NC = (size_t)cnx * cny;
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const int li = 2 * bx + (c & 1), lj = 2 * by + (c >> 1);
    C<T> vx = czero<T>(), vy = czero<T>();
    int gi = ox + li, gj = oy + lj;
    C<T> ph = wrap_any(gi, gj, nx, ny, g.xf, g.yf);
    const size_t k = gi + (size_t)gj * nx;
    sbx[lidx<R>(li, lj)] = ph * gbx[k];
    sby[lidx<R>(li, lj)] = ph * gby[k];
    if (!(MODE & 2)) {
      vx = gx[k];
      vy = gy[k];
      if (MODE & 4) {
        Geo<T> gc = g;
        gc.nx = cnx;
        gc.ny = cny;
        const C<T>* cx = XCin + (size_t)v * cs;
        const C<T>* cy = cx + NC;
        const int I = gi >> 1, J = gj >> 1;
        if (gj & 1) vx += T(0.25) * (gc.at(cx, I, J) + gc.at(cx, I, J + 1));
        else vx += T(0.5) * cx[I + (size_t)J * cnx];
        if (gi & 1) vy += T(0.25) * (gc.at(cy, I, J) + gc.at(cy, I + 1, J));
        else vy += T(0.5) * cy[I + (size_t)J * cnx];
      }
      vx = ph * vx;
      vy = ph * vy;
    }
    sx[lidx<R>(li, lj)] = vx;
    sy[lidx<R>(li, lj)] = vy;
  }
  // ---- eta of the nine cells the thread's four patches touch
  T er[3][3];
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int c = 0; c < 3; c++) er[a][c] = axy * eta_any(eta, ox + 2 * bx - 1 + a, oy + 2 * by - 1 + c, nx, ny);
  __syncthreads();

  // ---- colour sweeps
  for (int s = 0; s < nsweep; s++) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const int c = (MODE & 1) ? 3 - k : k;
      const int ci = c & 1, cj = c >> 1;
      const int i = 2 * bx + ci, j = 2 * by + cj;
      if (i >= 1 && i <= R - 2 && j >= 1 && j <= R - 2)
        tile_patch<R>(sx, sy, i, j, sbx[lidx<R>(i - 1, j)], sbx[lidx<R>(i, j)], sby[lidx<R>(i, j - 1)],
                      sby[lidx<R>(i, j)], er[ci][cj],
                   er[ci + 1][cj], er[ci][cj + 1], er[ci + 1][cj + 1], mx, my);
      __syncthreads();
    }
  }

  // ---- write back the owned nodes
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const int li = 2 * bx + (c & 1), lj = 2 * by + (c >> 1);
    const int gi = ox + li, gj = oy + lj;
    if (li >= TILE_H && li < TILE_H + (R - 2 * TILE_H) && lj >= TILE_H && lj < TILE_H + (R - 2 * TILE_H) && gi < nx && gj < ny) {
      const size_t k = gi + (size_t)gj * nx;
      ox_[k] = sx[lidx<R>(li, lj)];
      oy_[k] = sy[lidx<R>(li, lj)];
    }
  }

  if (MODE & 8) {
    // fine residual b - (K + M) x at the thread's four nodes
    C<T> rx[4], ry[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const int ci = c & 1, cj = c >> 1;
      const int i = 2 * bx + ci, j = 2 * by + cj;
      rx[c] = czero<T>();
      ry[c] = czero<T>();
      if (i >= 1 && i <= R - 2 && j >= 1 && j <= R - 2) {
        C<T> x00 = sx[lidx<R>(i, j)], x0m = sx[lidx<R>(i, j - 1)], x0p = sx[lidx<R>(i, j + 1)];
        C<T> xm0 = sx[lidx<R>(i - 1, j)], xmp = sx[lidx<R>(i - 1, j + 1)];
        C<T> y00 = sy[lidx<R>(i, j)], ym0 = sy[lidx<R>(i - 1, j)], yp0 = sy[lidx<R>(i + 1, j)];
        C<T> y0m = sy[lidx<R>(i, j - 1)], ypm = sy[lidx<R>(i + 1, j - 1)];
        C<T> c00 = x00 - x0p - y00 + yp0, c0m = x0m - x00 - y0m + ypm, cm0 = xm0 - xmp - ym0 + y00;
        C<T> kx = er[ci + 1][cj + 1] * c00 - er[ci + 1][cj] * c0m;
        C<T> ky = er[ci][cj + 1] * cm0 - er[ci + 1][cj + 1] * c00;
        rx[c] = sbx[lidx<R>(i, j)] - kx - mx * (T(4) * x00 + x0m + x0p);
        ry[c] = sby[lidx<R>(i, j)] - ky - my * (T(4) * y00 + ym0 + yp0);
      }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const int li = 2 * bx + (c & 1), lj = 2 * by + (c >> 1);
      sx[lidx<R>(li, lj)] = rx[c];
      sy[lidx<R>(li, lj)] = ry[c];
    }
    __syncthreads();
    const int nco = (R - 2 * TILE_H) / 2;
    if ((int)threadIdx.x < nco * nco) {
      const int cI = threadIdx.x % nco, cJ = threadIdx.x / nco;
      const int fi = TILE_H + 2 * cI, fj = TILE_H + 2 * cJ;
      const int GI = tileX * nco + cI, GJ = tileY * nco + cJ;
      if (GI < cnx && GJ < cny) {
        C<T> cxv = T(0.5) * (sx[lidx<R>(fi, fj)] + sx[lidx<R>(fi + 1, fj)]) +
                   T(0.25) * (sx[lidx<R>(fi, fj - 1)] + sx[lidx<R>(fi + 1, fj - 1)] + sx[lidx<R>(fi, fj + 1)] +
                              sx[lidx<R>(fi + 1, fj + 1)]);
        C<T> cyv = T(0.5) * (sy[lidx<R>(fi, fj)] + sy[lidx<R>(fi, fj + 1)]) +
                   T(0.25) * (sy[lidx<R>(fi - 1, fj)] + sy[lidx<R>(fi - 1, fj + 1)] + sy[lidx<R>(fi + 1, fj)] +
                              sy[lidx<R>(fi + 1, fj + 1)]);
        C<T>* bc = BC + (size_t)v * cs;
        C<T>* xc = XC + (size_t)v * cs;
        const size_t k = GI + (size_t)GJ * cnx;
        bc[k] = cxv;
        bc[NC + k] = cyv;
        xc[k] = czero<T>();
        xc[NC + k] = czero<T>();
      }
    }
  }
}

// ----------------------------------------------------------------- tile-fused nodal GS
// The nodal counterpart of k_afw_tile: pointwise Gauss-Seidel for the Q1
// Laplacian in four colours; a sweep moves the exact region inward by 4.
// x and b of the R x R region live in LDS.  R = 64, and FEW_R where a launch has
// few tiles (as k_afw_few).
#define FEW_R 32
template <typename T, int MODE, int R>
__global__ __launch_bounds__(R* R / 4) void k_node_tile(mxh_level lv, mxh_bloch bl, const C<T>* B, long long bs,
                                                    const C<T>* Xin, C<T>* Xout, long long xs, int nsweep,
                                                    const C<T>* XCin, C<T>* BC, C<T>* XC, long long cs, int ntx)
{
  __shared__ C<T> sx[R * R];
  __shared__ C<T> sb[R * R];
  const int v = blockIdx.y;
  const int nx = lv.nx, ny = lv.ny;
  const int tileX = blockIdx.x % ntx, tileY = blockIdx.x / ntx;
  const int TT = R - 2 * TILE_H;
  const int ox = tileX * TT - TILE_H, oy = tileY * TT - TILE_H;
  const int bx = threadIdx.x % (R / 2), by = threadIdx.x / (R / 2);
  Geo<T> g = make_geo<T>(lv, bl, v);
  const C<T>* gb = B + (size_t)v * bs;
  const C<T>* gx = Xin + (size_t)v * xs;
  C<T>* gout = Xout + (size_t)v * xs;
  NodeCoef<T> nc = node_coef<T>(lv, 1.0);
  const T iac = T(1) / nc.ac;
  const int cnx = nx >> 1, cny = ny >> 1;
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const int li = 2 * bx + (c & 1), lj = 2 * by + (c >> 1);
    int gi = ox + li, gj = oy + lj;
    C<T> ph = wrap_any(gi, gj, nx, ny, g.xf, g.yf);
    const size_t k = gi + (size_t)gj * nx;
    sb[lidx<R>(li, lj)] = ph * gb[k];
    C<T> vx = czero<T>();
    if (!(MODE & 2)) {
      vx = gx[k];
      if (MODE & 4) {
        Geo<T> gc = g;
        gc.nx = cnx;
        gc.ny = cny;
        const C<T>* xc = XCin + (size_t)v * cs;
        const int I = gi >> 1, J = gj >> 1;
        const T wx1 = (gi & 1) ? T(0.5) : T(0), wx0 = (gi & 1) ? T(0.5) : T(1);
        const T wy1 = (gj & 1) ? T(0.5) : T(0), wy0 = (gj & 1) ? T(0.5) : T(1);
        C<T> p = (wx0 * wy0) * xc[I + (size_t)J * cnx];
        if (gi & 1) p += (wx1 * wy0) * gc.at(xc, I + 1, J);
        if (gj & 1) p += (wx0 * wy1) * gc.at(xc, I, J + 1);
        if ((gi & 1) && (gj & 1)) p += (wx1 * wy1) * gc.at(xc, I + 1, J + 1);
        vx += p;
      }
      vx = ph * vx;
    }
    sx[lidx<R>(li, lj)] = vx;
  }
  __syncthreads();
  for (int s = 0; s < nsweep; s++) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const int c = (MODE & 1) ? 3 - k : k;
      const int i = 2 * bx + (c & 1), j = 2 * by + (c >> 1);
      if (i >= 1 && i <= R - 2 && j >= 1 && j <= R - 2) {
        C<T> off = nc.ax * (sx[lidx<R>(i - 1, j)] + sx[lidx<R>(i + 1, j)]) +
                   nc.ay * (sx[lidx<R>(i, j - 1)] + sx[lidx<R>(i, j + 1)]) +
                   nc.ad * (sx[lidx<R>(i - 1, j - 1)] + sx[lidx<R>(i + 1, j - 1)] + sx[lidx<R>(i - 1, j + 1)] +
                            sx[lidx<R>(i + 1, j + 1)]);
        sx[lidx<R>(i, j)] = iac * (sb[lidx<R>(i, j)] - off);
      }
      __syncthreads();
    }
  }
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const int li = 2 * bx + (c & 1), lj = 2 * by + (c >> 1);
    const int gi = ox + li, gj = oy + lj;
    if (li >= TILE_H && li < TILE_H + TT && lj >= TILE_H && lj < TILE_H + TT && gi < nx && gj < ny)
      gout[gi + (size_t)gj * nx] = sx[lidx<R>(li, lj)];
  }
  if (MODE & 8) {
    C<T> r[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const int i = 2 * bx + (c & 1), j = 2 * by + (c >> 1);
      r[c] = czero<T>();
      if (i >= 1 && i <= R - 2 && j >= 1 && j <= R - 2) {
        C<T> off = nc.ax * (sx[lidx<R>(i - 1, j)] + sx[lidx<R>(i + 1, j)]) +
                   nc.ay * (sx[lidx<R>(i, j - 1)] + sx[lidx<R>(i, j + 1)]) +
                   nc.ad * (sx[lidx<R>(i - 1, j - 1)] + sx[lidx<R>(i + 1, j - 1)] + sx[lidx<R>(i - 1, j + 1)] +
                            sx[lidx<R>(i + 1, j + 1)]);
        r[c] = sb[lidx<R>(i, j)] - nc.ac * sx[lidx<R>(i, j)] - off;
      }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 4; c++) sx[lidx<R>(2 * bx + (c & 1), 2 * by + (c >> 1))] = r[c];
    __syncthreads();
    const int nco = TT / 2;
    if ((int)threadIdx.x < nco * nco) {
      const int cI = threadIdx.x % nco, cJ = threadIdx.x / nco;
      const int fi = TILE_H + 2 * cI, fj = TILE_H + 2 * cJ;
      const int GI = tileX * nco + cI, GJ = tileY * nco + cJ;
      if (GI < cnx && GJ < cny) {
        C<T> acc = czero<T>();
#pragma unroll
        for (int dj = -1; dj <= 1; dj++)
#pragma unroll
          for (int di = -1; di <= 1; di++) {
            const T w = T((di == 0 ? 1.0 : 0.5) * (dj == 0 ? 1.0 : 0.5));
            acc += w * sx[lidx<R>(fi + di, fj + dj)];
          }
        const size_t k = GI + (size_t)GJ * cnx;
        BC[(size_t)v * cs + k] = acc;
        XC[(size_t)v * cs + k] = czero<T>();
      }
    }
  }
}

MXH_DEV int wrap_index(int i, int n)
{
  i %= n;
  return i < 0 ? i + n : i;
}

// ----------------------------------------------------------------- whole grids in LDS
// Grids of at most 64 x 64 (one thread per 2 x 2 node block) are smoothed with
// the whole periodic vector in LDS: no halo is loaded or computed (the square
// tiles redo a 64^2 FP64 grid five times over), a colour phase is one patch per
// thread.  Columns are split by parity, so a phase reads consecutive addresses
// across a wavefront; the Bloch phase is applied where a block's neighbour lies
// across the boundary.  What bounds it: vector issue of the patch solves at 64^2,
// the latency of the phases on smaller grids.  192 vectors of 64^2 in FP64, two
// sweeps and prolongation: 58.6 -> 34.9 us (square tiles before).
template <typename T>
struct GridBlock {
  int hx, hy, I, J;       // blocks per side, this thread's block
  int co[4], go[4];       // columns 2I - 1 .. 2I + 2: LDS offset, natural index
  int ro[4], gr[4];       // rows 2J - 1 .. 2J + 2: LDS offset, times nx
  bool wl, wr, wd, wu;    // the left, right, lower, upper neighbour lies across the boundary
  C<T> xf, yf;

  MXH_DEV void set(int nx, int ny, int block)
  {
    hx = nx >> 1;
    hy = ny >> 1;
    J = block / hx;
    I = block - J * hx;
    const int l = I ? I - 1 : hx - 1, r = I + 1 < hx ? I + 1 : 0;
    co[0] = hx + l;
    co[1] = I;
    co[2] = hx + I;
    co[3] = r;
    go[0] = 2 * l + 1;
    go[1] = 2 * I;
    go[2] = 2 * I + 1;
    go[3] = 2 * r;
    ro[0] = (J ? 2 * J - 1 : ny - 1) * nx;
    ro[1] = 2 * J * nx;
    ro[2] = (2 * J + 1) * nx;
    ro[3] = (J + 1 < hy ? 2 * J + 2 : 0) * nx;
#pragma unroll
    for (int a = 0; a < 4; a++) gr[a] = ro[a];
    wl = I == 0;
    wr = I == hx - 1;
    wd = J == 0;
    wu = J == hy - 1;
  }
  // block (I, J) of a region of R x R nodes whose first is (ox, oy), even, of the
  // periodic nx x ny grid; the region's rim has no patches
  template <int R>
  MXH_DEV void set_tile(int nx, int ny, int ox, int oy, int block)
  {
    constexpr int H = R / 2;
    hx = hy = H;
    J = block / H;
    I = block - J * H;
    co[0] = H + max(I - 1, 0);
    co[1] = I;
    co[2] = H + I;
    co[3] = min(I + 1, H - 1);
#pragma unroll
    for (int a = 0; a < 4; a++) ro[a] = min(max(2 * J - 1 + a, 0), R - 1) * R;
    const int x = wrap_index(ox + 2 * I, nx), y = wrap_index(oy + 2 * J, ny);
    wl = x == 0;
    wr = x == nx - 2;
    wd = y == 0;
    wu = y == ny - 2;
    go[0] = wl ? nx - 1 : x - 1;
    go[1] = x;
    go[2] = x + 1;
    go[3] = wr ? 0 : x + 2;
    gr[0] = (wd ? ny - 1 : y - 1) * nx;
    gr[1] = y * nx;
    gr[2] = (y + 1) * nx;
    gr[3] = (wu ? 0 : y + 2) * nx;
  }
  // value at node (2I + DI, 2J + DJ) of an array in LDS (parity-split columns)
  // or, GL, in memory
  template <int DI, int DJ, bool GL = false>
  MXH_DEV C<T> get(const C<T>* s) const
  {
    C<T> v = s[GL ? go[DI + 1] + gr[DJ + 1] : co[DI + 1] + ro[DJ + 1]];
    if (DI == -1 && wl) v = cconj(xf) * v;
    if (DI == 2 && wr) v = xf * v;
    if (DJ == -1 && wd) v = cconj(yf) * v;
    if (DJ == 2 && wu) v = yf * v;
    return v;
  }
  // the stored value of node (2I + DI, 2J + DJ), which get() returned as v,
  // plus d (v + d itself where no phase lies between)
  template <int DI, int DJ>
  MXH_DEV void put(C<T>* s, C<T> v, C<T> d) const
  {
    C<T>* p = s + co[DI + 1] + ro[DJ + 1];
    const bool wx = DI == -1 && wl, wy = DJ == -1 && wd;
    if (wx) d = xf * d;
    if (wy) d = yf * d;
    *p = wx || wy ? *p + d : v + d;
  }
};

// 1 / (hx hy eps) of the cells (2I - 1 .. 2I + 1) x (2J - 1 .. 2J + 1)
template <typename T>
MXH_DEV void grid_eta(const GridBlock<T>& g, const T* eta, T axy, T er[3][3])
{
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++) er[a][b] = axy * eta[g.go[a] + g.gr[b]];
}

// The AFW patch of node (2I + CI, 2J + CJ); b in LDS or, BG, in memory.
template <int CI, int CJ, bool BG, bool RELOAD, typename T>
MXH_DEV void grid_patch(const GridBlock<T>& g, C<T>* sx, C<T>* sy, const C<T>* bx, const C<T>* by,
                        const T er[3][3], T mx, T my)
{
  const C<T> b0 = g.template get<CI - 1, CJ, BG>(bx), b1 = g.template get<CI, CJ, BG>(bx);
  const C<T> b2 = g.template get<CI, CJ - 1, BG>(by), b3 = g.template get<CI, CJ, BG>(by);
  const C<T> xLm = g.template get<CI - 1, CJ - 1>(sx), xL0 = g.template get<CI - 1, CJ>(sx);
  const C<T> xLp = g.template get<CI - 1, CJ + 1>(sx), xRm = g.template get<CI, CJ - 1>(sx);
  const C<T> xR0 = g.template get<CI, CJ>(sx), xRp = g.template get<CI, CJ + 1>(sx);
  const C<T> yLm = g.template get<CI - 1, CJ - 1>(sy), yCm = g.template get<CI, CJ - 1>(sy);
  const C<T> yRm = g.template get<CI + 1, CJ - 1>(sy), yL0 = g.template get<CI - 1, CJ>(sy);
  const C<T> yC0 = g.template get<CI, CJ>(sy), yR0 = g.template get<CI + 1, CJ>(sy);
  T eLL = er[CI][CJ], eRL = er[CI + 1][CJ], eLU = er[CI][CJ + 1], eRU = er[CI + 1][CJ + 1];
  if (RELOAD) asm volatile("" : "+v"(eLL), "+v"(eRL), "+v"(eLU), "+v"(eRU));
  const C<T> qLL = eLL * (xLm - xL0 - yLm + yCm), qRL = eRL * (xRm - xR0 - yCm + yRm);
  const C<T> qLU = eLU * (xL0 - xLp - yL0 + yC0), qRU = eRU * (xR0 - xRp - yC0 + yR0);
  const C<T> r0 = b0 - (qLU - qLL) - mx * (T(4) * xL0 + xLm + xLp);
  const C<T> r1 = b1 - (qRU - qRL) - mx * (T(4) * xR0 + xRm + xRp);
  const C<T> r2 = b2 - (qLL - qRL) - my * (T(4) * yCm + yLm + yRm);
  const C<T> r3 = b3 - (qLU - qRU) - my * (T(4) * yC0 + yL0 + yR0);
  C<T> z0, z1, z2, z3;
  afw_local_solve(eLL, eRL, eLU, eRU, mx, my, r0, r1, r2, r3, z0, z1, z2, z3);
  g.template put<CI - 1, CJ>(sx, xL0, z0);
  g.template put<CI, CJ>(sx, xR0, z1);
  g.template put<CI, CJ - 1>(sy, yCm, z2);
  g.template put<CI, CJ>(sy, yC0, z3);
}

// keeps the compiler from lifting the loads through p out of the sweep loop
// (and, on eta, the coefficients of the local solves)
template <bool RELOAD, typename T>
MXH_DEV const T* reload(const T* p)
{
  if (RELOAD) asm volatile("" : "+s"(p));
  return p;
}

// One four-colour sweep (all threads of the workgroup; act: the thread owns a
// block).  Up to 256 threads a block's b and the coefficients of its local solves
// stay in registers over the sweeps; RELOAD: 1024 threads leave no room, b is
// read and the coefficients are formed again per patch.
template <bool BWD, bool BG, bool RELOAD = false, int NB = 1, typename T>
MXH_DEV void grid_sweep(const GridBlock<T> (&g)[NB], const bool (&act)[NB], C<T>* sx, C<T>* sy, const C<T>* bx,
                        const C<T>* by, const T (&er)[NB][3][3], T mx, T my)
{
#pragma unroll
  for (int k = 0; k < 4; k++) {
#pragma unroll
    for (int q = 0; q < NB; q++)
      if (act[q]) {
        const C<T>*px = reload<RELOAD>(bx), *py = reload<RELOAD>(by);
        switch (BWD ? 3 - k : k) {
        case 0: grid_patch<0, 0, BG, RELOAD>(g[q], sx, sy, px, py, er[q], mx, my); break;
        case 1: grid_patch<1, 0, BG, RELOAD>(g[q], sx, sy, px, py, er[q], mx, my); break;
        case 2: grid_patch<0, 1, BG, RELOAD>(g[q], sx, sy, px, py, er[q], mx, my); break;
        case 3: grid_patch<1, 1, BG, RELOAD>(g[q], sx, sy, px, py, er[q], mx, my); break;
        }
      }
    __syncthreads();
  }
}

// The residual of the block's nodes, restricted to its coarse node (cx, cy):
// the block's own part, then (after a barrier) what its neighbours below and
// to the left lend it, one sum each (px, py, one value per block in LDS).
template <bool BG, typename T>
MXH_DEV void grid_restrict_own(const GridBlock<T>& g, bool act, const C<T>* sx, const C<T>* sy, const C<T>* bx,
                           const C<T>* by, const T er[3][3], T mx, T my, C<T>* px, C<T>* py, C<T>& cx, C<T>& cy)
{
  const int k = g.I + g.J * g.hx;
  if (act) {
    // x(2I - 1 .. 2I + 1, 2J - 1 .. 2J + 2), y(2I - 1 .. 2I + 2, 2J - 1 .. 2J + 1)
    const C<T> x00 = g.template get<-1, 0>(sx), x01 = g.template get<-1, 1>(sx), x02 = g.template get<-1, 2>(sx);
    C<T> X[2][4], Y[4][2];
    X[0][0] = g.template get<0, -1>(sx);
    X[0][1] = g.template get<0, 0>(sx);
    X[0][2] = g.template get<0, 1>(sx);
    X[0][3] = g.template get<0, 2>(sx);
    X[1][0] = g.template get<1, -1>(sx);
    X[1][1] = g.template get<1, 0>(sx);
    X[1][2] = g.template get<1, 1>(sx);
    X[1][3] = g.template get<1, 2>(sx);
    Y[0][0] = g.template get<-1, 0>(sy);
    Y[0][1] = g.template get<-1, 1>(sy);
    Y[1][0] = g.template get<0, 0>(sy);
    Y[1][1] = g.template get<0, 1>(sy);
    Y[2][0] = g.template get<1, 0>(sy);
    Y[2][1] = g.template get<1, 1>(sy);
    Y[3][0] = g.template get<2, 0>(sy);
    Y[3][1] = g.template get<2, 1>(sy);
    const C<T> ym0 = g.template get<0, -1>(sy), ym1 = g.template get<1, -1>(sy), ym2 = g.template get<2, -1>(sy);
    // eta times the curl of the cells (0, 1) x (-1, 0, 1), and of (-1) x (0, 1)
    C<T> q[2][3];
    q[0][0] = er[1][0] * (X[0][0] - X[0][1] - ym0 + ym1);
    q[1][0] = er[2][0] * (X[1][0] - X[1][1] - ym1 + ym2);
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
      for (int b = 0; b < 2; b++) q[a][b + 1] = er[a + 1][b + 1] * (X[a][b + 1] - X[a][b + 2] - Y[a + 1][b] + Y[a + 2][b]);
    const C<T> l0 = er[0][1] * (x00 - x01 - Y[0][0] + Y[1][0]), l1 = er[0][2] * (x01 - x02 - Y[0][1] + Y[1][1]);
    C<T> rx[2][2], ry[2][2];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
      for (int b = 0; b < 2; b++) {
        rx[a][b] = cmk(T(0), T(0)) - (q[a][b + 1] - q[a][b]) - mx * (T(4) * X[a][b + 1] + X[a][b] + X[a][b + 2]);
        ry[a][b] = cmk(T(0), T(0)) - ((a ? q[0][b + 1] : (b ? l1 : l0)) - q[a][b + 1]) -
                   my * (T(4) * Y[a + 1][b] + Y[a][b] + Y[a + 2][b]);
      }
    rx[0][0] += g.template get<0, 0, BG>(bx);
    rx[1][0] += g.template get<1, 0, BG>(bx);
    rx[0][1] += g.template get<0, 1, BG>(bx);
    rx[1][1] += g.template get<1, 1, BG>(bx);
    ry[0][0] += g.template get<0, 0, BG>(by);
    ry[1][0] += g.template get<1, 0, BG>(by);
    ry[0][1] += g.template get<0, 1, BG>(by);
    ry[1][1] += g.template get<1, 1, BG>(by);
    px[k] = rx[0][1] + rx[1][1];
    py[k] = ry[1][0] + ry[1][1];
    cx = T(0.5) * (rx[0][0] + rx[1][0]) + T(0.25) * px[k];
    cy = T(0.5) * (ry[0][0] + ry[0][1]) + T(0.25) * py[k];
  }
}
template <typename T>
MXH_DEV void grid_restrict_lent(const GridBlock<T>& g, bool act, const C<T>* px, const C<T>* py, C<T>& cx, C<T>& cy)
{
  const int k = g.I + g.J * g.hx;
  if (act) {
    C<T> d = px[g.J ? k - g.hx : k + (g.hy - 1) * g.hx], l = py[g.I ? k - 1 : k + g.hx - 1];
    if (g.J == 0) d = cconj(g.yf) * d;
    if (g.I == 0) l = cconj(g.xf) * l;
    cx += T(0.25) * d;
    cy += T(0.25) * l;
  }
}

// x += P xc for the block's nodes: c0, c1 = cx(I, J), cx(I, J + 1), d0, d1 =
// cy(I, J), cy(I + 1, J), the upper and right one with their Bloch factors
template <typename T>
MXH_DEV void grid_prolong(const GridBlock<T>& g, C<T>* sx, C<T>* sy, C<T> c0, C<T> c1, C<T> d0, C<T> d1)
{
  if (g.wu) c1 = g.yf * c1;
  if (g.wr) d1 = g.xf * d1;
  const C<T> h = T(0.5) * c0, q = T(0.25) * (c0 + c1), u = T(0.5) * d0, w = T(0.25) * (d0 + d1);
  sx[g.co[1] + g.ro[1]] += h;
  sx[g.co[2] + g.ro[1]] += h;
  sx[g.co[1] + g.ro[2]] += q;
  sx[g.co[2] + g.ro[2]] += q;
  sy[g.co[1] + g.ro[1]] += u;
  sy[g.co[1] + g.ro[2]] += u;
  sy[g.co[2] + g.ro[1]] += w;
  sy[g.co[2] + g.ro[2]] += w;
}

// block's nodes between LDS and memory
template <typename T>
MXH_DEV void grid_copy_in(const GridBlock<T>& g, C<T>* s, const C<T>* a)
{
#pragma unroll
  for (int b = 1; b < 3; b++)
#pragma unroll
    for (int c = 1; c < 3; c++) s[g.co[c] + g.ro[b]] = a ? a[g.go[c] + g.gr[b]] : czero<T>();
}
template <typename T>
MXH_DEV void grid_copy_out(const GridBlock<T>& g, const C<T>* s, C<T>* a)
{
#pragma unroll
  for (int b = 1; b < 3; b++)
#pragma unroll
    for (int c = 1; c < 3; c++) a[g.go[c] + g.gr[b]] = s[g.co[c] + g.ro[b]];
}

template <typename T> struct GridCfg;
template <> struct GridCfg<float> { static constexpr int TB = 1024, NB = 1; };
template <> struct GridCfg<double> { static constexpr int TB = 512, NB = 2; };

// The passes of k_afw_tile (same modes) on a grid that fits; NB blocks per
// thread (64^2 in FP64: two of 512 threads', in the 256 registers a patch's
// values and coefficients want).
template <typename T, int MODE, int TB, int NB>
__global__ __launch_bounds__(TB) void k_afw_grid(mxh_level lv, mxh_bloch bl, const C<T>* B, long long bs,
                                                 const C<T>* Xin, C<T>* Xout, long long xs, const T* eta, int nsweep,
                                                 const C<T>* XCin, C<T>* BC, C<T>* XC, long long cs)
{
  extern __shared__ double smem[];
  const int v = blockIdx.x, nx = lv.nx, ny = lv.ny, N = nx * ny, NC = N >> 2;
  C<T>*sx = (C<T>*)smem, *sy = sx + N, *px = sy + N, *py = px + NC;  // px, py: MODE 8
  const Geo<T> geo = make_geo<T>(lv, bl, v);
  const C<T>*bx = B + (size_t)v * bs, *by = bx + N;
  const T mx = T(lv.hy / lv.hx / 6.0), my = T(lv.hx / lv.hy / 6.0);
  GridBlock<T> g[NB];
  bool act[NB];
  int kc[NB];
  T er[NB][3][3];
#pragma unroll
  for (int q = 0; q < NB; q++) {
    const int k = (int)threadIdx.x + q * TB;
    act[q] = k < NC;
    g[q].xf = geo.xf;
    g[q].yf = geo.yf;
    g[q].set(nx, ny, act[q] ? k : 0);
    kc[q] = g[q].I + g[q].J * g[q].hx;
    grid_eta(g[q], eta, T(1.0 / (lv.hx * lv.hy)), er[q]);
    if (act[q]) {
      const C<T>* x = (MODE & 2) ? nullptr : Xin + (size_t)v * xs;
      grid_copy_in(g[q], sx, x);
      grid_copy_in(g[q], sy, x ? x + N : nullptr);
      if (MODE & 4) {
        const C<T>*cx = XCin + (size_t)v * cs, *cy = cx + NC;
        grid_prolong(g[q], sx, sy, cx[kc[q]], cx[g[q].J + 1 < g[q].hy ? kc[q] + g[q].hx : g[q].I], cy[kc[q]],
                     cy[g[q].I + 1 < g[q].hx ? kc[q] + 1 : g[q].J * g[q].hx]);
      }
    }
  }
  __syncthreads();
  for (int s = 0; s < nsweep; s++)
    grid_sweep<(MODE & 1) != 0, true, (TB > 256), NB>(g, act, sx, sy, bx, by, er, mx, my);
#pragma unroll
  for (int q = 0; q < NB; q++)
    if (act[q]) {
      C<T>* x = Xout + (size_t)v * xs;
      grid_copy_out(g[q], sx, x);
      grid_copy_out(g[q], sy, x + N);
    }
  if (MODE & 8) {
    C<T> cx[NB], cy[NB];
#pragma unroll
    for (int q = 0; q < NB; q++)
      grid_restrict_own<true>(g[q], act[q], sx, sy, bx, by, er[q], mx, my, px, py, cx[q], cy[q]);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NB; q++) {
      grid_restrict_lent(g[q], act[q], px, py, cx[q], cy[q]);
      if (act[q]) {
        C<T>*bc = BC + (size_t)v * cs, *xc = XC + (size_t)v * cs;
        bc[kc[q]] = cx[q];
        bc[NC + kc[q]] = cy[q];
        xc[kc[q]] = czero<T>();
        xc[NC + kc[q]] = czero<T>();
      }
    }
  }
}

// The passes of k_afw_tile for launches that leave most of the chip idle (a
// vector or a few): regions of 32 x 32 with 12 x 12 owned nodes, one patch per
// thread and colour and one wave per SIMD, so that a launch is as short as its
// chain of eight phases allows (two sweeps of a vector of 128^2 in FP64 10 us,
// the larger tiles 17).  Copies of nodes across the boundary keep the values of the nodes they copy -- the
// Bloch phase is applied where a patch reaches over it, as in k_afw_grid -- so
// every copy is the same to the last bit and the residuals of a cell's edges
// see one curl: with copies in the tile's frame the difference in rounding
// excites gradient fields (error of a PINVIT step 6e-11 instead of 3e-12).
#define FEW_T (FEW_R - 2 * TILE_H)
template <typename T, int MODE>
__global__ __launch_bounds__(FEW_R* FEW_R / 4) void k_afw_few(mxh_level lv, mxh_bloch bl, const C<T>* B, long long bs,
                                                             const C<T>* Xin, C<T>* Xout, long long xs, const T* eta,
                                                             int nsweep, const C<T>* XCin, C<T>* BC, C<T>* XC,
                                                             long long cs, int ntx)
{
  constexpr int R = FEW_R, H = R / 2;
  __shared__ C<T> sx[R * R], sy[R * R], px[H * H], py[H * H];
  const int v = blockIdx.y, nx = lv.nx, ny = lv.ny, tid = threadIdx.x;
  const size_t N = (size_t)nx * ny, NC = N >> 2;
  const int tileX = blockIdx.x % ntx, tileY = blockIdx.x / ntx;
  const int ox = tileX * FEW_T - TILE_H, oy = tileY * FEW_T - TILE_H;
  const Geo<T> geo = make_geo<T>(lv, bl, v);
  const C<T>*bx = B + (size_t)v * bs, *by = bx + N;
  const T mx = T(lv.hy / lv.hx / 6.0), my = T(lv.hx / lv.hy / 6.0);
  GridBlock<T> g;
  g.xf = geo.xf;
  g.yf = geo.yf;
  g.template set_tile<R>(nx, ny, ox, oy, tid);
  T er[3][3];
  grid_eta(g, eta, T(1.0 / (lv.hx * lv.hy)), er);
  const C<T>* x = (MODE & 2) ? nullptr : Xin + (size_t)v * xs;
  grid_copy_in(g, sx, x);
  grid_copy_in(g, sy, x ? x + N : nullptr);
  const int GI = g.go[1] >> 1, GJ = g.gr[1] / (2 * nx), cnx = nx >> 1;
  if (MODE & 4) {
    const C<T>*cx = XCin + (size_t)v * cs, *cy = cx + NC;
    const int k = GI + GJ * cnx;
    grid_prolong(g, sx, sy, cx[k], cx[g.wu ? GI : k + cnx], cy[k], cy[g.wr ? GJ * cnx : k + 1]);
  }
  __syncthreads();
  const bool l = g.I > 0, d = g.J > 0;
  for (int s = 0; s < nsweep; s++)
#pragma unroll
    for (int k = 0; k < 4; k++) {
      switch ((MODE & 1) ? 3 - k : k) {
      case 0: if (l && d) grid_patch<0, 0, true, false>(g, sx, sy, bx, by, er, mx, my); break;
      case 1: if (g.I < H - 1 && d) grid_patch<1, 0, true, false>(g, sx, sy, bx, by, er, mx, my); break;
      case 2: if (l && g.J < H - 1) grid_patch<0, 1, true, false>(g, sx, sy, bx, by, er, mx, my); break;
      case 3: if (g.I < H - 1 && g.J < H - 1) grid_patch<1, 1, true, false>(g, sx, sy, bx, by, er, mx, my); break;
      }
      __syncthreads();
    }
  // owned blocks: the last tiles of a row and column may pass the grid's end
  const bool own = g.I >= TILE_H / 2 && g.I < H - TILE_H / 2 && g.J >= TILE_H / 2 && g.J < H - TILE_H / 2 &&
                   ox + 2 * g.I < nx && oy + 2 * g.J < ny;
  if (own) {
    C<T>* xo = Xout + (size_t)v * xs;
    grid_copy_out(g, sx, xo);
    grid_copy_out(g, sy, xo + N);
  }
  if (MODE & 8) {
    C<T> cx, cy;
    const bool act = l && d && g.I < H - 1 && g.J < H - 1;
    grid_restrict_own<true>(g, act, sx, sy, bx, by, er, mx, my, px, py, cx, cy);
    __syncthreads();
    if (own) {
      const int k = g.I + g.J * H;
      C<T> dn = px[k - H], lf = py[k - 1];
      if (g.wd) dn = cconj(g.yf) * dn;
      if (g.wl) lf = cconj(g.xf) * lf;
      C<T>*bc = BC + (size_t)v * cs, *xc = XC + (size_t)v * cs;
      const size_t kc = GI + (size_t)GJ * cnx;
      bc[kc] = cx + T(0.25) * dn;
      bc[NC + kc] = cy + T(0.25) * lf;
      xc[kc] = czero<T>();
      xc[NC + kc] = czero<T>();
    }
  }
}

// ---- the coarse end of a V-cycle in one launch: levels of at most 32 x 32.
// One workgroup per vector keeps x of every level, b of the lower ones and the
// lent sums in LDS; the coarsest level is a product with the inverse of its
// matrix.  It replaces two launches a level and the triangular solves, all
// latency-bound at any batch size, as it is: 192 vectors from 32^2 to 4^2 in FP64
// 51 us against 160, 640 in FP32 85 us against 330 (phases of one wave on 16^2 and
// 8^2, and the barriers between them).
#define CYCLE_MAXL 6
struct CycleLevels {
  int n;  // levels 0 .. n - 1
  int nx[CYCLE_MAXL], ny[CYCLE_MAXL];
  double hx[CYCLE_MAXL], hy[CYCLE_MAXL];
  const void* eta[CYCLE_MAXL];  // edge cycles
  void *b[CYCLE_MAXL], *x[CYCLE_MAXL];  // where the lower levels' vectors go (null: nowhere)
};

// out = W-product of the coarsest level: x_r = sum_c conj(W[c n + r]) b_c over
// nc = n components laid out as `comp` arrays of nx x ny (parity-split in LDS)
template <typename T>
MXH_DEV void cycle_coarse(int n, int nx, int N, const C<double>* W, const C<T>* b, C<T>* x, double* red)
{
  const int tid = threadIdx.x, grp = max(1, (int)blockDim.x / n);
  auto at = [&](int k) {
    const int c = k / N, q = k - c * N, j = q / nx, i = q - j * nx;
    return c * N + j * nx + (i & 1) * (nx >> 1) + (i >> 1);
  };
  C<double>* part = (C<double>*)red;
  for (int w = tid; w < grp * n; w += blockDim.x) {
    const int r = w % n, q = w / n;
    C<double> s = czero<double>();
    for (int c = q; c < n; c += grp) s += cconj(W[(size_t)c * n + r]) * ccast<double>(b[at(c)]);
    part[w] = s;
  }
  __syncthreads();
  for (int r = tid; r < n; r += blockDim.x) {
    C<double> s = part[r];
    for (int q = 1; q < grp; q++) s += part[q * n + r];
    x[at(r)] = ccast<T>(s);
  }
  __syncthreads();
}

template <typename T>
__global__ __launch_bounds__(256, 2) void k_edge_cycle(CycleLevels cl, mxh_bloch bl, int nu, const C<T>* B, long long bs,
                                                    const int* bmap, C<T>* X, long long xs, int xzero, const double* W0,
                                                    int wper)
{
  extern __shared__ double smem[];
  const int v = blockIdx.x, top = cl.n - 1, tid = threadIdx.x;
  mxh_level lv;
  lv.nx = cl.nx[top];
  lv.ny = cl.ny[top];
  const Geo<T> geo = make_geo<T>(lv, bl, v);
  const int gv = bl.vmap ? bl.vmap[v] : v;
  GridBlock<T> gb[1];
  GridBlock<T>& g = gb[0];
  g.xf = geo.xf;
  g.yf = geo.yf;
  const int NT = lv.nx * lv.ny, n0 = 2 * cl.nx[0] * cl.ny[0];
  const C<double>* W = (const C<double>*)W0 + (wper ? (size_t)(gv / bl.vpp) * n0 * n0 : 0);
  // LDS: x of levels top .. 0, b of levels top - 1 .. 0, lent sums, coarse partial sums
  C<T>* xl = (C<T>*)smem;
  int xtot = 0;
  for (int l = 0; l <= top; l++) xtot += 2 * cl.nx[l] * cl.ny[l];
  C<T>* bl_ = xl + xtot;                 // b of level top - 1 first
  C<T>* px = bl_ + (xtot - 2 * NT);
  C<T>* py = px + (NT >> 2);
  double* red = (double*)(px + (top ? NT >> 1 : 2 * NT));
  const C<T>*gbx = B + (size_t)(bmap ? bmap[v] : v) * bs, *gby = gbx + NT;
  C<T>* xout = X + (size_t)v * xs;

  C<T>*x = xl, *b = bl_ - 2 * NT;  // of the current level (b: lower levels)
  for (int l = top; l > 0; l--) {
    const int nx = cl.nx[l], ny = cl.ny[l], N = nx * ny;
    const bool acts[1] = {tid < (N >> 2)}, act = acts[0];
    g.set(nx, ny, act ? tid : 0);
    const T axy = T(1.0 / (cl.hx[l] * cl.hy[l]));
    const T mx = T(cl.hy[l] / cl.hx[l] / 6.0), my = T(cl.hx[l] / cl.hy[l] / 6.0);
    T er[1][3][3];
    grid_eta(g, (const T*)cl.eta[l], axy, er[0]);
    if (act) {
      const C<T>* src = l == top && !xzero ? xout : nullptr;
      grid_copy_in(g, x, src);
      grid_copy_in(g, x + N, src ? src + N : nullptr);
    }
    __syncthreads();
    C<T> cx, cy;
    if (l == top) {
      for (int s = 0; s < nu; s++) grid_sweep<false, true>(gb, acts, x, x + N, gbx, gby, er, mx, my);
      grid_restrict_own<true>(g, act, x, x + N, gbx, gby, er[0], mx, my, px, py, cx, cy);
    } else {
      for (int s = 0; s < nu; s++) grid_sweep<false, false>(gb, acts, x, x + N, b, b + N, er, mx, my);
      grid_restrict_own<false>(g, act, x, x + N, b, b + N, er[0], mx, my, px, py, cx, cy);
    }
    __syncthreads();
    grid_restrict_lent(g, act, px, py, cx, cy);
    x += 2 * N;
    b += 2 * N;
    if (act) {
      const int NC = N >> 2, k = g.J * g.hx + (g.I & 1) * (g.hx >> 1) + (g.I >> 1);
      b[k] = cx;
      b[NC + k] = cy;
    }
    __syncthreads();
  }
  const int nx0 = cl.nx[0], N0 = nx0 * cl.ny[0];
  if (top == 0) {  // the coarsest level alone
    for (int k = tid; k < 2 * N0; k += blockDim.x) {
      const int c = k / N0, q = k - c * N0, j = q / nx0, i = q - j * nx0;
      px[c * N0 + j * nx0 + (i & 1) * (nx0 >> 1) + (i >> 1)] = gbx[k];
    }
    __syncthreads();
    b = px;
  }
  cycle_coarse(n0, nx0, N0, W, b, x, red);
  for (int l = 1; l <= top; l++) {
    const int nx = cl.nx[l], ny = cl.ny[l], N = nx * ny, NC = N >> 2;
    const bool acts[1] = {tid < NC}, act = acts[0];
    g.set(nx, ny, act ? tid : 0);
    const C<T>* xc = x;
    x -= 2 * N;
    b -= 2 * N;
    const T axy = T(1.0 / (cl.hx[l] * cl.hy[l]));
    const T mx = T(cl.hy[l] / cl.hx[l] / 6.0), my = T(cl.hx[l] / cl.hy[l] / 6.0);
    T er[1][3][3];
    grid_eta(g, (const T*)cl.eta[l], axy, er[0]);
    if (act) {
      // the coarse vector's columns are split by parity too
      auto at = [&](int I, int J) { return J * g.hx + (I & 1) * (g.hx >> 1) + (I >> 1); };
      const int Jp = g.J + 1 < g.hy ? g.J + 1 : 0, Ip = g.I + 1 < g.hx ? g.I + 1 : 0;
      grid_prolong(g, x, x + N, xc[at(g.I, g.J)], xc[at(g.I, Jp)], xc[NC + at(g.I, g.J)], xc[NC + at(Ip, g.J)]);
    }
    __syncthreads();
    if (l == top)
      for (int s = 0; s < nu; s++) grid_sweep<true, true>(gb, acts, x, x + N, gbx, gby, er, mx, my);
    else
      for (int s = 0; s < nu; s++) grid_sweep<true, false>(gb, acts, x, x + N, b, b + N, er, mx, my);
  }
  // out: the top level's x, and the lower levels where asked
  if (top > 0) {
    const bool act = tid < (NT >> 2);
    g.set(lv.nx, lv.ny, act ? tid : 0);
    if (act) {
      grid_copy_out(g, xl, xout);
      grid_copy_out(g, xl + NT, xout + NT);
    }
  } else {
    for (int k = tid; k < 2 * N0; k += blockDim.x) {
      const int c = k / N0, q = k - c * N0, j = q / nx0, i = q - j * nx0;
      xout[k] = x[c * N0 + j * nx0 + (i & 1) * (nx0 >> 1) + (i >> 1)];
    }
  }
  C<T>*xk = xl + 2 * NT, *bk = bl_;
  for (int l = top - 1; l >= 0; l--) {
    const int nx = cl.nx[l], N = nx * cl.ny[l];
    C<T>*xo = (C<T>*)cl.x[l], *bo = (C<T>*)cl.b[l];
    if (xo)
      for (int k = tid; k < 2 * N; k += blockDim.x) {
        const int c = k / N, q = k - c * N, j = q / nx, i = q - j * nx;
        const int s = c * N + j * nx + (i & 1) * (nx >> 1) + (i >> 1);
        xo[k] = xk[s];
        bo[k] = bk[s];
      }
    xk += 2 * N;
    bk += 2 * N;
  }
}

// W[r n + c] = (A^-1)[r, c] from the Cholesky factor L of A (n x n,
// column-major, per problem).  The columns of the inverse are independent: a wave
// solves for two of them, row lane + 64 q of each in lane `lane`, by forward and
// back substitution with no barrier.  A step's unknown goes to all lanes by
// v_readlane and leaves their rows at once; the entries of L it needs depend on
// nothing, so eight steps' are loaded ahead.  What bounds it is that chain of 2 n
// steps: 20 us at 32 rows, 34 at 64, 41 at 72, 126 at 200 (64 problems: 530).  One
// workgroup per problem, with a barrier a row up to 64 rows and a thread per column
// above, took 31, 106, 644 and 5305 (7340).
#define INV_COLS 2

template <int R>
__global__ __launch_bounds__(256) void k_coarse_inverse(int n, const double* L0, double* W0)
{
  const int lane = threadIdx.x & 63;
  const int c0 = __builtin_amdgcn_readfirstlane(((int)blockIdx.y * 4 + (int)(threadIdx.x >> 6)) * INV_COLS);
  if (c0 >= n) return;
  const C<double>* L = (const C<double>*)L0 + (size_t)blockIdx.x * n * n;
  C<double>* W = (C<double>*)W0 + (size_t)blockIdx.x * n * n;
  C<double> w[INV_COLS][R];
  int row[R];  // (lanes past the last row read it and keep zeros)
#pragma unroll
  for (int q = 0; q < R; q++) {
    row[q] = min(lane + 64 * q, n - 1);
#pragma unroll
    for (int c = 0; c < INV_COLS; c++) w[c][q] = cmk(lane + 64 * q == c0 + c ? 1.0 : 0.0, 0.0);
  }
  // L y = unit vector, from the first unit's row on
#pragma unroll
  for (int b = 0; b < R; b++)
    for (int l0 = max(0, c0 - 64 * b) & ~7; l0 < 64 && 64 * b + l0 < n; l0 += 8) {
      C<double> a[8][R];
#pragma unroll
      for (int u = 0; u < 8; u++)
#pragma unroll
        for (int q = b; q < R; q++) a[u][q] = L[row[q] + (size_t)min(64 * b + l0 + u, n - 1) * n];
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const int k = 64 * b + l0 + u;
        if (k >= n) break;  // uniform
        const double inv = 1.0 / a[u][b].r;
#pragma unroll
        for (int c = 0; c < INV_COLS; c++) {
          const C<double> f = lane_value(inv * w[c][b], l0 + u);
          if (lane == l0 + u) w[c][b] = f;
#pragma unroll
          for (int q = b; q < R; q++)
            if (lane + 64 * q > k && lane + 64 * q < n) w[c][q] -= a[u][q] * f;
        }
      }
    }
  // L^H x = y, from the last row up
#pragma unroll
  for (int b = R - 1; b >= 0; b--)
    for (int l0 = min(63, n - 1 - 64 * b) & ~7; l0 >= 0; l0 -= 8) {
      C<double> a[8][R];
#pragma unroll
      for (int u = 0; u < 8; u++)
#pragma unroll
        for (int q = 0; q <= b; q++) a[u][q] = cconj(L[min(64 * b + l0 + u, n - 1) + (size_t)row[q] * n]);
#pragma unroll
      for (int u = 7; u >= 0; u--) {
        const int k = 64 * b + l0 + u;
        if (k >= n) continue;  // uniform
        const double inv = 1.0 / a[u][b].r;
#pragma unroll
        for (int c = 0; c < INV_COLS; c++) {
          const C<double> f = lane_value(inv * w[c][b], l0 + u);
          if (lane == l0 + u) w[c][b] = f;
#pragma unroll
          for (int q = 0; q <= b; q++)
            if (lane + 64 * q < k) w[c][q] -= a[u][q] * f;
        }
      }
    }
  // Hermitian: column c as row c
#pragma unroll
  for (int c = 0; c < INV_COLS; c++)
    if (c0 + c < n)
#pragma unroll
      for (int q = 0; q < R; q++)
        if (lane + 64 * q < n) W[(size_t)(c0 + c) * n + lane + 64 * q] = cconj(w[c][q]);
}

// ---- the nodal counterpart: Gauss-Seidel for the Q1 Laplacian
template <int CI, int CJ, typename T>
MXH_DEV C<T> grid_node_off(const GridBlock<T>& g, const C<T>* s, const NodeCoef<T>& nc)
{
  return nc.ax * (g.template get<CI - 1, CJ>(s) + g.template get<CI + 1, CJ>(s)) +
         nc.ay * (g.template get<CI, CJ - 1>(s) + g.template get<CI, CJ + 1>(s)) +
         nc.ad * (g.template get<CI - 1, CJ - 1>(s) + g.template get<CI + 1, CJ - 1>(s) +
                  g.template get<CI - 1, CJ + 1>(s) + g.template get<CI + 1, CJ + 1>(s));
}
template <int CI, int CJ, bool BG, typename T>
MXH_DEV void grid_node_update(const GridBlock<T>& g, bool act, C<T>* s, const C<T>* b, const NodeCoef<T>& nc, T iac)
{
  if (act) s[g.co[CI + 1] + g.ro[CJ + 1]] = iac * (g.template get<CI, CJ, BG>(b) - grid_node_off<CI, CJ>(g, s, nc));
  __syncthreads();
}
template <bool BWD, bool BG, typename T>
MXH_DEV void grid_node_sweep(const GridBlock<T>& g, bool act, C<T>* s, const C<T>* b, const NodeCoef<T>& nc, T iac)
{
  if (BWD) {
    grid_node_update<1, 1, BG>(g, act, s, b, nc, iac);
    grid_node_update<0, 1, BG>(g, act, s, b, nc, iac);
    grid_node_update<1, 0, BG>(g, act, s, b, nc, iac);
    grid_node_update<0, 0, BG>(g, act, s, b, nc, iac);
  } else {
    grid_node_update<0, 0, BG>(g, act, s, b, nc, iac);
    grid_node_update<1, 0, BG>(g, act, s, b, nc, iac);
    grid_node_update<0, 1, BG>(g, act, s, b, nc, iac);
    grid_node_update<1, 1, BG>(g, act, s, b, nc, iac);
  }
}
// the residual restricted to the block's coarse node; p: three lent values per block
template <bool BG, typename T>
MXH_DEV C<T> grid_node_restrict(const GridBlock<T>& g, bool act, const C<T>* s, const C<T>* b, const NodeCoef<T>& nc,
                                C<T>* p)
{
  const int NC = g.hx * g.hy, k = g.I + g.J * g.hx;
  C<T> acc = czero<T>();
  if (act) {
    const C<T> r00 = g.template get<0, 0, BG>(b) - nc.ac * g.template get<0, 0>(s) - grid_node_off<0, 0>(g, s, nc);
    const C<T> r10 = g.template get<1, 0, BG>(b) - nc.ac * g.template get<1, 0>(s) - grid_node_off<1, 0>(g, s, nc);
    const C<T> r01 = g.template get<0, 1, BG>(b) - nc.ac * g.template get<0, 1>(s) - grid_node_off<0, 1>(g, s, nc);
    const C<T> r11 = g.template get<1, 1, BG>(b) - nc.ac * g.template get<1, 1>(s) - grid_node_off<1, 1>(g, s, nc);
    p[k] = r10;
    p[NC + k] = r01;
    p[2 * NC + k] = r11;
    acc = r00 + T(0.5) * (r10 + r01) + T(0.25) * r11;
  }
  __syncthreads();
  if (act) {
    const int kl = g.I ? k - 1 : k + g.hx - 1, kd = g.J ? k - g.hx : k + (g.hy - 1) * g.hx;
    const int kld = g.J ? kl - g.hx : kl + (g.hy - 1) * g.hx;
    C<T> l = T(0.5) * p[kl] + T(0.25) * p[2 * NC + kl], d = T(0.5) * p[NC + kd] + T(0.25) * p[2 * NC + kd];
    C<T> ld = T(0.25) * p[2 * NC + kld];
    if (g.I == 0) {
      l = cconj(g.xf) * l;
      ld = cconj(g.xf) * ld;
    }
    if (g.J == 0) {
      d = cconj(g.yf) * d;
      ld = cconj(g.yf) * ld;
    }
    acc += l + d + ld;
  }
  return acc;
}

template <typename T>
__global__ __launch_bounds__(256) void k_node_cycle(CycleLevels cl, mxh_bloch bl, int nu, const C<T>* B, long long bs,
                                                    C<T>* X, long long xs, int xzero, const double* W0, int wper)
{
  extern __shared__ double smem[];
  const int v = blockIdx.x, top = cl.n - 1, tid = threadIdx.x;
  mxh_level lv;
  lv.nx = cl.nx[top];
  lv.ny = cl.ny[top];
  const Geo<T> geo = make_geo<T>(lv, bl, v);
  const int gv = bl.vmap ? bl.vmap[v] : v;
  GridBlock<T> g;
  g.xf = geo.xf;
  g.yf = geo.yf;
  const int NT = lv.nx * lv.ny, n0 = cl.nx[0] * cl.ny[0];
  const C<double>* W = (const C<double>*)W0 + (wper ? (size_t)(gv / bl.vpp) * n0 * n0 : 0);
  C<T>* xl = (C<T>*)smem;
  int xtot = 0;
  for (int l = 0; l <= top; l++) xtot += cl.nx[l] * cl.ny[l];
  C<T>*bl_ = xl + xtot, *p = bl_ + (xtot - NT);
  double* red = (double*)(p + NT);
  const C<T>* gb = B + (size_t)v * bs;
  C<T>* xout = X + (size_t)v * xs;
  auto coef = [&](int l) {
    mxh_level q;
    q.hx = cl.hx[l];
    q.hy = cl.hy[l];
    return node_coef<T>(q, 1.0);
  };
  C<T>*x = xl, *b = bl_ - NT;
  for (int l = top; l > 0; l--) {
    const int nx = cl.nx[l], ny = cl.ny[l], N = nx * ny;
    const bool act = tid < (N >> 2);
    g.set(nx, ny, act ? tid : 0);
    const NodeCoef<T> nc = coef(l);
    const T iac = T(1) / nc.ac;
    if (act) grid_copy_in(g, x, l == top && !xzero ? (const C<T>*)xout : nullptr);
    __syncthreads();
    C<T> c;
    if (l == top) {
      for (int s = 0; s < nu; s++) grid_node_sweep<false, true>(g, act, x, gb, nc, iac);
      c = grid_node_restrict<true>(g, act, x, gb, nc, p);
    } else {
      for (int s = 0; s < nu; s++) grid_node_sweep<false, false>(g, act, x, b, nc, iac);
      c = grid_node_restrict<false>(g, act, x, b, nc, p);
    }
    x += N;
    b += N;
    if (act) b[g.J * g.hx + (g.I & 1) * (g.hx >> 1) + (g.I >> 1)] = c;
    __syncthreads();
  }
  const int nx0 = cl.nx[0];
  auto split = [&](int k) {
    const int j = k / nx0, i = k - j * nx0;
    return j * nx0 + (i & 1) * (nx0 >> 1) + (i >> 1);
  };
  if (top == 0) {
    for (int k = tid; k < n0; k += blockDim.x) p[split(k)] = gb[k];
    __syncthreads();
    b = p;
  }
  cycle_coarse(n0, nx0, n0, W, b, x, red);
  for (int l = 1; l <= top; l++) {
    const int nx = cl.nx[l], ny = cl.ny[l], N = nx * ny;
    const bool act = tid < (N >> 2);
    g.set(nx, ny, act ? tid : 0);
    const C<T>* xc = x;
    x -= N;
    b -= N;
    const NodeCoef<T> nc = coef(l);
    const T iac = T(1) / nc.ac;
    if (act) {
      auto at = [&](int I, int J) { return J * g.hx + (I & 1) * (g.hx >> 1) + (I >> 1); };
      const int Jp = g.J + 1 < g.hy ? g.J + 1 : 0, Ip = g.I + 1 < g.hx ? g.I + 1 : 0;
      const C<T> c00 = xc[at(g.I, g.J)];
      C<T> c10 = xc[at(Ip, g.J)], c01 = xc[at(g.I, Jp)], c11 = xc[at(Ip, Jp)];
      if (Ip == 0) {
        c10 = g.xf * c10;
        c11 = g.xf * c11;
      }
      if (Jp == 0) {
        c01 = g.yf * c01;
        c11 = g.yf * c11;
      }
      x[g.co[1] + g.ro[1]] += c00;
      x[g.co[2] + g.ro[1]] += T(0.5) * (c00 + c10);
      x[g.co[1] + g.ro[2]] += T(0.5) * (c00 + c01);
      x[g.co[2] + g.ro[2]] += T(0.25) * (c00 + c10 + c01 + c11);
    }
    __syncthreads();
    if (l == top)
      for (int s = 0; s < nu; s++) grid_node_sweep<true, true>(g, act, x, gb, nc, iac);
    else
      for (int s = 0; s < nu; s++) grid_node_sweep<true, false>(g, act, x, b, nc, iac);
  }
  if (top > 0) {
    const bool act = tid < (NT >> 2);
    g.set(lv.nx, lv.ny, act ? tid : 0);
    if (act) grid_copy_out(g, xl, xout);
  } else {
    for (int k = tid; k < n0; k += blockDim.x) xout[k] = x[split(k)];
  }
  C<T>*xk = xl + NT, *bk = bl_;
  for (int l = top - 1; l >= 0; l--) {
    const int nx = cl.nx[l], N = nx * cl.ny[l];
    C<T>*xo = (C<T>*)cl.x[l], *bo = (C<T>*)cl.b[l];
    if (xo)
      for (int k = tid; k < N; k += blockDim.x) {
        const int j = k / nx, i = k - j * nx, s = j * nx + (i & 1) * (nx >> 1) + (i >> 1);
        xo[k] = xk[s];
        bo[k] = bk[s];
      }
    xk += N;
    bk += N;
  }
}

// ----------------------------------------------------------------- row-marching smoothers
// A workgroup smooths an owned block of W x Hgt nodes of one vector.  It reads
// the (W + 2H) x (Hgt + 2H) region around it row by row, from the bottom, and
// keeps only a ring of rows of x, y and eta in LDS (parity-split columns), so
// the region can be tall: the halo re-read is (1 + 2H/W)(1 + 2H/Hgt) instead
// of the square tile's (R / (R - 2H))^2, and several workgroups share a CU,
// so one workgroup's loads overlap another's patch solves.
//
// The 4-colour sweep is pipelined over rows.  Forward (colours 0,1 on even
// rows, then 2,3 on odd rows): step s runs colour 0 on row 2s together with
// colour 2 on row 2s-3, then colour 1 on row 2s with colour 3 on row 2s-3.
// A colour-2/3 patch on odd row r needs colours 0,1 done on rows r-1 and
// r+1 and must come after every colour-0/1 patch that reads row r, which is
// exactly rows r-1 and r+1; the three-row skew satisfies both, so the result
// is that of the whole-grid colour sweep.  Backward mirrors it (colours 3,2
// on odd row 2s+1 with colours 1,0 on even row 2s-2).
//
// NSW sweeps run in one pass: sweep q trails sweep q-1 by six rows (its
// leading row needs the previous sweep finished on the rows around it, which
// happens one step after that sweep's trailing group passes them), so x, b
// and eta are read once for NSW sweeps.  Wave w runs sweep w/2 on its
// leading (w even) or trailing row group.  The halo H covers the exactness
// margin of NSW sweeps plus the residual (4 per forward sweep, 5 backward, +1).
// After step s, rows f0 = 2s - 4 + bwd - 6 (NSW - 1) and f0 + 1 are final:
// they are written out and (forward, MODE 8) their residual is formed; the
// coarse row f0 / 2 - 1 is then restricted.
#define MARCH_W 128

template <int NSW>
struct MarchCfg {
  static constexpr int H = NSW == 1 ? 6 : 10;     // halo (nodes)
  // rows of the LDS ring: live rows of one step are r0 - 11 .. r0 + 1 with
  // two sweeps (13), r0 - 5 .. r0 + 1 with one (7).  A power of two keeps
  // the slot arithmetic to a mask; FP64 two-sweep AFW passes use the tight
  // 13 rows (with a 3-row residual ring) so that the residual mode fits two
  // workgroups per CU in LDS (the kernels may choose otherwise per mode).
  template <typename T>
  static constexpr int ring() { return NSW == 1 ? 8 : (sizeof(T) == 8 ? 13 : 16); }
  template <typename T>
  static constexpr int rres() { return sizeof(T) == 8 ? 3 : 4; }
  static constexpr int THREADS = MARCH_W * NSW;
};

// LDS slot of ring row r, column c: rows of MARCH_W values, split by column
// parity (a colour phase reads consecutive addresses across a wavefront);
// the row part is wave-uniform, the column part fixed per lane.
MXH_DEV int mcol(int c) { return (c & 1) * (MARCH_W / 2) + (c >> 1); }
template <int RING>
MXH_DEV int rrow(int r)
{
  // r is wave-uniform at every use: keep the modulo in scalar registers
  if ((RING & (RING - 1)) == 0) return r & (RING - 1);
  return __builtin_amdgcn_readfirstlane(((r % RING) + RING) % RING);
}
template <int RING>
MXH_DEV int msl(int r, int c) { return rrow<RING>(r) * MARCH_W + mcol(c); }
// residual rows: three are live (the restriction of coarse row J reads fine
// rows 2J - 1 .. 2J + 1); rings of 3 (FP64) or 4 rows
template <int RRES>
MXH_DEV int rsl(int r, int c) { return rrow<RRES>(r) * MARCH_W + mcol(c); }

// Region-local geometry of a marching tile: local (0,0) is global node
// (ox, oy).  The halo reaches at most H nodes past the grid and the host
// requires nx, ny >= H and a last tile that ends within one period past the
// grid, so one wrap suffices.  Values are loaded raw
// from wrapped addresses and the Bloch phase is applied where they are used,
// so a load is never waited for before the next barrier.
template <typename T>
struct MarchGeo {
  int nx, ny, ox, oy;
  C<T> xf, yf;
  // value at unwrapped local (lc, lr) from the raw value stored at the
  // wrapped address
  MXH_DEV C<T> fix(C<T> raw, int lc, int lr) const
  {
    const int gi = ox + lc, gj = oy + lr;
    if ((unsigned)gi < (unsigned)nx && (unsigned)gj < (unsigned)ny) return raw;
    C<T> ph = cmk(T(1), T(0));
    if (gi < 0) ph = cconj(xf);
    else if (gi >= nx) ph = xf;
    if (gj < 0) ph = ph * cconj(yf);
    else if (gj >= ny) ph = ph * yf;
    return ph * raw;
  }
  // the column part of fix's phase at local column lc (a lane's columns are
  // fixed for a whole pass, so this is formed once per lane)
  MXH_DEV C<T> colph(int lc) const
  {
    const int gi = ox + lc;
    return gi < 0 ? cconj(xf) : (gi >= nx ? xf : cmk(T(1), T(0)));
  }
  // fix with the column phase cph = colph(lc) given; lr wave-uniform.  The
  // same products in the same order as fix (a phase of exactly 1 leaves raw
  // as it is)
  MXH_DEV C<T> fixc(C<T> raw, C<T> cph, int lr) const
  {
    const int gj = oy + lr;
    if (gj < 0) cph = cph * cconj(yf);
    else if (gj >= ny) cph = cph * yf;
    return cph * raw;
  }
};

// Raw loads of one region row at one column (x, y, eta).
template <typename T>
struct MarchRow {
  C<T> x, y;
  T e;
};

// mode bits as for k_afw_tile: 1 backward, 2 x starts at zero, 4 add the
// prolongation of XC at load, 8 (forward only) residual + restriction to BC
// (and XC = 0).
template <typename T, int MODE, int NSW>
__global__ __launch_bounds__(MarchCfg<NSW>::THREADS) void k_afw_march(mxh_level lv, mxh_bloch bl, const C<T>* B,
                                                                     long long bs, const int* bmap,
                                                                     const C<T>* Xin, C<T>* Xout,
                                                                     long long xs, const T* eta, const C<T>* XCin,
                                                                     C<T>* BC, C<T>* XC, long long cs, int ntx,
                                                                     int W, int Hgt)
{
  constexpr int BWD = MODE & 1;
  constexpr bool ZERO = MODE & 2, PROL = MODE & 4, RES = MODE & 8;
  // two-sweep FP32 passes with a residual or a prolongation take the tight
  // 13-row ring and 3 residual rows as FP64 does: their LDS (37-39 KB) then
  // fits four workgroups per CU
  constexpr bool TIGHT = NSW == 2 && (RES || PROL);
  constexpr int H = MarchCfg<NSW>::H, RING = TIGHT ? 13 : MarchCfg<NSW>::template ring<T>();
  constexpr int RRES = TIGHT ? 3 : MarchCfg<NSW>::template rres<T>();
  constexpr int NRR = RES ? RRES * MARCH_W : 1;
  __shared__ C<T> sx[RING * MARCH_W];
  __shared__ C<T> sy[RING * MARCH_W];
  __shared__ T se[RING * MARCH_W];
  __shared__ C<T> rxs[NRR];
  __shared__ C<T> rys[NRR];
  // MODE 4: coarse x- and y-edge rows of the prolongation, 4-row rings of
  // MARCH_W / 2 + 1 coarse columns, staged one step ahead (as in k_node_march)
  constexpr int NCW = MARCH_W / 2 + 1;
  __shared__ C<T> scx[PROL ? 4 * NCW : 1];
  __shared__ C<T> scy[PROL ? 4 * NCW : 1];
  const int v = blockIdx.y;
  const int nx = lv.nx, ny = lv.ny, cnx = nx >> 1, cny = ny >> 1;
  const size_t N = (size_t)nx * ny, NC = (size_t)cnx * cny;
  const int tileX = blockIdx.x % ntx, tileY = blockIdx.x / ntx;
  const int RW = W + 2 * H, RH = Hgt + 2 * H;
  const Geo<T> g = make_geo<T>(lv, bl, v);
  const MarchGeo<T> mg{nx, ny, tileX * W - H, tileY * Hgt - H, g.xf, g.yf};
  // a region that does not cross the periodic boundary needs no Bloch phases
  const bool inter = mg.ox >= 0 && mg.ox + RW <= nx && mg.oy >= 0 && mg.oy + RH <= ny;
  // the right-hand side of vector v: slot bmap[v] of B when mapped
  const C<T>* gbx = B + (size_t)(bmap ? bmap[v] : v) * bs;
  const C<T>* gby = gbx + N;
  const C<T>* gx = Xin + (size_t)v * xs;
  const C<T>* gy = gx + N;
  const C<T>* cxp = PROL ? XCin + (size_t)v * cs : nullptr;
  const C<T>* cyp = PROL ? cxp + NC : nullptr;
  C<T>* outx = Xout + (size_t)v * xs;
  C<T>* outy = outx + N;
  const T axy = T(1.0 / (lv.hx * lv.hy));
  const T mx = T(lv.hy / lv.hx / 6.0), my = T(lv.hx / lv.hy / 6.0);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int sweep = wave >> 1, lead = !(wave & 1);
  const int c = tid & (MARCH_W - 1);  // column for row loads, write-out, residuals
  const int half = wave >> 1;         // NSW = 2: the row of a pair this thread's wave handles
  const bool cin = c < RW;
  const int ciA = BWD, ciB = 1 - BWD;
  const int pcA = 2 * lane + ciA, pcB = 2 * lane + ciB;
  auto validc = [&](int pc) { return pc >= 1 && pc <= RW - 2; };
  auto validr = [&](int pr) { return pr >= 1 && pr <= RH - 2; };
  // wrapped global column of region column lc (clamped into the region), and
  // wrapped global row of region row lr (wave-uniform)
  auto wcol = [&](int lc) {
    lc = lc < 0 ? 0 : (lc >= RW ? RW - 1 : lc);
    const int gi = mg.ox + lc;
    return gi < 0 ? gi + nx : (gi >= nx ? gi - nx : gi);
  };
  auto wrow = [&](int lr) {
    lr = lr < 0 ? 0 : (lr >= RH ? RH - 1 : lr);
    const int gj = mg.oy + lr;
    return (gj < 0 ? gj + ny : (gj >= ny ? gj - ny : gj));
  };
  // whether values of region row lr need a Bloch phase (lr is wave-uniform
  // at every use: one scalar test per row, so rows of a region inside the
  // grid's columns skip the per-lane test of mg.fix)
  const bool cwrap = mg.ox < 0 || mg.ox + RW > nx;
  auto needfix = [&](int lr) { return !inter && (cwrap || (unsigned)(mg.oy + lr) >= (unsigned)ny); };
  // Bloch phases of the thread's column c and of its lane's patch columns
  // 2 lane, 2 lane + 1 are formed once (colph) and applied per row (fixc):
  // the FP32 residual pass that reads x went from 4.7 to 4.45 ms.  The FP32
  // zero-start residual pass keeps the per-value form (fix): with the
  // precomputed phases its loop compiled slower (4.1 -> 4.5 ms)
  constexpr bool PRECOL = MODE != 10 || sizeof(T) == 8;
  const C<T> phc = mg.colph(c), ph0 = mg.colph(2 * lane), ph1 = mg.colph(2 * lane + 1);
  auto fixcol = [&](C<T> v, C<T> cph, int lc, int lr) { return PRECOL ? mg.fixc(v, cph, lr) : mg.fix(v, lc, lr); };
  const int gC = wcol(c);

  auto load_row = [&](int r, MarchRow<T>& R) {
    const int wj = wrow(r);
    const size_t k = gC + (size_t)wj * nx;
    R.e = eta[k];
    if (!ZERO) {
      R.x = gx[k];
      R.y = gy[k];
    }
  };
  // coarse row lr of the region (global row oy / 2 + lr, wrapped; rows past
  // the region clamped like wrow's), column tid (< NCW) of it
  const int ocx = mg.ox >> 1, ocy = mg.oy >> 1;  // the region's origin is even
  // (a true modulus: where nx is close to the halo, column RW / 2 of a
  // region lies a whole period past the grid, and the columns tid > RW / 2
  // that are staged but never read lie further)
  auto ccol = [&](int li) {
    const int gi = (ocx + li) % cnx;
    return gi < 0 ? gi + cnx : gi;
  };
  auto crow = [&](int lr) {
    const int last = (RH - 1) >> 1;
    lr = lr > last + 1 ? last + 1 : lr;
    const int gj = (ocy + lr) % cny;
    return gj < 0 ? gj + cny : gj;
  };
  const int gcc = PROL && tid < NCW ? ccol(tid) : 0;
  auto store_row = [&](int r, const MarchRow<T>& R) {
    C<T> vx = czero<T>(), vy = czero<T>();
    if (!ZERO) {
      vx = R.x;
      vy = R.y;
      if (PROL) {
        const int wj = wrow(r), I = gC >> 1, J = wj >> 1;
        // the raw coarse values a direct load reads: coarse column c / 2 (+1)
        // and row r / 2 (+1) of the region, wrapped
        const int lI = c >> 1, s0 = ((r >> 1) & 3) * NCW, s1 = (((r >> 1) + 1) & 3) * NCW;
        const C<T> c0 = scx[s0 + lI], d0 = scy[s0 + lI];
        if (wj & 1) {
          const C<T> c1 = scx[s1 + lI];
          vx += T(0.25) * (c0 + (J + 1 == cny ? g.yf * c1 : c1));
        } else {
          vx += T(0.5) * c0;
        }
        if (gC & 1) {
          const C<T> d1 = scy[s0 + lI + 1];
          vy += T(0.25) * (d0 + (I + 1 == cnx ? g.xf * d1 : d1));
        } else {
          vy += T(0.5) * d0;
        }
      }
      if (needfix(r)) {
        vx = fixcol(vx, phc, c, r);
        vy = fixcol(vy, phc, c, r);
      }
    }
    const int k = msl<RING>(r, c);
    sx[k] = vx;
    sy[k] = vy;
    se[k] = axy * R.e;
  };

  // row pairs are loaded one step ahead: NSW = 1: rows r0, r0 + 1 by every
  // thread; NSW = 2: row r0 + half
  MarchRow<T> R0, R1;
  C<T> cpx = czero<T>(), cpy = czero<T>();  // coarse row staged at the end of the step
  if (PROL) {
    if (tid < NCW) {
      scx[tid] = cxp[gcc + (size_t)crow(0) * cnx];
      scy[tid] = cyp[gcc + (size_t)crow(0) * cnx];
      scx[NCW + tid] = cxp[gcc + (size_t)crow(1) * cnx];
      scy[NCW + tid] = cyp[gcc + (size_t)crow(1) * cnx];
      cpx = cxp[gcc + (size_t)crow(2) * cnx];
      cpy = cyp[gcc + (size_t)crow(2) * cnx];
    }
    __syncthreads();
  }
  if (BWD) {
    if (NSW == 1 || half == 0) {
      load_row(0, R0);
      if (cin) store_row(0, R0);
    }
  }
  if (NSW == 1) {
    load_row(BWD, R0);
    load_row(BWD + 1, R1);
  } else {
    load_row(BWD + half, R0);
  }
  const int NS = RH / 2 + 2 + 3 * (NSW - 1);
  // Raw right-hand sides.  Lane l of a wave holds, for its wave's patch row
  // pr, bx and by at columns 2l and 2l + 1 and by at those columns of row
  // pr - 1 (each value loaded once, coalesced): a patch at column pc = 2l
  // takes bx(pc - 1) from lane l - 1 by a cross-lane shuffle, a patch at
  // pc = 2l + 1 has all four values.  Groups are reloaded for the next step
  // right after their last use (the by pair of phase A's parity after phase
  // A, the rest after phase B), so a load has most of a step to land and no
  // register is copied while a load into it is in flight.  Loads are
  // unconditional (clamped addresses): straight-line code lets the compiler
  // count outstanding loads exactly.  nb[8..11]: residual rows.
  C<T> nb[12];  // 0 bx(2l) 1 bx(2l+1) 2 by(2l) 3 by(2l+1) 4 by(2l,pr-1) 5 by(2l+1,pr-1)
  auto prow = [&](int s2) { return 2 * s2 + BWD - 6 * sweep - (lead ? 0 : 3); };
  auto frow = [&](int s2) { return 2 * s2 - 4 + BWD - 6 * (NSW - 1); };
  const int gE = wcol(2 * lane), gO = wcol(2 * lane + 1);
  auto load_by = [&](int s2, int parity) {  // the by pair of one column parity
    const size_t r0o = (size_t)wrow(prow(s2)) * nx, rmo = (size_t)wrow(prow(s2) - 1) * nx;
    const int gc = parity ? gO : gE;
    nb[2 + parity] = gby[gc + r0o];
    nb[4 + parity] = gby[gc + rmo];
  };
  auto load_bx = [&](int s2) {
    const size_t r0o = (size_t)wrow(prow(s2)) * nx;
    nb[0] = gbx[gE + r0o];
    nb[1] = gbx[gO + r0o];
  };
  // (NSW = 2: the wave's one row, f0 + half, in nb[8..9])
  auto load_bR = [&](int s2) {
    if (RES) {
#pragma unroll
      for (int q = 0; q < 2; q++) {
        if (NSW == 2 && q != half) continue;
        const int sl = NSW == 2 ? 0 : q;
        const size_t ro = (size_t)wrow(frow(s2) + q) * nx;
        nb[8 + 2 * sl] = gbx[gC + ro];
        nb[9 + 2 * sl] = gby[gC + ro];
      }
    }
  };
  auto shfl_up1 = [](C<T> v) {
    C<T> r;
    r.r = __shfl_up(v.r, 1, 64);
    r.i = __shfl_up(v.i, 1, 64);
    return r;
  };
  load_bx(0);
  load_by(0, 0);
  load_by(0, 1);
  load_bR(0);
  // restriction of the residual rows of one step (coarse row f0 / 2); run
  // at the top of the next step, after its barrier, so that it needs no
  // barrier of its own and overlaps the other waves' row loads.  FP32: by
  // the first wave; FP64: the x-edges by the first wave, the y-edges by the
  // second (8.9 -> 8.4-8.6 ms for mode 8, 9.1 -> 8.9 ms for mode 10; the
  // same split measured slower in FP32, 4.15 -> 4.6 ms for mode 10)
  auto restrict_row = [&](int f0) {
    if constexpr (sizeof(T) == 4) {
      const int J = f0 / 2, I = tid;  // region-local coarse indices (f0 even)
      const int fi = 2 * I, fj = 2 * J;
      if (f0 >= 0 && tid < MARCH_W / 2 && I >= H / 2 && I < (H + W) / 2 && J >= H / 2 && J < (H + Hgt) / 2) {
        const int GI = mg.ox / 2 + I, GJ = mg.oy / 2 + J;
        if (GI < cnx && GJ < cny) {
          C<T> cxv = T(0.5) * (rxs[rsl<RRES>(fj, fi)] + rxs[rsl<RRES>(fj, fi + 1)]) +
                     T(0.25) * (rxs[rsl<RRES>(fj - 1, fi)] + rxs[rsl<RRES>(fj - 1, fi + 1)] +
                                rxs[rsl<RRES>(fj + 1, fi)] + rxs[rsl<RRES>(fj + 1, fi + 1)]);
          C<T> cyv = T(0.5) * (rys[rsl<RRES>(fj, fi)] + rys[rsl<RRES>(fj + 1, fi)]) +
                     T(0.25) * (rys[rsl<RRES>(fj, fi - 1)] + rys[rsl<RRES>(fj + 1, fi - 1)] +
                                rys[rsl<RRES>(fj, fi + 1)] + rys[rsl<RRES>(fj + 1, fi + 1)]);
          C<T>* bc = BC + (size_t)v * cs;
          C<T>* xc = XC + (size_t)v * cs;
          const size_t k = GI + (size_t)GJ * cnx;
          bc[k] = cxv;
          bc[NC + k] = cyv;
          xc[k] = czero<T>();
          xc[NC + k] = czero<T>();
        }
      }
    } else {
      const int J = f0 / 2, I = lane;
      const int fi = 2 * I, fj = 2 * J;
      if (f0 >= 0 && wave < 2 && I >= H / 2 && I < (H + W) / 2 && J >= H / 2 && J < (H + Hgt) / 2) {
        const int GI = mg.ox / 2 + I, GJ = mg.oy / 2 + J;
        if (GI < cnx && GJ < cny) {
          const size_t k = GI + (size_t)GJ * cnx + (wave ? NC : 0);
          C<T> cv;
          if (wave == 0)
            cv = T(0.5) * (rxs[rsl<RRES>(fj, fi)] + rxs[rsl<RRES>(fj, fi + 1)]) +
                 T(0.25) * (rxs[rsl<RRES>(fj - 1, fi)] + rxs[rsl<RRES>(fj - 1, fi + 1)] +
                            rxs[rsl<RRES>(fj + 1, fi)] + rxs[rsl<RRES>(fj + 1, fi + 1)]);
          else
            cv = T(0.5) * (rys[rsl<RRES>(fj, fi)] + rys[rsl<RRES>(fj + 1, fi)]) +
                 T(0.25) * (rys[rsl<RRES>(fj, fi - 1)] + rys[rsl<RRES>(fj + 1, fi - 1)] +
                            rys[rsl<RRES>(fj, fi + 1)] + rys[rsl<RRES>(fj + 1, fi + 1)]);
          BC[(size_t)v * cs + k] = cv;
          XC[(size_t)v * cs + k] = czero<T>();
        }
      }
    }
  };
  for (int s = 0; s < NS; s++) {
    const int r0 = 2 * s + BWD;
    const int pr = prow(s);
    const bool rv = validr(pr);
    const int f0 = frow(s);
    __syncthreads();
    if (RES && s > 0) restrict_row(frow(s - 1));
    if (NSW == 1) {
      if (cin && r0 < RH) store_row(r0, R0);
      if (cin && r0 + 1 < RH) store_row(r0 + 1, R1);
      load_row(r0 + 2, R0);
      load_row(r0 + 3, R1);
    } else {
      if (cin && r0 + half < RH) store_row(r0 + half, R0);
      load_row(r0 + 2 + half, R0);
    }
    __syncthreads();
#pragma unroll
    for (int ph = 0; ph < 2; ph++) {
      const int pc = ph == 0 ? pcA : pcB;
      const int ci = ph == 0 ? ciA : ciB;
      // Bloch phases of this phase's right-hand sides, applied in place once
      // they are needed (the bx pair in phase A, the phase's by pair); the
      // shuffle below then moves a value already phased for its column
      if (needfix(pr) || needfix(pr - 1)) {
        if (ph == 0) {
          nb[0] = fixcol(nb[0], ph0, 2 * lane, pr);
          nb[1] = fixcol(nb[1], ph1, 2 * lane + 1, pr);
        }
        nb[2 + ci] = fixcol(nb[2 + ci], ci ? ph1 : ph0, pc, pr);
        nb[4 + ci] = fixcol(nb[4 + ci], ci ? ph1 : ph0, pc, pr - 1);
      }
      // bx(pc - 1): for an even column the odd value of lane l - 1 (all lanes
      // take part in the shuffle, outside the patch guard)
      const C<T> bl = ci ? nb[0] : shfl_up1(nb[1]);
      if (rv && validc(pc)) {
        const C<T> b0 = bl, b1 = ci ? nb[1] : nb[0];
        const C<T> b2 = nb[4 + ci], b3 = nb[2 + ci];
        const int rm = rrow<RING>(pr - 1) * MARCH_W, r0_ = rrow<RING>(pr) * MARCH_W;
        const int rp = rrow<RING>(pr + 1) * MARCH_W;
        const int cm = mcol(pc - 1), c0 = mcol(pc), cp = mcol(pc + 1);
        const T eLL = se[rm + cm], eRL = se[rm + c0];
        const T eLU = se[r0_ + cm], eRU = se[r0_ + c0];
        const int iL0 = r0_ + cm, iR0 = r0_ + c0, iCm = rm + c0, iC0 = iR0;
        C<T> xLm = sx[rm + cm], xL0 = sx[iL0], xLp = sx[rp + cm];
        C<T> xRm = sx[iCm], xR0 = sx[iR0], xRp = sx[rp + c0];
        C<T> yLm = sy[rm + cm], yCm = sy[iCm], yRm = sy[rm + cp];
        C<T> yL0 = sy[iL0], yC0 = sy[iC0], yR0 = sy[r0_ + cp];
        C<T> qLL = eLL * (xLm - xL0 - yLm + yCm);
        C<T> qRL = eRL * (xRm - xR0 - yCm + yRm);
        C<T> qLU = eLU * (xL0 - xLp - yL0 + yC0);
        C<T> qRU = eRU * (xR0 - xRp - yC0 + yR0);
        C<T> s0 = b0 - (qLU - qLL) - mx * (T(4) * xL0 + xLm + xLp);
        C<T> s1 = b1 - (qRU - qRL) - mx * (T(4) * xR0 + xRm + xRp);
        C<T> s2 = b2 - (qLL - qRL) - my * (T(4) * yCm + yLm + yRm);
        C<T> s3 = b3 - (qLU - qRU) - my * (T(4) * yC0 + yL0 + yR0);
        C<T> z0, z1, z2, z3;
        afw_local_solve(eLL, eRL, eLU, eRU, mx, my, s0, s1, s2, s3, z0, z1, z2, z3);
        sx[iL0] = xL0 + z0;
        sx[iR0] = xR0 + z1;
        sy[iCm] = yCm + z2;
        sy[iC0] = yC0 + z3;
      }
      if (s + 1 < NS) {
        if (ph == 0) {
          load_by(s + 1, ciA);
        } else {
          load_bx(s + 1);
          load_by(s + 1, ciB);
        }
      }
      // No barrier between the two phases: phase B reads what phase A wrote
      // in the same wave (LDS operations of a wave complete in order), and
      // within a step the four waves' patch rows pr, pr - 3, pr - 6, pr - 9
      // write rows {pr - 1, pr} and read rows pr - 1 .. pr + 1 of their own,
      // which no other wave of the step writes.  The barrier after phase B
      // orders the last sweep's rows before the final rows read them.
      if (ph == 1) __syncthreads();
    }
    // final rows: write the owned part, form residuals
    if (cin) {
#pragma unroll
      for (int q = 0; q < 2; q++) {
        if (NSW == 2 && q != half) continue;
        const int f = f0 + q;
        if (f < 0 || f >= RH) continue;
        const int gi = mg.ox + c, gj = mg.oy + f;
        const int k0 = msl<RING>(f, c);
        if (c >= H && c < H + W && f >= H && f < H + Hgt && gi < nx && gj < ny) {
          outx[gi + (size_t)gj * nx] = sx[k0];
          outy[gi + (size_t)gj * nx] = sy[k0];
        }
        if (RES) {
          C<T> rx = czero<T>(), ry = czero<T>();
          if (validc(c) && validr(f)) {
            const int fm = rrow<RING>(f - 1) * MARCH_W, fr = rrow<RING>(f) * MARCH_W;
            const int fp = rrow<RING>(f + 1) * MARCH_W;
            const int cm = mcol(c - 1), c0 = mcol(c), cp = mcol(c + 1);
            C<T> x00 = sx[k0], x0m = sx[fm + c0], x0p = sx[fp + c0];
            C<T> xm0 = sx[fr + cm], xmp = sx[fp + cm];
            C<T> y00 = sy[k0], ym0 = sy[fr + cm], yp0 = sy[fr + cp];
            C<T> y0m = sy[fm + c0], ypm = sy[fm + cp];
            C<T> c00 = x00 - x0p - y00 + yp0, c0m = x0m - x00 - y0m + ypm, cm0 = xm0 - xmp - ym0 + y00;
            const T e00 = se[k0], e0m = se[fm + c0], em0 = se[fr + cm];
            C<T> kx = e00 * c00 - e0m * c0m;
            C<T> ky = em0 * cm0 - e00 * c00;
            const int sl = NSW == 2 ? 0 : q;
            C<T> bxr = nb[8 + 2 * sl], byr = nb[9 + 2 * sl];
            if (needfix(f)) {
              bxr = fixcol(bxr, phc, c, f);
              byr = fixcol(byr, phc, c, f);
            }
            rx = bxr - kx - mx * (T(4) * x00 + x0m + x0p);
            ry = byr - ky - my * (T(4) * y00 + ym0 + yp0);
          }
          rxs[rsl<RRES>(f, c)] = rx;
          rys[rsl<RRES>(f, c)] = ry;
        }
      }
    }
    if (s + 1 < NS) load_bR(s + 1);
    if (PROL && tid < NCW) {
      // coarse row s + 2 (needed from the next step on; its slot was last
      // read two steps ago), then row s + 3 in flight for the step after
      scx[((s + 2) & 3) * NCW + tid] = cpx;
      scy[((s + 2) & 3) * NCW + tid] = cpy;
      const size_t ro = (size_t)crow(s + 3) * cnx;
      cpx = cxp[gcc + ro];
      cpy = cyp[gcc + ro];
    }
  }
  if (RES) {
    __syncthreads();
    restrict_row(frow(NS - 1));
  }
}

// The nodal counterpart of k_afw_march: pointwise Gauss-Seidel for the Q1
// Laplacian in four colours, the same row pipeline (a node of colour 2/3 on
// odd row r needs colours 0,1 done on rows r-1 and r+1, and colour 0/1 on
// row r+1 reads row r before colour 2/3 touches it) and the same trailing of
// further sweeps, with a ring of x.
template <typename T, int MODE, int NSW>
__global__ __launch_bounds__(MarchCfg<NSW>::THREADS) void k_node_march(mxh_level lv, mxh_bloch bl, const C<T>* B,
                                                                      long long bs, const C<T>* Xin, C<T>* Xout,
                                                                      long long xs, const C<T>* XCin, C<T>* BC,
                                                                      C<T>* XC, long long cs, int ntx, int W, int Hgt)
{
  // two sweeps: a 16-row ring in both precisions (FP64 too: its 42 KB of
  // LDS at three workgroups per CU with two barriers per step beat 36 KB at
  // four with three, 3.35 -> 3.13 ms for the residual pass)
  constexpr int H = MarchCfg<NSW>::H, RING = NSW == 2 ? 16 : MarchCfg<NSW>::template ring<T>();
  constexpr int RRES = MarchCfg<NSW>::template rres<T>();
  constexpr int BWD = MODE & 1;
  constexpr bool ZERO = MODE & 2, PROL = MODE & 4, RES = MODE & 8;
  constexpr int NRR = RES ? RRES * MARCH_W : 1;
  // FP32: the right-hand side rides in the ring with x (loaded once per pass
  // for both sweeps and the residual); FP64 keeps it in registers (LDS)
  constexpr bool BRING = sizeof(T) == 4;
  __shared__ C<T> sx[RING * MARCH_W];
  __shared__ C<T> sb[BRING ? RING * MARCH_W : 1];
  __shared__ C<T> rs[NRR];
  // MODE 4: coarse rows of the prolongation, 4-row ring of MARCH_W / 2 + 1
  // coarse columns: region row r needs coarse rows r / 2 and r / 2 + 1
  // (region-local; the region's origin is even), staged one step ahead so
  // that a fine node reads its four coarse values from LDS
  constexpr int NCW = MARCH_W / 2 + 1;
  __shared__ C<T> scx[PROL ? 4 * NCW : 1];
  // Two barriers per step instead of three where the ring is long enough:
  // the rows a step stores (r0 + half, r0 + 1 + half) then reuse slots of
  // rows RING behind, below every row the previous step's final rows read
  // (f0 - 1 = r0 - 13 for two sweeps), so the step's stores need not wait
  // for the previous step to end.  What the barrier at the top also ordered
  // moves behind the others: the restriction of the previous step's
  // residual rows runs after the stores' barrier, and the next coarse row
  // of the prolongation is staged before the final rows' barrier (the
  // stores of the next step read it; this step's read rows s and s + 1).
  constexpr bool NOTOP = NSW == 2 && RING >= 14;
  const int v = blockIdx.y;
  const int nx = lv.nx, ny = lv.ny, cnx = nx >> 1, cny = ny >> 1;
  const int tileX = blockIdx.x % ntx, tileY = blockIdx.x / ntx;
  const int RW = W + 2 * H, RH = Hgt + 2 * H;
  const Geo<T> g = make_geo<T>(lv, bl, v);
  const MarchGeo<T> mg{nx, ny, tileX * W - H, tileY * Hgt - H, g.xf, g.yf};
  const bool inter = mg.ox >= 0 && mg.ox + RW <= nx && mg.oy >= 0 && mg.oy + RH <= ny;
  const C<T>* gb = B + (size_t)v * bs;
  const C<T>* gx = Xin + (size_t)v * xs;
  const C<T>* xcp = PROL ? XCin + (size_t)v * cs : nullptr;
  C<T>* out = Xout + (size_t)v * xs;
  const NodeCoef<T> nc = node_coef<T>(lv, 1.0);
  const T iac = T(1) / nc.ac;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int sweep = wave >> 1, lead = !(wave & 1);
  const int c = tid & (MARCH_W - 1);
  const int half = wave >> 1;
  const bool cin = c < RW;
  const int ciA = BWD, ciB = 1 - BWD;
  const int pcA = 2 * lane + ciA, pcB = 2 * lane + ciB;
  auto wcol = [&](int lc) {
    lc = lc < 0 ? 0 : (lc >= RW ? RW - 1 : lc);
    const int gi = mg.ox + lc;
    return gi < 0 ? gi + nx : (gi >= nx ? gi - nx : gi);
  };
  auto wrow = [&](int lr) {
    lr = lr < 0 ? 0 : (lr >= RH ? RH - 1 : lr);
    const int gj = mg.oy + lr;
    return (gj < 0 ? gj + ny : (gj >= ny ? gj - ny : gj));
  };
  // whether values of region row lr need a Bloch phase (lr is wave-uniform
  // at every use: one scalar test per row, so rows of a region inside the
  // grid's columns skip the per-lane test of mg.fix)
  const bool cwrap = mg.ox < 0 || mg.ox + RW > nx;
  auto needfix = [&](int lr) { return !inter && (cwrap || (unsigned)(mg.oy + lr) >= (unsigned)ny); };
  const int gA = wcol(pcA), gB = wcol(pcB), gC = wcol(c);

  // raw loads of a row: x and (FP32) b
  struct NRow {
    C<T> x, b;
  };
  auto load_row = [&](int r, NRow& R) {
    const int wj = wrow(r);
    if (BRING) R.b = gb[gC + (size_t)wj * nx];
    if (!ZERO) R.x = gx[gC + (size_t)wj * nx];
  };
  // coarse row lr of the region (global row oy / 2 + lr, wrapped; rows past
  // the region are clamped like wrow's), column tid (< NCW) of it
  const int ocx = mg.ox >> 1, ocy = mg.oy >> 1;  // the region's origin is even
  // (a true modulus: where nx is close to the halo, column RW / 2 of a
  // region lies a whole period past the grid, and the columns tid > RW / 2
  // that are staged but never read lie further)
  auto ccol = [&](int li) {
    const int gi = (ocx + li) % cnx;
    return gi < 0 ? gi + cnx : gi;
  };
  auto crow = [&](int lr) {
    const int last = (RH - 1) >> 1;
    lr = lr > last + 1 ? last + 1 : lr;
    const int gj = (ocy + lr) % cny;
    return gj < 0 ? gj + cny : gj;
  };
  const int gcc = PROL && tid < NCW ? ccol(tid) : 0;
  auto load_crow = [&](int lr) { return xcp[gcc + (size_t)crow(lr) * cnx]; };
  auto finish_row = [&](int r, const NRow& R) {
    C<T> vx = czero<T>();
    if (!ZERO) {
      vx = R.x;
      if (PROL) {
        const int wj = wrow(r), wi = gC;
        const int I = wi >> 1, J = wj >> 1;
        const bool ox1 = I + 1 == cnx, oy1 = J + 1 == cny;
        const T wx1 = (wi & 1) ? T(0.5) : T(0), wx0 = (wi & 1) ? T(0.5) : T(1);
        const T wy1 = (wj & 1) ? T(0.5) : T(0), wy0 = (wj & 1) ? T(0.5) : T(1);
        // the same raw coarse values a direct load reads: coarse column c / 2
        // (+1) and row r / 2 (+1) of the region, wrapped
        const int lI = c >> 1, s0 = ((r >> 1) & 3) * NCW, s1 = (((r >> 1) + 1) & 3) * NCW;
        const C<T> p00 = scx[s0 + lI], p10 = scx[s0 + lI + 1];
        const C<T> p01 = (wj & 1) ? scx[s1 + lI] : czero<T>(), p11 = (wj & 1) ? scx[s1 + lI + 1] : czero<T>();
        C<T> p = (wx0 * wy0) * p00;
        if (wi & 1) p += (wx1 * wy0) * (ox1 ? g.xf * p10 : p10);
        if (wj & 1) p += (wx0 * wy1) * (oy1 ? g.yf * p01 : p01);
        if ((wi & 1) && (wj & 1)) {
          C<T> q = p11;
          if (ox1) q = g.xf * q;
          if (oy1) q = g.yf * q;
          p += (wx1 * wy1) * q;
        }
        vx += p;
      }
      if (needfix(r)) vx = mg.fix(vx, c, r);
    }
    sx[msl<RING>(r, c)] = vx;
    if (BRING) sb[msl<RING>(r, c)] = needfix(r) ? mg.fix(R.b, c, r) : R.b;
  };
  auto validc = [&](int pc) { return pc >= 1 && pc <= RW - 2; };
  auto validr = [&](int pr) { return pr >= 1 && pr <= RH - 2; };
  auto offd = [&](int pc, int pr) {
    const int rm = rrow<RING>(pr - 1) * MARCH_W, r0_ = rrow<RING>(pr) * MARCH_W;
    const int rp = rrow<RING>(pr + 1) * MARCH_W;
    const int cm = mcol(pc - 1), c0 = mcol(pc), cp = mcol(pc + 1);
    return nc.ax * (sx[r0_ + cm] + sx[r0_ + cp]) + nc.ay * (sx[rm + c0] + sx[rp + c0]) +
           nc.ad * (sx[rm + cm] + sx[rm + cp] + sx[rp + cm] + sx[rp + cp]);
  };

  NRow R0, R1;
  C<T> cpre = czero<T>();  // coarse row staged at the end of the step
  if (PROL) {
    if (tid < NCW) {
      scx[tid] = load_crow(0);
      scx[NCW + tid] = load_crow(1);
      cpre = load_crow(2);
    }
    __syncthreads();
  }
  if (BWD) {
    if (NSW == 1 || half == 0) {
      load_row(0, R0);
      if (cin) finish_row(0, R0);
    }
  }
  // FP32, NSW = 2: the wave's row of a step is loaded two steps ahead, into
  // R0 for even steps and R1 for odd ones (the loop below is unrolled by two,
  // so each register set is named statically and the load counts stay
  // exact): the FP32 passes 4-7% faster.  FP64 loads one step ahead (two
  // measured 15% slower there).
  constexpr bool PF2 = NSW == 2 && sizeof(T) == 4;
  if (NSW == 1) {
    load_row(BWD, R0);
    load_row(BWD + 1, R1);
  } else {
    load_row(BWD + half, R0);
    if (PF2) load_row(BWD + 2 + half, R1);
  }
  const int NS = RH / 2 + 2 + 3 * (NSW - 1);
  // raw right-hand sides (patch A, patch B, residual rows), each reloaded for
  // the next step right after its last use
  C<T> nb[4];
  auto prow = [&](int s2) { return 2 * s2 + BWD - 6 * sweep - (lead ? 0 : 3); };
  auto frow = [&](int s2) { return 2 * s2 - 4 + BWD - 6 * (NSW - 1); };
  auto load_bA = [&](int s2) {
    if (!BRING) nb[0] = gb[gA + (size_t)wrow(prow(s2)) * nx];
  };
  auto load_bB = [&](int s2) {
    if (!BRING) nb[1] = gb[gB + (size_t)wrow(prow(s2)) * nx];
  };
  auto bval = [&](int slot, int pc, int prr) {
    return BRING ? sb[msl<RING>(prr, pc)] : (needfix(prr) ? mg.fix(nb[slot], pc, prr) : nb[slot]);
  };
  auto load_bR = [&](int s2) {
    if (RES && !BRING) {
#pragma unroll
      for (int q = 0; q < 2; q++) {
        if (NSW == 2 && q != half) continue;
        nb[NSW == 2 ? 2 : 2 + q] = gb[gC + (size_t)wrow(frow(s2) + q) * nx];
      }
    }
  };
  load_bA(0);
  load_bB(0);
  load_bR(0);
  // restriction of the residual rows of one step (coarse row f0 / 2), run at
  // the top of the next step after its barrier (see k_afw_march)
  auto restrict_row = [&](int f0) {
    const int J = f0 / 2, I = tid;
    const int fi = 2 * I, fj = 2 * J;
    if (f0 >= 0 && tid < MARCH_W / 2 && I >= H / 2 && I < (H + W) / 2 && J >= H / 2 && J < (H + Hgt) / 2) {
      const int GI = mg.ox / 2 + I, GJ = mg.oy / 2 + J;
      if (GI < cnx && GJ < cny) {
        C<T> acc = czero<T>();
#pragma unroll
        for (int dj = -1; dj <= 1; dj++)
#pragma unroll
          for (int di = -1; di <= 1; di++) {
            const T w = T((di == 0 ? 1.0 : 0.5) * (dj == 0 ? 1.0 : 0.5));
            acc += w * rs[rsl<RRES>(fj + dj, fi + di)];
          }
        const size_t k = GI + (size_t)GJ * cnx;
        BC[(size_t)v * cs + k] = acc;
        XC[(size_t)v * cs + k] = czero<T>();
      }
    }
  };
  auto step = [&](int s, NRow& Rc) {
    const int r0 = 2 * s + BWD;
    const int pr = prow(s);
    const bool rv = validr(pr);
    const bool vA = rv && validc(pcA), vB = rv && validc(pcB);
    const int f0 = frow(s);
    if (!NOTOP) {
      __syncthreads();
      if (RES && s > 0) restrict_row(frow(s - 1));
    }
    if (NSW == 1) {
      if (cin && r0 < RH) finish_row(r0, R0);
      if (cin && r0 + 1 < RH) finish_row(r0 + 1, R1);
      load_row(r0 + 2, R0);
      load_row(r0 + 3, R1);
    } else {
      if (cin && r0 + half < RH) finish_row(r0 + half, Rc);
      load_row(r0 + (PF2 ? 4 : 2) + half, Rc);
    }
    __syncthreads();
    if (NOTOP && RES && s > 0) restrict_row(frow(s - 1));
    // colours A and B of a row in one wave with no barrier between them (as
    // in k_afw_march: a wave's rows pr - 1 .. pr + 1 are written by no other
    // wave within the step)
    if (vA) sx[msl<RING>(pr, pcA)] = iac * (bval(0, pcA, pr) - offd(pcA, pr));
    if (s + 1 < NS) load_bA(s + 1);
    if (vB) sx[msl<RING>(pr, pcB)] = iac * (bval(1, pcB, pr) - offd(pcB, pr));
    if (s + 1 < NS) load_bB(s + 1);
    if (NOTOP && PROL && tid < NCW) {
      scx[((s + 2) & 3) * NCW + tid] = cpre;
      cpre = load_crow(s + 3);
    }
    __syncthreads();
    if (cin) {
#pragma unroll
      for (int q = 0; q < 2; q++) {
        if (NSW == 2 && q != half) continue;
        const int f = f0 + q;
        if (f < 0 || f >= RH) continue;
        const int gi = mg.ox + c, gj = mg.oy + f;
        if (c >= H && c < H + W && f >= H && f < H + Hgt && gi < nx && gj < ny)
          out[gi + (size_t)gj * nx] = sx[msl<RING>(f, c)];
        if (RES) {
          C<T> r = czero<T>();
          if (validc(c) && validr(f)) r = bval(NSW == 2 ? 2 : 2 + q, c, f) - nc.ac * sx[msl<RING>(f, c)] - offd(c, f);
          rs[rsl<RRES>(f, c)] = r;
        }
      }
    }
    if (s + 1 < NS) load_bR(s + 1);
    if (!NOTOP && PROL && tid < NCW) {
      // coarse row s + 2 (needed from the next step on; its slot was last
      // read two steps ago), then row s + 3 in flight for the step after
      scx[((s + 2) & 3) * NCW + tid] = cpre;
      cpre = load_crow(s + 3);
    }
  };
  if (PF2) {
    int s = 0;
    for (; s + 1 < NS; s += 2) {
      step(s, R0);
      step(s + 1, R1);
    }
    if (s < NS) step(s, R0);
  } else {
    for (int s = 0; s < NS; s++) step(s, R0);
  }
  if (RES) {
    __syncthreads();
    restrict_row(frow(NS - 1));
  }
}

// ================================================================= launchers
#define LAUNCH_CHECK() do { hipError_t _e = hipGetLastError(); if (_e != hipSuccess) return (int)_e; } while (0)

static int grid_attrs();

extern "C" {

int mxh_init(void)
{
  if (g_stream) return 0;
  int n = 0, dev = 0;
  hipError_t e = hipGetDeviceCount(&n);
  if (e != hipSuccess) return (int)e;
  if (n < 1) return (int)hipErrorNoDevice;
  e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= MXH_MAX_DEVICES) return (int)hipErrorInvalidDevice;
  // the device address of this device's copy of the static scratch array
  // (the array's name is a host-side stand-in, not a device address)
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    g_scratch_ptr[dev] = p;
  }
  // kernels that may use more dynamic LDS than the default limit of a launch
  const void* big[] = {(const void*)k_fft_solve<double>, (const void*)k_fft_solve<float>,
                       (const void*)k_fft_cols<double>, (const void*)k_fft_cols<float>,
                       (const void*)k_fft_rows<double, -1>, (const void*)k_fft_rows<double, 1>,
                       (const void*)k_fft_rows<float, -1>, (const void*)k_fft_rows<float, 1>,
                       (const void*)k_edge_cycle<double>, (const void*)k_edge_cycle<float>,
                       (const void*)k_node_cycle<double>, (const void*)k_node_cycle<float>,
                       (const void*)k_gram<4, 4>, (const void*)k_gram<5, 5>, (const void*)k_gram<6, 5>,
                       (const void*)k_gram<6, 6>, (const void*)k_hh_coef};
  for (const void* f : big) {
    e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, LDS_MAX);
    if (e != hipSuccess) return (int)e;
  }
  // (static LDS counts too)
  e = hipFuncSetAttribute((const void*)k_ritz, hipFuncAttributeMaxDynamicSharedMemorySize,
                          3 * sizeof(C<double>) * RITZ_MAX * RITZ_MAX);
  if (e != hipSuccess || grid_attrs()) return (int)hipErrorInvalidValue;
  e = hipStreamCreateWithFlags(&g_stream, hipStreamNonBlocking);
  if (e != hipSuccess) {
    g_stream = nullptr;
    return (int)e;
  }
  g_device = dev;
  return 0;
}

void* mxh_stream(void) { return (void*)g_stream; }

int mxh_sync(void) { return (int)hipStreamSynchronize(g_stream); }

const char* mxh_error_string(int err)
{
  if (err == MXH_ESCRATCH) return "request exceeds the static scratch of mxh_gram_static";
  return hipGetErrorString((hipError_t)err);
}

void* mxh_malloc(size_t bytes)
{
  void* p = nullptr;
  if (bytes == 0) bytes = 256;
  if (hipMalloc(&p, bytes) != hipSuccess) return nullptr;
  return p;
}

void mxh_free(void* p)
{
  if (p) (void)hipFree(p);
}

int mxh_h2d(void* dst, const void* src, size_t bytes)
{
  return (int)hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, g_stream);
}

int mxh_d2h(void* dst, const void* src, size_t bytes)
{
  hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, g_stream);
  if (e != hipSuccess) return (int)e;
  return (int)hipStreamSynchronize(g_stream);
}

int mxh_h2d_rows(void* dst, size_t dst_pitch, const void* src, size_t row, int rows)
{
  if (dst_pitch == row) return mxh_h2d(dst, src, row * (size_t)rows);
  return (int)hipMemcpy2DAsync(dst, dst_pitch, src, row, row, rows, hipMemcpyHostToDevice, g_stream);
}

int mxh_d2h_rows(void* dst, const void* src, size_t src_pitch, size_t row, int rows)
{
  if (src_pitch == row) return mxh_d2h(dst, src, row * (size_t)rows);
  hipError_t e = hipMemcpy2DAsync(dst, row, src, src_pitch, row, rows, hipMemcpyDeviceToHost, g_stream);
  if (e != hipSuccess) return (int)e;
  return (int)hipStreamSynchronize(g_stream);
}

int mxh_d2h_async(void* dst, const void* src, size_t bytes)
{
  return (int)hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, g_stream);
}

void* mxh_host_alloc(size_t bytes)
{
  void* p = nullptr;
  if (hipHostMalloc(&p, bytes ? bytes : 256, hipHostMallocDefault) != hipSuccess) return nullptr;
  return p;
}

void mxh_host_free(void* p)
{
  if (p) (void)hipHostFree(p);
}

int mxh_event_sync(void* ev) { return (int)hipEventSynchronize((hipEvent_t)ev); }

int mxh_d2d(void* dst, const void* src, size_t bytes)
{
  // up to a few MB a launch of our own is queued sooner than the runtime's copy
  if (bytes && bytes <= ((size_t)4 << 20) && !(((size_t)dst | (size_t)src | bytes) & 15)) {
    hipLaunchKernelGGL(k_copy, dim3(nblocks((long long)(bytes / 16))), dim3(TPB), 0, g_stream, bytes / 16,
                       (const uint4*)src, (uint4*)dst);
    LAUNCH_CHECK();
    return 0;
  }
  return (int)hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, g_stream);
}

int mxh_memset(void* dst, int value, size_t bytes)
{
  return (int)hipMemsetAsync(dst, value, bytes, g_stream);
}



int mxh_addeval(int prec, const mxh_level* lv, const mxh_bloch* bl, int nv, mxh_vecs x, mxh_vecs y,
                const void* eta, const mxh_coef* cf, int accumulate)
{
  const long long N = (long long)lv->nx * lv->ny;
  dim3 grid(nblocks(N), nv);
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_addeval<double>, grid, dim3(TPB), 0, g_stream, *lv, *bl, (const C<double>*)x.p,
                       x.stride, (C<double>*)y.p, y.stride, (const double*)eta, *cf, accumulate);
  else
    hipLaunchKernelGGL(k_addeval<float>, grid, dim3(TPB), 0, g_stream, *lv, *bl, (const C<float>*)x.p,
                       x.stride, (C<float>*)y.p, y.stride, (const float*)eta, *cf, accumulate);
  LAUNCH_CHECK();
  return 0;
}

int mxh_defect(int rprec, const mxh_level* lv, const mxh_bloch* bl, int nv, mxh_vecs e, mxh_vecs r,
               const double* eta64, const double* lam, double* out, double* work)
{
  const unsigned nb = band_blocks(lv, nv);
  auto go = [&](auto kernel, auto* to) {
    hipLaunchKernelGGL(kernel, dim3(nb, nv), dim3(TPB), 0, g_stream, *lv, *bl, (const C<double>*)e.p, e.stride, e.map, to,
                       r.stride, eta64, lam, work);
  };
  if (rprec == MXH_F64)
    narrow(lv) ? go(k_defect<double, true>, (C<double>*)r.p) : go(k_defect<double, false>, (C<double>*)r.p);
  else
    narrow(lv) ? go(k_defect<float, true>, (C<float>*)r.p) : go(k_defect<float, false>, (C<float>*)r.p);
  LAUNCH_CHECK();
  hipLaunchKernelGGL(k_reduce_partials, dim3(reduce_blocks(2 * nv)), dim3(TPB), 0, g_stream, work, (int)nb, 2 * nv,
                     out, 0);
  LAUNCH_CHECK();
  return 0;
}

int mxh_afw_phase(int prec, const mxh_level* lv, const mxh_bloch* bl, int nv, mxh_vecs b, mxh_vecs x,
                  const void* eta, double alpha, double beta, int colour)
{
  if ((lv->nx & 1) || (lv->ny & 1)) return (int)hipErrorInvalidValue;
  const long long np = (long long)(lv->nx / 2) * (lv->ny / 2);
  dim3 grid(nblocks(np), nv);
  const int ci = colour & 1, cj = colour >> 1;
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_afw_phase<double>, grid, dim3(TPB), 0, g_stream, *lv, *bl, (const C<double>*)b.p,
                       b.stride, (C<double>*)x.p, x.stride, (const double*)eta, alpha, beta, ci, cj);
  else
    hipLaunchKernelGGL(k_afw_phase<float>, grid, dim3(TPB), 0, g_stream, *lv, *bl, (const C<float>*)b.p,
                       b.stride, (C<float>*)x.p, x.stride, (const float*)eta, alpha, beta, ci, cj);
  LAUNCH_CHECK();
  return 0;
}

int mxh_edge_gs_phase(int prec, const mxh_level* lv, const mxh_bloch* bl, int nv, mxh_vecs b, mxh_vecs x,
                      const void* eta, const mxh_coef* cf, int colour)
{
  if ((lv->nx & 1) || (lv->ny & 1) || colour < 0 || colour > 3) return (int)hipErrorInvalidValue;
  const long long np = (long long)lv->nx * lv->ny / 2;
  dim3 grid(nblocks(np), nv);
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_edge_gs_phase<double>, grid, dim3(TPB), 0, g_stream, *lv, *bl, (const C<double>*)b.p,
                       b.stride, (C<double>*)x.p, x.stride, (const double*)eta, *cf, colour);
  else
    hipLaunchKernelGGL(k_edge_gs_phase<float>, grid, dim3(TPB), 0, g_stream, *lv, *bl, (const C<float>*)b.p,
                       b.stride, (C<float>*)x.p, x.stride, (const float*)eta, *cf, colour);
  LAUNCH_CHECK();
  return 0;
}

extern "C++" {
template <typename T, int MODE>
static void launch_tile(dim3 grid, dim3 block, const mxh_level* lv, const mxh_bloch* bl, mxh_vecs b, mxh_vecs x,
                        mxh_vecs xo, const void* eta, int nsweep, mxh_vecs xc_in, mxh_vecs bc, mxh_vecs xc,
                        long long cs, int ntx)
{
  hipLaunchKernelGGL((k_afw_tile<T, MODE>), grid, block, 0, g_stream, *lv, *bl, (const C<T>*)b.p, b.stride,
                     (const C<T>*)x.p, (C<T>*)xo.p, x.stride, (const T*)eta, nsweep, (const C<T>*)xc_in.p,
                     (C<T>*)bc.p, (C<T>*)xc.p, cs, ntx);
}

template <typename T>
static int launch_tile_mode(int mode, dim3 grid, dim3 block, const mxh_level* lv, const mxh_bloch* bl, mxh_vecs b,
                            mxh_vecs x, mxh_vecs xo, const void* eta, int nsweep, mxh_vecs xc_in, mxh_vecs bc,
                            mxh_vecs xc, long long cs, int ntx)
{
  switch (mode) {
  case 0: launch_tile<T, 0>(grid, block, lv, bl, b, x, xo, eta, nsweep, xc_in, bc, xc, cs, ntx); break;
  case 2: launch_tile<T, 2>(grid, block, lv, bl, b, x, xo, eta, nsweep, xc_in, bc, xc, cs, ntx); break;
  case 8: launch_tile<T, 8>(grid, block, lv, bl, b, x, xo, eta, nsweep, xc_in, bc, xc, cs, ntx); break;
  case 10: launch_tile<T, 10>(grid, block, lv, bl, b, x, xo, eta, nsweep, xc_in, bc, xc, cs, ntx); break;
  case 1: launch_tile<T, 1>(grid, block, lv, bl, b, x, xo, eta, nsweep, xc_in, bc, xc, cs, ntx); break;
  case 5: launch_tile<T, 5>(grid, block, lv, bl, b, x, xo, eta, nsweep, xc_in, bc, xc, cs, ntx); break;
  default: return (int)hipErrorInvalidValue;
  }
  return 0;
}
}  // extern "C++"

extern "C++" {
// grids smoothed whole in LDS: one thread per 2 x 2 block (1024 at most), the
// vector and the lent sums within 160 KB (64 x 64 in both precisions)
static bool afw_grid_fits(int prec, const mxh_level* lv)
{
  const long long N = (long long)lv->nx * lv->ny;
  return N <= 4096 && (prec == MXH_F64 ? 40 : 20) * N <= LDS_MAX && lv->nx >= 4 && lv->ny >= 4;
}

// Launches of few tiles: k_afw_few and the small tiles of k_node_tile.  Up to
// two tiles per compute unit they are the shorter launch (us, two sweeps and
// residual, FP64 edges / nodes, against the large tiles: 128^2 one vector 10 / 6
// against 17 / 10, four 16 / 8 against 19 / 11; 256^2 one 15 / 8 against 19 / 10,
// two 23 / 11 both; FP32 128^2 four 10 against 16), beyond they repeat
// the halo's work (384^2 one 30 / 13 against 25 / 12); callers that need k_afw_few's
// rounding ask for it (mode 16).  Edge grids of up to 32 x 32 nodes stay whole in
// LDS (32 vectors: 10 us against 14).
#define FEW_MAX 512
static bool few_fits(const mxh_level* lv, int nv)
{
  const long long t = (long long)((lv->nx + FEW_T - 1) / FEW_T) * ((lv->ny + FEW_T - 1) / FEW_T);
  return t * nv <= FEW_MAX;
}

template <typename T, int MODE>
static void launch_few(const mxh_level* lv, const mxh_bloch* bl, int nv, mxh_vecs b, mxh_vecs x, mxh_vecs xo,
                       const void* eta, int nsweep, mxh_vecs xc_in, mxh_vecs bc, mxh_vecs xc, long long cs)
{
  const int ntx = (lv->nx + FEW_T - 1) / FEW_T, nty = (lv->ny + FEW_T - 1) / FEW_T;
  hipLaunchKernelGGL((k_afw_few<T, MODE>), dim3(ntx * nty, nv), dim3(FEW_R * FEW_R / 4), 0, g_stream, *lv, *bl,
                     (const C<T>*)b.p, b.stride, (const C<T>*)x.p, (C<T>*)xo.p, x.stride, (const T*)eta, nsweep,
                     (const C<T>*)xc_in.p, (C<T>*)bc.p, (C<T>*)xc.p, cs, ntx);
}

template <typename T, int MODE>
static void launch_grid(const mxh_level* lv, const mxh_bloch* bl, int nv, mxh_vecs b, mxh_vecs x, mxh_vecs xo,
                        const void* eta, int nsweep, mxh_vecs xc_in, mxh_vecs bc, mxh_vecs xc, long long cs)
{
  const int N = lv->nx * lv->ny, blocks = N / 4;
  const size_t sh = sizeof(C<T>) * (2 * (size_t)N + ((MODE & 8) ? N / 2 : 0));
  auto go = [&](auto kernel, int threads) {
    hipLaunchKernelGGL(kernel, dim3(nv), dim3(threads), sh, g_stream, *lv, *bl, (const C<T>*)b.p, b.stride,
                       (const C<T>*)x.p, (C<T>*)xo.p, x.stride, (const T*)eta, nsweep, (const C<T>*)xc_in.p,
                       (C<T>*)bc.p, (C<T>*)xc.p, cs);
  };
  if (blocks <= 256) go(k_afw_grid<T, MODE, 256, 1>, (blocks + 63) / 64 * 64);
  else go(k_afw_grid<T, MODE, GridCfg<T>::TB, GridCfg<T>::NB>, GridCfg<T>::TB);
}

template <typename T>
static int launch_grid_mode(bool few, int mode, const mxh_level* lv, const mxh_bloch* bl, int nv, mxh_vecs b,
                            mxh_vecs x, mxh_vecs xo, const void* eta, int nsweep, mxh_vecs xc_in, mxh_vecs bc,
                            mxh_vecs xc)
{
  const long long cs = (mode & 8) ? bc.stride : (mode & 4) ? xc_in.stride : 0;
#define GRID_CASE(M)                                                            \
  case M:                                                                       \
    (few ? launch_few<T, M> : launch_grid<T, M>)(lv, bl, nv, b, x, xo, eta, nsweep, xc_in, bc, xc, cs); \
    break;
  switch (mode) {
    GRID_CASE(0)
    GRID_CASE(1)
    GRID_CASE(2)
    GRID_CASE(5)
    GRID_CASE(8)
    GRID_CASE(10)
  default: return (int)hipErrorInvalidValue;
  }
#undef GRID_CASE
  LAUNCH_CHECK();
  return 0;
}

template <typename T, int MODE>
static int grid_attr()
{
  const void* f[] = {(const void*)k_afw_grid<T, MODE, 256, 1>,
                     (const void*)k_afw_grid<T, MODE, GridCfg<T>::TB, GridCfg<T>::NB>};
  for (const void* q : f) {
    const hipError_t e = hipFuncSetAttribute(q, hipFuncAttributeMaxDynamicSharedMemorySize, LDS_MAX);
    if (e != hipSuccess) return (int)e;
  }
  return 0;
}

}  // extern "C++"
static int grid_attrs()
{
  return grid_attr<double, 0>() | grid_attr<double, 1>() | grid_attr<double, 2>() | grid_attr<double, 5>() |
         grid_attr<double, 8>() | grid_attr<double, 10>() | grid_attr<float, 0>() | grid_attr<float, 1>() |
         grid_attr<float, 2>() | grid_attr<float, 5>() | grid_attr<float, 8>() | grid_attr<float, 10>();
}
extern "C++" {
static bool cycle_levels(const mxh_cycle* cy, CycleLevels* cl)
{
  if (cy->n < 1 || cy->n > CYCLE_MAXL) return false;
  cl->n = cy->n;
  for (int l = 0; l < cy->n; l++) {
    const mxh_level* v = &cy->lv[l];
    if (v->nx < 2 || v->ny < 2 || (v->nx & 1) || (v->ny & 1)) return false;
    if (l && (v->nx != 2 * cy->lv[l - 1].nx || v->ny != 2 * cy->lv[l - 1].ny)) return false;
    cl->nx[l] = v->nx;
    cl->ny[l] = v->ny;
    cl->hx[l] = v->hx;
    cl->hy[l] = v->hy;
    cl->eta[l] = cy->eta[l];
    cl->b[l] = cy->b[l];
    cl->x[l] = cy->x[l];
    if ((cl->b[l] != nullptr) != (cl->x[l] != nullptr)) return false;
  }
  return cl->nx[cy->n - 1] * cl->ny[cy->n - 1] <= 1024;
}
// LDS of a cycle: x of all levels, b of the lower ones, the lent sums (or the
// coarsest b where it is the only level), 4 KB of partial sums
static size_t cycle_lds(int prec, const CycleLevels& cl, int comp)
{
  size_t tot = 0;
  const size_t top = (size_t)cl.nx[cl.n - 1] * cl.ny[cl.n - 1];
  for (int l = 0; l < cl.n; l++) tot += (size_t)comp * cl.nx[l] * cl.ny[l];
  const size_t lent = comp == 1 ? top : cl.n > 1 ? top / 2 : 2 * top;
  return csize(prec) * (2 * tot - comp * top + lent) + 16 * 256;
}
}  // extern "C++"

int mxh_cycle_supported(int prec, const mxh_cycle* cy)
{
  CycleLevels cl;
  return cycle_levels(cy, &cl) && 2 * cl.nx[0] * cl.ny[0] <= 256 && cycle_lds(prec, cl, 2) <= LDS_MAX;
}

int mxh_coarse_inverse(int n, int nprob, const double* L, double* W)
{
  if (n < 1 || n > 256 || nprob < 1) return (int)hipErrorInvalidValue;
  const dim3 grid(nprob, (n + 4 * INV_COLS - 1) / (4 * INV_COLS));
  auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(256), 0, g_stream, n, L, W); };
  if (n <= 64) go(k_coarse_inverse<1>);
  else if (n <= 128) go(k_coarse_inverse<2>);
  else go(k_coarse_inverse<4>);
  LAUNCH_CHECK();
  return 0;
}

int mxh_edge_cycle(int prec, const mxh_cycle* cy, const mxh_bloch* bl, int nv, int nu, mxh_vecs b, mxh_vecs x,
                   int xzero, const double* W, int per_problem)
{
  CycleLevels cl;
  if (!W || nu < 1 || nv < 1 || !mxh_cycle_supported(prec, cy) || !cycle_levels(cy, &cl))
    return (int)hipErrorInvalidValue;
  if (nv > 1 && cl.x[0]) return (int)hipErrorInvalidValue;  // lower levels are returned for one vector
  const int blocks = cl.nx[cl.n - 1] * cl.ny[cl.n - 1] / 4;
  const dim3 tb(blocks <= 64 ? 64 : blocks <= 128 ? 128 : 256);
  const size_t sh = cycle_lds(prec, cl, 2);
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_edge_cycle<double>, dim3(nv), tb, sh, g_stream, cl, *bl, nu, (const C<double>*)b.p, b.stride,
                       b.map, (C<double>*)x.p, x.stride, xzero, W, per_problem);
  else
    hipLaunchKernelGGL(k_edge_cycle<float>, dim3(nv), tb, sh, g_stream, cl, *bl, nu, (const C<float>*)b.p, b.stride,
                       b.map, (C<float>*)x.p, x.stride, xzero, W, per_problem);
  LAUNCH_CHECK();
  return 0;
}

int mxh_node_cycle(int prec, const mxh_cycle* cy, const mxh_bloch* bl, int nv, int nu, mxh_vecs b, mxh_vecs x,
                   int xzero, const double* W, int per_problem)
{
  CycleLevels cl;
  if (!W || nu < 1 || nv < 1 || !mxh_cycle_supported(prec, cy) || !cycle_levels(cy, &cl))
    return (int)hipErrorInvalidValue;
  if (nv > 1 && cl.x[0]) return (int)hipErrorInvalidValue;
  const int blocks = cl.nx[cl.n - 1] * cl.ny[cl.n - 1] / 4;
  const dim3 tb(blocks <= 64 ? 64 : blocks <= 128 ? 128 : 256);
  const size_t sh = cycle_lds(prec, cl, 1);
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_node_cycle<double>, dim3(nv), tb, sh, g_stream, cl, *bl, nu, (const C<double>*)b.p, b.stride,
                       (C<double>*)x.p, x.stride, xzero, W, per_problem);
  else
    hipLaunchKernelGGL(k_node_cycle<float>, dim3(nv), tb, sh, g_stream, cl, *bl, nu, (const C<float>*)b.p, b.stride,
                       (C<float>*)x.p, x.stride, xzero, W, per_problem);
  LAUNCH_CHECK();
  return 0;
}

int mxh_afw_tile(int prec, const mxh_level* lv, const mxh_bloch* bl, int nv, mxh_vecs b, mxh_vecs x, mxh_vecs xo,
                 const void* eta, int nsweep, int mode, mxh_vecs xc_in, mxh_vecs bc, mxh_vecs xc)
{
  if (!xo.p || xo.p == x.p || xo.stride != x.stride) return (int)hipErrorInvalidValue;
  if ((lv->nx & 1) || (lv->ny & 1) || nsweep < 1) return (int)hipErrorInvalidValue;
  const bool exact = mode & 16;
  mode &= ~16;
  if ((mode & 8) && (mode & 1)) return (int)hipErrorInvalidValue;
  // the halo must cover the sweeps (and the residual with its restriction)
  if (nsweep * ((mode & 1) ? TILE_SHRINK_BWD : TILE_SHRINK_FWD) + ((mode & 8) ? TILE_SHRINK_RES : 0) > TILE_H)
    return (int)hipErrorInvalidValue;
  if ((mode & 4) && !xc_in.p) return (int)hipErrorInvalidValue;
  if ((mode & 8) && (!bc.p || !xc.p || bc.stride != xc.stride)) return (int)hipErrorInvalidValue;
  const int R = prec == MXH_F64 ? TileCfg<double>::R : TileCfg<float>::R, TT = R - 2 * TILE_H;
  const int ntx = (lv->nx + TT - 1) / TT, nty = (lv->ny + TT - 1) / TT;
  const long long N = (long long)lv->nx * lv->ny;
  // small tiles, else the whole grid, else square tiles.  A whole FP64 grid near
  // 64 x 64 takes 28 us (two sweeps and residual) however few its vectors; while
  // the square tiles fill at most one workgroup per compute unit they are done
  // before (16 vectors 21 us, 24: 25; 32: 40).  Grids of 48 x 48 take 21 either way.
  bool few = N > 1024 && few_fits(lv, nv);
  const bool tiles = prec == MXH_F64 && N > 3072 && (long long)ntx * nty * nv <= mxh_cu_count();
  const bool whole = !few && afw_grid_fits(prec, lv) && (exact || !tiles);
  few |= exact && !whole;
  if (few || whole)
    return prec == MXH_F64 ? launch_grid_mode<double>(few, mode, lv, bl, nv, b, x, xo, eta, nsweep, xc_in, bc, xc)
                           : launch_grid_mode<float>(few, mode, lv, bl, nv, b, x, xo, eta, nsweep, xc_in, bc, xc);
  dim3 grid(ntx * nty, nv), block((R / 2) * (R / 2));
  long long cs = (mode & 8) ? bc.stride : (mode & 4) ? xc_in.stride : 0;
  int e = prec == MXH_F64
              ? launch_tile_mode<double>(mode, grid, block, lv, bl, b, x, xo, eta, nsweep, xc_in, bc, xc, cs, ntx)
              : launch_tile_mode<float>(mode, grid, block, lv, bl, b, x, xo, eta, nsweep, xc_in, bc, xc, cs, ntx);
  if (e) return e;
  LAUNCH_CHECK();
  return 0;
}

extern "C++" {
template <typename T, int MODE, int R>
static void launch_ntile(dim3 grid, const mxh_level* lv, const mxh_bloch* bl, mxh_vecs b, mxh_vecs x, mxh_vecs xo,
                         int nsweep, mxh_vecs xc_in, mxh_vecs bc, mxh_vecs xc, long long cs, int ntx)
{
  hipLaunchKernelGGL((k_node_tile<T, MODE, R>), grid, dim3(R * R / 4), 0, g_stream, *lv, *bl, (const C<T>*)b.p, b.stride,
                     (const C<T>*)x.p, (C<T>*)xo.p, x.stride, nsweep, (const C<T>*)xc_in.p, (C<T>*)bc.p,
                     (C<T>*)xc.p, cs, ntx);
}

template <typename T, int R>
static int launch_ntile_mode(int mode, dim3 grid, const mxh_level* lv, const mxh_bloch* bl, mxh_vecs b, mxh_vecs x,
                             mxh_vecs xo, int nsweep, mxh_vecs xc_in, mxh_vecs bc, mxh_vecs xc, long long cs, int ntx)
{
  switch (mode) {
  case 0: launch_ntile<T, 0, R>(grid, lv, bl, b, x, xo, nsweep, xc_in, bc, xc, cs, ntx); break;
  case 2: launch_ntile<T, 2, R>(grid, lv, bl, b, x, xo, nsweep, xc_in, bc, xc, cs, ntx); break;
  case 8: launch_ntile<T, 8, R>(grid, lv, bl, b, x, xo, nsweep, xc_in, bc, xc, cs, ntx); break;
  case 10: launch_ntile<T, 10, R>(grid, lv, bl, b, x, xo, nsweep, xc_in, bc, xc, cs, ntx); break;
  case 1: launch_ntile<T, 1, R>(grid, lv, bl, b, x, xo, nsweep, xc_in, bc, xc, cs, ntx); break;
  case 5: launch_ntile<T, 5, R>(grid, lv, bl, b, x, xo, nsweep, xc_in, bc, xc, cs, ntx); break;
  default: return (int)hipErrorInvalidValue;
  }
  return 0;
}
}  // extern "C++"

int mxh_node_tile(int prec, const mxh_level* lv, const mxh_bloch* bl, int nv, mxh_vecs b, mxh_vecs x, mxh_vecs xo,
                  int nsweep, int mode, mxh_vecs xc_in, mxh_vecs bc, mxh_vecs xc)
{
  if (!xo.p || xo.p == x.p || xo.stride != x.stride) return (int)hipErrorInvalidValue;
  if ((lv->nx & 1) || (lv->ny & 1) || nsweep < 1) return (int)hipErrorInvalidValue;
  if ((mode & 8) && (mode & 1)) return (int)hipErrorInvalidValue;
  // the halo must cover the sweeps (and the residual with its restriction);
  // backward sweeps are counted as the AFW's, which is conservative
  if (nsweep * ((mode & 1) ? TILE_SHRINK_BWD : TILE_SHRINK_FWD) + ((mode & 8) ? TILE_SHRINK_RES : 0) > TILE_H)
    return (int)hipErrorInvalidValue;
  if ((mode & 4) && !xc_in.p) return (int)hipErrorInvalidValue;
  if ((mode & 8) && (!bc.p || !xc.p || bc.stride != xc.stride)) return (int)hipErrorInvalidValue;
  const bool few = few_fits(lv, nv);
  const int TT = (few ? FEW_R : 64) - 2 * TILE_H;
  const int ntx = (lv->nx + TT - 1) / TT, nty = (lv->ny + TT - 1) / TT;
  dim3 grid(ntx * nty, nv);
  long long cs = (mode & 8) ? bc.stride : (mode & 4) ? xc_in.stride : 0;
  int e;
  if (few)
    e = prec == MXH_F64
            ? launch_ntile_mode<double, FEW_R>(mode, grid, lv, bl, b, x, xo, nsweep, xc_in, bc, xc, cs, ntx)
            : launch_ntile_mode<float, FEW_R>(mode, grid, lv, bl, b, x, xo, nsweep, xc_in, bc, xc, cs, ntx);
  else
    e = prec == MXH_F64 ? launch_ntile_mode<double, 64>(mode, grid, lv, bl, b, x, xo, nsweep, xc_in, bc, xc, cs, ntx)
                        : launch_ntile_mode<float, 64>(mode, grid, lv, bl, b, x, xo, nsweep, xc_in, bc, xc, cs, ntx);
  if (e) return e;
  LAUNCH_CHECK();
  return 0;
}

extern "C++" {
// region geometry of the marching kernels: owned W x Hgt, even, W + 2H <= MARCH_W
static void march_geometry(const mxh_level* lv, int rows, int H, int& ntx, int& nty, int& W, int& Hgt)
{
  const int wmax = MARCH_W - 2 * H;
  ntx = (lv->nx + wmax - 1) / wmax;
  W = (lv->nx + ntx - 1) / ntx;
  W += W & 1;
  if (rows < 2) rows = 128;
  nty = (lv->ny + rows - 1) / rows;
  Hgt = (lv->ny + nty - 1) / nty;
  Hgt += Hgt & 1;
}

extern "C" long long mxh_march_workgroups(const mxh_level* lv, int rows, int nsweep, int nv)
{
  int ntx, nty, W, Hgt;
  march_geometry(lv, rows, nsweep == 2 ? MarchCfg<2>::H : MarchCfg<1>::H, ntx, nty, W, Hgt);
  return (long long)ntx * nty * nv;
}

extern "C" int mxh_cu_count(void)
{
  static int cus = 0;
  if (!cus) {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0)
      cus = n;
    else
      return 256;
  }
  return cus;
}

template <typename T, int MODE, int NSW, bool NODE>
static void launch_march(dim3 grid, const mxh_level* lv, const mxh_bloch* bl, mxh_vecs b, mxh_vecs x, mxh_vecs xo,
                         const void* eta, mxh_vecs xc_in, mxh_vecs bc, mxh_vecs xc, long long cs, int ntx, int W,
                         int Hgt)
{
  if (NODE)
    hipLaunchKernelGGL((k_node_march<T, MODE, NSW>), grid, dim3(MarchCfg<NSW>::THREADS), 0, g_stream, *lv, *bl,
                       (const C<T>*)b.p, b.stride, (const C<T>*)x.p, (C<T>*)xo.p, x.stride, (const C<T>*)xc_in.p,
                       (C<T>*)bc.p, (C<T>*)xc.p, cs, ntx, W, Hgt);
  else
    hipLaunchKernelGGL((k_afw_march<T, MODE, NSW>), grid, dim3(MarchCfg<NSW>::THREADS), 0, g_stream, *lv, *bl,
                       (const C<T>*)b.p, b.stride, b.map, (const C<T>*)x.p, (C<T>*)xo.p, x.stride, (const T*)eta,
                       (const C<T>*)xc_in.p, (C<T>*)bc.p, (C<T>*)xc.p, cs, ntx, W, Hgt);
}

template <typename T, int NSW, bool NODE>
static int launch_march_mode(int mode, dim3 grid, const mxh_level* lv, const mxh_bloch* bl, mxh_vecs b, mxh_vecs x,
                             mxh_vecs xo, const void* eta, mxh_vecs xc_in, mxh_vecs bc, mxh_vecs xc, long long cs,
                             int ntx, int W, int Hgt)
{
#define MARCH_CASE(M)                                                                                      \
  case M:                                                                                                  \
    launch_march<T, M, NSW, NODE>(grid, lv, bl, b, x, xo, eta, xc_in, bc, xc, cs, ntx, W, Hgt);            \
    break;
  switch (mode) {
    MARCH_CASE(0)
    MARCH_CASE(2)
    MARCH_CASE(8)
    MARCH_CASE(10)
    MARCH_CASE(1)
    MARCH_CASE(5)
  default: return (int)hipErrorInvalidValue;
  }
#undef MARCH_CASE
  return 0;
}

template <bool NODE>
static int march_common(int prec, const mxh_level* lv, const mxh_bloch* bl, int nv, mxh_vecs b, mxh_vecs x,
                        mxh_vecs xo, const void* eta, int mode, mxh_vecs xc_in, mxh_vecs bc, mxh_vecs xc, int rows,
                        int nsweep)
{
  if (!xo.p || xo.p == x.p || xo.stride != x.stride) return (int)hipErrorInvalidValue;
  if (nsweep != 1 && nsweep != 2) return (int)hipErrorInvalidValue;
  // the halo wraps at most once: nx, ny >= H
  const int H = nsweep == 1 ? MarchCfg<1>::H : MarchCfg<2>::H;
  if ((lv->nx & 1) || (lv->ny & 1) || lv->nx < H || lv->ny < H) return (int)hipErrorInvalidValue;
  if ((mode & 8) && (mode & 1)) return (int)hipErrorInvalidValue;
  if ((mode & 4) && !xc_in.p) return (int)hipErrorInvalidValue;
  if ((mode & 8) && (!bc.p || !xc.p || bc.stride != xc.stride)) return (int)hipErrorInvalidValue;
  if (!NODE && !eta) return (int)hipErrorInvalidValue;
  int ntx, nty, W, Hgt;
  march_geometry(lv, rows, H, ntx, nty, W, Hgt);
  if (W + 2 * H > MARCH_W) return (int)hipErrorInvalidValue;
  // the last tile's region (tiles rounded up to even sizes) ends within one
  // period past the grid (very short tiles on a grid of about the halo's size
  // would not)
  if (ntx * W + H > 2 * lv->nx || nty * Hgt + H > 2 * lv->ny) return (int)hipErrorInvalidValue;
  dim3 grid(ntx * nty, nv);
  long long cs = (mode & 8) ? bc.stride : (mode & 4) ? xc_in.stride : 0;
  int e;
  if (nsweep == 1)
    e = prec == MXH_F64
            ? launch_march_mode<double, 1, NODE>(mode, grid, lv, bl, b, x, xo, eta, xc_in, bc, xc, cs, ntx, W, Hgt)
            : launch_march_mode<float, 1, NODE>(mode, grid, lv, bl, b, x, xo, eta, xc_in, bc, xc, cs, ntx, W, Hgt);
  else
    e = prec == MXH_F64
            ? launch_march_mode<double, 2, NODE>(mode, grid, lv, bl, b, x, xo, eta, xc_in, bc, xc, cs, ntx, W, Hgt)
            : launch_march_mode<float, 2, NODE>(mode, grid, lv, bl, b, x, xo, eta, xc_in, bc, xc, cs, ntx, W, Hgt);
  if (e) return e;
  LAUNCH_CHECK();
  return 0;
}
}  // extern "C++"

int mxh_afw_march(int prec, const mxh_level* lv, const mxh_bloch* bl, int nv, mxh_vecs b, mxh_vecs x, mxh_vecs xo,
                  const void* eta, int mode, mxh_vecs xc_in, mxh_vecs bc, mxh_vecs xc, int rows, int nsweep)
{
  return march_common<false>(prec, lv, bl, nv, b, x, xo, eta, mode, xc_in, bc, xc, rows, nsweep);
}

int mxh_node_march(int prec, const mxh_level* lv, const mxh_bloch* bl, int nv, mxh_vecs b, mxh_vecs x, mxh_vecs xo,
                   int mode, mxh_vecs xc_in, mxh_vecs bc, mxh_vecs xc, int rows, int nsweep)
{
  return march_common<true>(prec, lv, bl, nv, b, x, xo, nullptr, mode, xc_in, bc, xc, rows, nsweep);
}

int mxh_resid_restrict(int prec, const mxh_level* fine, const mxh_bloch* bl, int nv, mxh_vecs bf, mxh_vecs xf,
                       const void* eta_f, mxh_vecs bc, mxh_vecs xc)
{
  if ((fine->nx & 1) || (fine->ny & 1)) return (int)hipErrorInvalidValue;
  const long long NC = (long long)(fine->nx / 2) * (fine->ny / 2);
  dim3 grid(nblocks(NC), nv);
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_resid_restrict<double>, grid, dim3(TPB), 0, g_stream, *fine, *bl,
                       (const C<double>*)bf.p, bf.stride, (const C<double>*)xf.p, xf.stride,
                       (const double*)eta_f, (C<double>*)bc.p, bc.stride, (C<double>*)xc.p, xc.stride);
  else
    hipLaunchKernelGGL(k_resid_restrict<float>, grid, dim3(TPB), 0, g_stream, *fine, *bl,
                       (const C<float>*)bf.p, bf.stride, (const C<float>*)xf.p, xf.stride,
                       (const float*)eta_f, (C<float>*)bc.p, bc.stride, (C<float>*)xc.p, xc.stride);
  LAUNCH_CHECK();
  return 0;
}

int mxh_prolong(int prec, const mxh_level* fine, const mxh_bloch* bl, int nv, mxh_vecs c, mxh_vecs f,
                double alpha)
{
  if ((fine->nx & 1) || (fine->ny & 1)) return (int)hipErrorInvalidValue;
  const long long NC = (long long)(fine->nx / 2) * (fine->ny / 2);
  dim3 grid(nblocks(NC), nv);
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_prolong<double>, grid, dim3(TPB), 0, g_stream, *fine, *bl, (const C<double>*)c.p,
                       c.stride, (C<double>*)f.p, f.stride, alpha);
  else
    hipLaunchKernelGGL(k_prolong<float>, grid, dim3(TPB), 0, g_stream, *fine, *bl, (const C<float>*)c.p,
                       c.stride, (C<float>*)f.p, f.stride, (float)alpha);
  LAUNCH_CHECK();
  return 0;
}

int mxh_restrict(int prec, const mxh_level* fine, const mxh_bloch* bl, int nv, mxh_vecs f, mxh_vecs c,
                 double alpha)
{
  if ((fine->nx & 1) || (fine->ny & 1)) return (int)hipErrorInvalidValue;
  const long long NC = (long long)(fine->nx / 2) * (fine->ny / 2);
  dim3 grid(nblocks(NC), nv);
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_restrict<double>, grid, dim3(TPB), 0, g_stream, *fine, *bl, (const C<double>*)f.p,
                       f.stride, (C<double>*)c.p, c.stride, alpha);
  else
    hipLaunchKernelGGL(k_restrict<float>, grid, dim3(TPB), 0, g_stream, *fine, *bl, (const C<float>*)f.p,
                       f.stride, (C<float>*)c.p, c.stride, (float)alpha);
  LAUNCH_CHECK();
  return 0;
}

int mxh_coarse_setup(int n0, int nprob, const double* bloch, const double* eta0, double* Ae, double* An,
                     int* info)
{
  const int ne = 2 * n0 * n0, nn = n0 * n0;
  if (n0 < 1 || ne > MXH_COARSE_SETUP_MAX || nprob < 1) return (int)hipErrorInvalidValue;
  const size_t sh = sizeof(C<double>) * ((size_t)ne * ne + (size_t)nn * nn) + 8 * sizeof(double);
  hipLaunchKernelGGL(k_coarse_setup, dim3(nprob), dim3(TPB), sh, g_stream, n0, bloch, eta0, Ae, An, info);
  LAUNCH_CHECK();
  return 0;
}

int mxh_coarse_solve(int prec, int n, const double* L, const double* Lper, int vpp, const int* vmap, int nv,
                     mxh_vecs b, mxh_vecs x)
{
  if (n > TPB || n < 1) return (int)hipErrorInvalidValue;
  size_t sh = sizeof(double) * 2 * n;
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_coarse_solve<double>, dim3(nv), dim3(TPB), sh, g_stream, n, L, Lper, vpp, vmap,
                       (const C<double>*)b.p, b.stride, (C<double>*)x.p, x.stride);
  else
    hipLaunchKernelGGL(k_coarse_solve<float>, dim3(nv), dim3(TPB), sh, g_stream, n, L, Lper, vpp, vmap,
                       (const C<float>*)b.p, b.stride, (C<float>*)x.p, x.stride);
  LAUNCH_CHECK();
  return 0;
}

// Partial-sum sets of a Gram launch: bands * nprob <= GRAM_SETS, or nprob
// (one band per problem) when there are more problems than that.
#define GRAM_SETS 2048

size_t mxh_gram_work_bytes(int m, int nprob)
{
  const size_t sets = nprob > GRAM_SETS ? (size_t)nprob : GRAM_SETS;
  return sizeof(double) * 4 * (size_t)(m * (m + 1) / 2) * sets;
}

// A workgroup's time over r rows and q tiles with p tile pairs, in units of about
// 0.09 us: a strip's row costs its products and features, a strip its first loads,
// the workgroup the sums of its waves (fitted to 16^2 to 512^2, within about 15%).
static double gram_group_cost(const mxh_level* lv, int r, int p, int q)
{
  const int ns = (lv->nx + GRAM_STRIP - 1) / GRAM_STRIP;
  const double strips = ns < 4 ? ns : (ns + 3) / 4, rows = ns < 4 ? 0.25 * (r + 3) : r;
  if (p > 15) return strips * (rows * (2 * p + 2 * q) + 72.0) + 5.5 * p;  // (two passes)
  return strips * (rows * (2 * p + q) + 24.0) + 5.5 * p;
}

// The launch's time with wgs bands of r rows and the first f tiles in one workgroup:
// rounds of `slots` workgroups (one to four per compute unit, by the registers of the
// tiles' sums), those of the later tiles in the places that the last round leaves, then
// in rounds of their own.
static double gram_cost(const mxh_level* lv, int wgs, int nt, int f, int r, int slots)
{
  const int rounds = (wgs + slots - 1) / slots;
  const double c0 = gram_group_cost(lv, r, f * (f + 1) / 2, f), t = rounds * c0;
  if (f == nt) return t;
  const double c1 = gram_group_cost(lv, r, nt, nt), beside = (rounds - 1) * c0 + c1;
  const int left = wgs * (nt - f) - (rounds * slots - wgs) * (c0 > c1 ? (int)(c0 / c1) : 1);
  return (t > beside ? t : beside) + (left > 0 ? (left + slots - 1) / slots * c1 : 0.0);
}

// The Gram launch with at most max(sets_cap, nprob) partial-sum sets in work.
static int gram_launch(const mxh_level* lv, const mxh_bloch* bl, int nprob, const int* pmap, const int* cmap, int m,
                       mxh_vecs u, const double* eta64, double* out, void* work, int sets_cap)
{
  if (m < 1 || m > GRAM_MMAX || nprob < 1 || sets_cap < 1) return (int)hipErrorInvalidValue;
  const int np = m * (m + 1) / 2, nt = (m + 7) / 8;
  // Row bands: bands * nprob partial sets (sets_cap or nprob) fit the work
  // buffer.  Heights from the least that the buffer takes to twice that, or 64:
  // with 64 as the limit always, tall grids and many problems had one band a
  // problem (256 x 4096, 33 problems of 12 columns: 24.3 ms against 3.0).  Blocks of
  // more than three tiles run whole or with the tiles after the third (of six, after
  // the fifth) in workgroups of their own, which shortens the longest workgroup
  // where units would be idle, but loads the first tiles again: for a fifth (a
  // tenth) less by the model.  36 columns (us, whole and split): one problem of
  // 16^2 18.8 and 11.4, 72^2 26.0 and 18.1, 500 x 20 78 and 65; 16 problems of 16^2
  // 27.8 and 20.3, 64 x 256 120 and 170, 128^2 121 and 176.  48 columns (whole, after
  // the fifth, after the third): one problem of 16^2 37, 19, 12, seven of 72^2 75,
  // 58, 64, 16 of 512^2 2580, 2800, -.
  const int sets = nprob > sets_cap ? nprob : sets_cap;
  const int slots = mxh_cu_count() * (nt == 1 ? 4 : nt == 2 ? 2 : 1);
  const int most = sets / nprob, least = (lv->ny + most - 1) / most;
  int rpb = least, first = nt;
  double cost = -1.0;
  for (int f = nt; f > 0; f = f == 6 ? 5 : f > 3 ? 3 : 0)
    for (int r = least; r <= (least > 32 ? 2 * least : 64) && r <= lv->ny; r++) {
      const int wgs = (lv->ny + r - 1) / r * nprob;
      const double c = gram_cost(lv, wgs, nt, f, r, slots) * (f == nt ? 1.0 : f == 5 ? 1.1 : 1.25);
      if (cost < 0.0 || c < cost) {
        cost = c;
        first = f;
        rpb = r;
      }
      if (wgs * (nt - f + 1) <= slots) break;  // one round: higher bands only take longer
    }
  const int bands = (lv->ny + rpb - 1) / rpb;
  // The waves' sums in LDS, 256 of each tile pair: of the first tiles, at least as many
  // as a later tile's.  Six tiles whole take 128 of 21 pairs at a time, but a problem's
  // column list may fill five only.
  const int most5 = first < 5 ? first : 5;
  const size_t sh = 4 * sizeof(double) * 128 * (size_t)(most5 * (most5 + 1));
  const dim3 grid(bands, nprob, nt - first + 1);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(TPB), sh, g_stream, *lv, *bl, m, pmap, cmap, (const C<double>*)u.p, u.stride,
                       eta64, (double*)work, rpb);
  };
  switch (10 * nt + first) {
  case 11: go(k_gram<1, 1>); break;
  case 22: go(k_gram<2, 2>); break;
  case 33: go(k_gram<3, 3>); break;
  case 43: go(k_gram<4, 3>); break;
  case 44: go(k_gram<4, 4>); break;
  case 53: go(k_gram<5, 3>); break;
  case 55: go(k_gram<5, 5>); break;
  case 63: go(k_gram<6, 3>); break;
  case 65: go(k_gram<6, 5>); break;
  case 66: go(k_gram<6, 6>); break;
  }
  LAUNCH_CHECK();
  int width = 4 * np * nprob;
  hipLaunchKernelGGL(k_reduce_partials, dim3(reduce_blocks(width)), dim3(TPB), 0, g_stream, (const double*)work,
                     bands, width, out, 0);
  LAUNCH_CHECK();
  return 0;
}

int mxh_gram(const mxh_level* lv, const mxh_bloch* bl, int nprob, const int* pmap, int m, mxh_vecs u,
             const double* eta64, double* out, void* work)
{
  return gram_launch(lv, bl, nprob, pmap, nullptr, m, u, eta64, out, work, GRAM_SETS);
}

int mxh_gram_cols(const mxh_level* lv, const mxh_bloch* bl, int nprob, const int* pmap, const int* cmap, int m,
                  mxh_vecs u, const double* eta64, double* out, void* work)
{
  if (!cmap) return (int)hipErrorInvalidValue;
  return gram_launch(lv, bl, nprob, pmap, cmap, m, u, eta64, out, work, GRAM_SETS);
}

int mxh_gram_static(const mxh_level* lv, const mxh_bloch* bl, int nprob, const int* pmap, int m, mxh_vecs u,
                    const double* eta64, double* out)
{
  if (!g_stream || g_device < 0 || !g_scratch_ptr[g_device]) return (int)hipErrorNotInitialized;
  if (m < 1 || m > GRAM_MMAX || nprob < 1) return (int)hipErrorInvalidValue;
  // the partial-sum sets that fit the scratch array; every set the kernel
  // uses is written in full before the reduction reads it, so nothing needs
  // clearing between calls
  const size_t set_bytes = sizeof(double) * 4 * (size_t)(m * (m + 1) / 2);
  const size_t cap = MXH_GRAM_SCRATCH_BYTES / set_bytes;
  if ((size_t)nprob > cap) return MXH_ESCRATCH;
  const int sets_cap = cap < (size_t)GRAM_SETS ? (int)cap : GRAM_SETS;
  return gram_launch(lv, bl, nprob, pmap, nullptr, m, u, eta64, out, g_scratch_ptr[g_device], sets_cap);
}

int mxh_ritz(int m, int basis, int nprob, const int* pmap, const int* cmap, const double* gram, double sk,
             double pivot, double* Cm, double* lam, int vpp, int* status)
{
  const int k = basis ? basis : m;
  if (m < 1 || k < m || k > RITZ_MAX || nprob < 1) return (int)hipErrorInvalidValue;
  // threads: the items of a Jacobi round, k^2 / 4 blocks and k^2 / 2 rows, in at
  // most two goes
  hipLaunchKernelGGL(k_ritz, dim3(nprob), dim3(k <= 12 ? 128 : k <= 16 ? 256 : k <= 24 ? 512 : 1024),
                     3 * sizeof(C<double>) * (size_t)k * k, g_stream, m, basis, pmap, cmap, gram, sk, pivot, Cm, lam,
                     vpp, status);
  LAUNCH_CHECK();
  return 0;
}

int mxh_block_combine(long long n, int nprob, const int* pmap, int m, mxh_vecs u, mxh_vecs e, const double* Cm)
{
  if (m < 1 || m > COMB_MMAX || nprob < 1) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(k_block_combine, dim3(nblocks(n), nprob), dim3(TPB), 0, g_stream, n, m, pmap,
                     (const C<double>*)u.p, u.stride, (C<double>*)e.p, e.stride, Cm);
  LAUNCH_CHECK();
  return 0;
}

int mxh_combine_x(long long n, int nprob, const int* pmap, int nin, int nout, int nsplit, int gap, mxh_vecs x,
                  int xvpp, mxh_vecs y, int yvpp, const double* Cm)
{
  if (nin < 1 || nin > COMBX_NIN_MAX || nout < 1 || nout > 32 || nprob < 1 || nsplit < 0 || gap < 0)
    return (int)hipErrorInvalidValue;
  dim3 grid(nblocks(n), nprob);
  if (nout <= 16)
    hipLaunchKernelGGL(k_combine_x<16>, grid, dim3(TPB), 0, g_stream, n, nin, nout, nsplit, gap, pmap,
                       (const C<double>*)x.p, x.stride, xvpp, (C<double>*)y.p, y.stride, yvpp, Cm);
  else
    hipLaunchKernelGGL(k_combine_x<32>, grid, dim3(TPB), 0, g_stream, n, nin, nout, nsplit, gap, pmap,
                       (const C<double>*)x.p, x.stride, xvpp, (C<double>*)y.p, y.stride, yvpp, Cm);
  LAUNCH_CHECK();
  return 0;
}

int mxh_lobpcg_combine(long long n, int nprob, const int* pmap, int m, mxh_vecs x, mxh_vecs y, const double* Cm)
{
  if (m < 2 || m > 16 || (m & 1) || nprob < 1) return (int)hipErrorInvalidValue;
  dim3 grid(nblocks(n), nprob);
  if (m <= 8)
    hipLaunchKernelGGL(k_lobpcg_combine<8>, grid, dim3(TPB), 0, g_stream, n, m, pmap, (const C<double>*)x.p,
                       x.stride, (C<double>*)y.p, y.stride, Cm);
  else if (m <= 12)
    hipLaunchKernelGGL(k_lobpcg_combine<12>, grid, dim3(TPB), 0, g_stream, n, m, pmap, (const C<double>*)x.p,
                       x.stride, (C<double>*)y.p, y.stride, Cm);
  else
    hipLaunchKernelGGL(k_lobpcg_combine<16>, grid, dim3(TPB), 0, g_stream, n, m, pmap, (const C<double>*)x.p,
                       x.stride, (C<double>*)y.p, y.stride, Cm);
  LAUNCH_CHECK();
  return 0;
}

size_t mxh_orthonormalize_work_bytes(int k)
{
  // HhWork and a table of k vectors
  return sizeof(double) * ((6 + 2 * HH_NB + 4 * (size_t)k) * (size_t)k) + sizeof(void*) * (size_t)k;
}

static int hh_run(const mxh_level* lv, double xr, double xi, double yr, double yi, int k, HhVecs X, HhVecs V, double* work,
                  double* tau, double* host)
{
  const long long N = (long long)lv->nx * lv->ny;
  const HhWork wk = hh_work(work, k);
  C<double> xf, yf;
  xf.r = xr;
  xf.i = xi;
  yf.r = yr;
  yf.i = yi;
  const int nb = N < 256 * HH_NB ? (int)nblocks(N) : HH_NB;
  const int ub = max(nb, min(HH_NB, (k + 15) / 16));
  for (int i = 0; i < k; i++) {
    hipLaunchKernelGGL(k_hh_row, dim3(nb, k), dim3(256), 0, g_stream, *lv, xf, yf, i, X, wk);
    LAUNCH_CHECK();
    hipLaunchKernelGGL(k_hh_update, dim3(ub, k - i), dim3(256), 0, g_stream, *lv, i, k, nb, X, wk);
    LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(k_hh_coef, dim3(k <= HH_LDS ? 1 : (k + HH_COLS - 1) / HH_COLS), dim3(1024),
                     k <= HH_LDS ? 2 * sizeof(C<double>) * k * k : 0, g_stream, *lv, k, X, wk, tau, host);
  LAUNCH_CHECK();
  hipLaunchKernelGGL(k_hh_out, dim3(nblocks(2 * N, 64)), dim3(64), 0, g_stream, *lv, k, X, V, (const C<double>*)wk.W);
  LAUNCH_CHECK();
  return 0;
}

int mxh_orthonormalize(const mxh_level* lv, double xr, double xi, double yr, double yi, const double* eta64, int k,
                       double* X, double* V, double* tmp, double* tau, double* work)
{
  (void)eta64;  // M does not depend on it
  (void)tmp;
  if (k < 1 || lv->ny < 2 || (long long)k > (long long)lv->nx * (lv->ny / 2)) return (int)hipErrorInvalidValue;
  const long long n = 2LL * lv->nx * lv->ny;
  return hh_run(lv, xr, xi, yr, yi, k, HhVecs{(C<double>*)X, n, nullptr}, HhVecs{(C<double>*)V, n, nullptr},
                work, tau, nullptr);
}

int mxh_orthonormalize_vecs(const mxh_level* lv, double xr, double xi, double yr, double yi, int k, void* const* x,
                            double* tau, double* work)
{
  if (k < 1 || lv->ny < 2 || (long long)k > (long long)lv->nx * (lv->ny / 2)) return (int)hipErrorInvalidValue;
  const HhWork wk = hh_work(work, k);
  void* table = wk.W + 2 * (size_t)k * k;
  int e = (int)hipMemcpyAsync(table, x, sizeof(void*) * k, hipMemcpyHostToDevice, g_stream);
  if (e) return e;
  const HhVecs X{nullptr, 0, (C<double>* const*)table};
  return hh_run(lv, xr, xi, yr, yi, k, X, X, work, nullptr, tau);
}

int mxh_gather(int prec, long long n, int nv, mxh_vecs dst, mxh_vecs src)
{
  if (!src.map || nv < 1) return (int)hipErrorInvalidValue;
  dim3 grid(nblocks(n), nv);
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_gather<double>, grid, dim3(TPB), 0, g_stream, n, (C<double>*)dst.p, dst.stride,
                       (const C<double>*)src.p, src.stride, src.map);
  else
    hipLaunchKernelGGL(k_gather<float>, grid, dim3(TPB), 0, g_stream, n, (C<float>*)dst.p, dst.stride,
                       (const C<float>*)src.p, src.stride, src.map);
  LAUNCH_CHECK();
  return 0;
}

int mxh_node_addeval(int prec, const mxh_level* lv, const mxh_bloch* bl, int nv, mxh_vecs x, mxh_vecs y,
                     double ar, double ai, int accumulate)
{
  const long long N = (long long)lv->nx * lv->ny;
  dim3 grid(nblocks(N), nv);
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_node_addeval<double>, grid, dim3(TPB), 0, g_stream, *lv, *bl, (const C<double>*)x.p,
                       x.stride, (C<double>*)y.p, y.stride, ar, ai, accumulate);
  else
    hipLaunchKernelGGL(k_node_addeval<float>, grid, dim3(TPB), 0, g_stream, *lv, *bl, (const C<float>*)x.p,
                       x.stride, (C<float>*)y.p, y.stride, ar, ai, accumulate);
  LAUNCH_CHECK();
  return 0;
}

int mxh_node_gs_phase(int prec, const mxh_level* lv, const mxh_bloch* bl, int nv, mxh_vecs b, mxh_vecs x,
                      double alpha, int colour)
{
  if ((lv->nx & 1) || (lv->ny & 1)) return (int)hipErrorInvalidValue;
  const long long np = (long long)(lv->nx / 2) * (lv->ny / 2);
  dim3 grid(nblocks(np), nv);
  const int ci = colour & 1, cj = colour >> 1;
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_node_gs_phase<double>, grid, dim3(TPB), 0, g_stream, *lv, *bl, (const C<double>*)b.p,
                       b.stride, (C<double>*)x.p, x.stride, alpha, ci, cj);
  else
    hipLaunchKernelGGL(k_node_gs_phase<float>, grid, dim3(TPB), 0, g_stream, *lv, *bl, (const C<float>*)b.p,
                       b.stride, (C<float>*)x.p, x.stride, alpha, ci, cj);
  LAUNCH_CHECK();
  return 0;
}

int mxh_node_resid_restrict(int prec, const mxh_level* fine, const mxh_bloch* bl, int nv, mxh_vecs bf,
                            mxh_vecs xf, mxh_vecs bc, mxh_vecs xc)
{
  if ((fine->nx & 1) || (fine->ny & 1)) return (int)hipErrorInvalidValue;
  const long long NC = (long long)(fine->nx / 2) * (fine->ny / 2);
  dim3 grid(nblocks(NC), nv);
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_node_resid_restrict<double>, grid, dim3(TPB), 0, g_stream, *fine, *bl,
                       (const C<double>*)bf.p, bf.stride, (const C<double>*)xf.p, xf.stride, (C<double>*)bc.p,
                       bc.stride, (C<double>*)xc.p, xc.stride);
  else
    hipLaunchKernelGGL(k_node_resid_restrict<float>, grid, dim3(TPB), 0, g_stream, *fine, *bl,
                       (const C<float>*)bf.p, bf.stride, (const C<float>*)xf.p, xf.stride, (C<float>*)bc.p,
                       bc.stride, (C<float>*)xc.p, xc.stride);
  LAUNCH_CHECK();
  return 0;
}

int mxh_node_prolong(int prec, const mxh_level* fine, const mxh_bloch* bl, int nv, mxh_vecs c, mxh_vecs f,
                     double ar, double ai)
{
  if ((fine->nx & 1) || (fine->ny & 1)) return (int)hipErrorInvalidValue;
  const long long NC = (long long)(fine->nx / 2) * (fine->ny / 2);
  dim3 grid(nblocks(NC), nv);
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_node_prolong<double>, grid, dim3(TPB), 0, g_stream, *fine, *bl, (const C<double>*)c.p,
                       c.stride, (C<double>*)f.p, f.stride, ar, ai);
  else
    hipLaunchKernelGGL(k_node_prolong<float>, grid, dim3(TPB), 0, g_stream, *fine, *bl, (const C<float>*)c.p,
                       c.stride, (C<float>*)f.p, f.stride, ar, ai);
  LAUNCH_CHECK();
  return 0;
}

int mxh_node_restrict(int prec, const mxh_level* fine, const mxh_bloch* bl, int nv, mxh_vecs f, mxh_vecs c,
                      double ar, double ai)
{
  if ((fine->nx & 1) || (fine->ny & 1)) return (int)hipErrorInvalidValue;
  const long long NC = (long long)(fine->nx / 2) * (fine->ny / 2);
  dim3 grid(nblocks(NC), nv);
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_node_restrict<double>, grid, dim3(TPB), 0, g_stream, *fine, *bl, (const C<double>*)f.p,
                       f.stride, (C<double>*)c.p, c.stride, ar, ai);
  else
    hipLaunchKernelGGL(k_node_restrict<float>, grid, dim3(TPB), 0, g_stream, *fine, *bl, (const C<float>*)f.p,
                       f.stride, (C<float>*)c.p, c.stride, ar, ai);
  LAUNCH_CHECK();
  return 0;
}

// k_lift_rhs over the interior and the frame; with coef the plane-wave sums
// phi^H d per vector go to the returned place in work
static int lift_rhs_launch(int prec, const mxh_level* lv, const mxh_bloch* bl, int nv, mxh_vecs e, mxh_vecs x,
                           mxh_vecs u, mxh_vecs bg, mxh_vecs xg, const double* coef, double* work, double** csum)
{
  const unsigned nb = lift_blocks(lv->ny), nf = frame_blocks(lv);
  const dim3 grid(nb, nv), gridf(nf, nv);
  double* ph = coef ? work : nullptr;
  if (prec == MXH_F64) {
    hipLaunchKernelGGL((k_lift_rhs<double, false>), grid, dim3(TPB), 0, g_stream, *lv, *bl, (const C<double>*)e.p,
                       e.stride, e.map, (const C<double>*)x.p, x.stride, (C<double>*)u.p, u.stride, u.map,
                       (C<double>*)bg.p, bg.stride, (C<double>*)xg.p, xg.stride, ph, 0);
    hipLaunchKernelGGL((k_lift_rhs<double, true>), gridf, dim3(TPB), 0, g_stream, *lv, *bl, (const C<double>*)e.p,
                       e.stride, e.map, (const C<double>*)x.p, x.stride, (C<double>*)u.p, u.stride, u.map,
                       (C<double>*)bg.p, bg.stride, (C<double>*)xg.p, xg.stride, ph, (int)nb);
  } else {
    hipLaunchKernelGGL((k_lift_rhs<float, false>), grid, dim3(TPB), 0, g_stream, *lv, *bl, (const C<double>*)e.p,
                       e.stride, e.map, (const C<float>*)x.p, x.stride, (C<double>*)u.p, u.stride, u.map,
                       (C<float>*)bg.p, bg.stride, (C<float>*)xg.p, xg.stride, ph, 0);
    hipLaunchKernelGGL((k_lift_rhs<float, true>), gridf, dim3(TPB), 0, g_stream, *lv, *bl, (const C<double>*)e.p,
                       e.stride, e.map, (const C<float>*)x.p, x.stride, (C<double>*)u.p, u.stride, u.map,
                       (C<float>*)bg.p, bg.stride, (C<float>*)xg.p, xg.stride, ph, (int)nb);
  }
  LAUNCH_CHECK();
  if (coef) {
    *csum = work + (size_t)(nb + nf) * 2 * nv;
    hipLaunchKernelGGL(k_reduce_partials, dim3(reduce_blocks(2 * nv)), dim3(TPB), 0, g_stream, work, (int)(nb + nf),
                       2 * nv, *csum, 0);
    LAUNCH_CHECK();
  }
  return 0;
}

int mxh_lift_rhs(int prec, const mxh_level* lv, const mxh_bloch* bl, int nv, mxh_vecs e, mxh_vecs x,
                 mxh_vecs u, mxh_vecs bg, mxh_vecs xg, double* coef, double* work)
{
  if (x.p && u.p && u.p == e.p) return (int)hipErrorInvalidValue;
  if (coef && !work) return (int)hipErrorInvalidValue;
  double* csum = nullptr;
  const int err = lift_rhs_launch(prec, lv, bl, nv, e, x, u, bg, xg, coef, work, &csum);
  if (err) return err;
  if (coef) {
    dim3 g2(row_blocks(lv->ny), nv);
    if (prec == MXH_F64)
      hipLaunchKernelGGL(k_lift_deflate<double>, g2, dim3(TPB), 0, g_stream, *lv, *bl, (C<double>*)bg.p, bg.stride,
                         csum, coef);
    else
      hipLaunchKernelGGL(k_lift_deflate<float>, g2, dim3(TPB), 0, g_stream, *lv, *bl, (C<float>*)bg.p, bg.stride,
                         csum, coef);
    LAUNCH_CHECK();
  }
  return 0;
}

static int lift_apply_launch(int prec, const mxh_level* lv, const mxh_bloch* bl, int nv, mxh_vecs xg, mxh_vecs u,
                             mxh_vecs x, mxh_vecs e, double alpha, const double* coef, const double* pdot)
{
  dim3 grid(row_blocks(lv->ny), nv);
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_lift_apply<double>, grid, dim3(TPB), 0, g_stream, *lv, *bl, (const C<double>*)xg.p,
                       xg.stride, (const C<double>*)u.p, u.stride, u.map, (const C<double>*)x.p, x.stride,
                       (C<double>*)e.p, e.stride, e.map, alpha, coef, pdot);
  else
    hipLaunchKernelGGL(k_lift_apply<float>, grid, dim3(TPB), 0, g_stream, *lv, *bl, (const C<float>*)xg.p,
                       xg.stride, (const C<double>*)u.p, u.stride, u.map, (const C<float>*)x.p, x.stride,
                       (C<double>*)e.p, e.stride, e.map, alpha, coef, pdot);
  LAUNCH_CHECK();
  return 0;
}

int mxh_lift_apply(int prec, const mxh_level* lv, const mxh_bloch* bl, int nv, mxh_vecs xg, mxh_vecs u,
                   mxh_vecs x, mxh_vecs e, double alpha, const double* coef, double* work)
{
  if (coef && !work) return (int)hipErrorInvalidValue;
  const unsigned nb = row_blocks(lv->ny);
  double* pdot = nullptr;
  if (coef) {
    pdot = work + (size_t)nb * 2 * nv;
    if (prec == MXH_F64)
      hipLaunchKernelGGL(k_phi_dot<double>, dim3(nb, nv), dim3(TPB), 0, g_stream, *lv, *bl,
                         (const C<double>*)xg.p, xg.stride, work);
    else
      hipLaunchKernelGGL(k_phi_dot<float>, dim3(nb, nv), dim3(TPB), 0, g_stream, *lv, *bl, (const C<float>*)xg.p,
                         xg.stride, work);
    LAUNCH_CHECK();
    hipLaunchKernelGGL(k_reduce_partials, dim3(reduce_blocks(2 * nv)), dim3(TPB), 0, g_stream, work, (int)nb, 2 * nv,
                       pdot, 0);
    LAUNCH_CHECK();
  }
  return lift_apply_launch(prec, lv, bl, nv, xg, u, x, e, alpha, coef, pdot);
}

// Factor n = 2^a, 3 2^a or 5 2^a into stages, the odd radix first (every span
// is then a power of two).
static bool fft_plan(int n, FftPlan* p)
{
  if (n < 2) return false;
  p->n = n;
  p->ns = 0;
  int rest = n;
  auto push = [&](int r) {
    rest /= r;
    int lm = 0;
    while ((1 << lm) < rest) lm++;
    p->r[p->ns] = r;
    p->lm[p->ns++] = lm;
  };
  if (rest % 5 == 0) push(5);
  else if (rest % 3 == 0) push(3);
  if (rest & (rest - 1)) return false;
  while (rest > 1) push(rest % 8 == 0 && rest != 16 ? 8 : (rest % 4 == 0 ? 4 : 2));
  return p->ns <= FFT_MAXS;
}

// LDS of the one-launch solve: the vector, the phases and the mode terms
static size_t fft_solve_lds(int prec, const mxh_level* lv)
{
  const size_t c = csize(prec), s = (size_t)lv->nx + lv->ny;
  return c * ((size_t)lv->ny * (lv->nx | 1) + s) + c / 2 * s;
}
// columns per workgroup: 128-byte row segments, fewer where the columns are
// long (at least 32 bytes of a row; 0: columns too long for LDS)
static int fft_cols(int prec, const mxh_level* lv)
{
  const size_t c = csize(prec);
  int cb = (int)(128 / c);
  while (cb * c >= 32 && c * cb * lv->ny + c / 2 * (lv->ny + cb) > LDS_MAX) cb >>= 1;
  return cb * c >= 32 ? cb : 0;
}
// rows per workgroup: about 36 KB, so that four workgroups share a CU
static int fft_rows(int prec, const mxh_level* lv)
{
  int rb = 64;
  while (rb > 1 && (rb >= 2 * lv->ny || csize(prec) * rb * (size_t)(lv->nx | 1) > 36 * 1024)) rb >>= 1;
  return rb;
}

int mxh_lift_supported(int prec, const mxh_level* lv)
{
  FftPlan p;
  return fft_plan(lv->nx, &p) && fft_plan(lv->ny, &p) && fft_cols(prec, lv) > 0 &&
         csize(prec) * (2 * (size_t)lv->nx + 2) <= 64 * 1024;
}

int mxh_lift_launches(int prec, const mxh_level* lv) { return fft_solve_lds(prec, lv) <= LDS_MAX ? 6 : 8; }

size_t mxh_lift_table_bytes(int prec, const mxh_level* lv) { return csize(prec) * ((size_t)lv->nx + lv->ny); }

int mxh_lift_table(int prec, const mxh_level* lv, void* table)
{
  for (int k = 0; k < 2; k++) {
    const int n = k ? lv->ny : lv->nx;
    if (prec == MXH_F64)
      hipLaunchKernelGGL(k_fft_table<double>, dim3(nblocks(n)), dim3(TPB), 0, g_stream, n,
                         (C<double>*)table + (k ? lv->nx : 0));
    else
      hipLaunchKernelGGL(k_fft_table<float>, dim3(nblocks(n)), dim3(TPB), 0, g_stream, n,
                         (C<float>*)table + (k ? lv->nx : 0));
    LAUNCH_CHECK();
  }
  return 0;
}

extern "C++" {
template <typename T>
static int node_direct(int prec, const mxh_level* lv, const mxh_bloch* bl, int nv, mxh_vecs b, mxh_vecs x,
                       const C<T>* tw)
{
  FftPlan px, py;
  if (!fft_plan(lv->nx, &px) || !fft_plan(lv->ny, &py)) return (int)hipErrorInvalidValue;
  const C<T>*twx = tw, *twy = tw + lv->nx;
  const C<T>* B = (const C<T>*)b.p;
  C<T>* X = (C<T>*)x.p;
  const size_t one = fft_solve_lds(prec, lv);
  if (one <= LDS_MAX) {
    const long long N = (long long)lv->nx * lv->ny;
    hipLaunchKernelGGL(k_fft_solve<T>, dim3(nv), dim3(N >= 8192 ? 1024 : N >= 2048 ? 512 : 256), one, g_stream, *lv,
                       *bl, px, py, twx, twy, B, b.stride, X, x.stride);
    LAUNCH_CHECK();
    return 0;
  }
  const int RB = fft_rows(prec, lv), CB = fft_cols(prec, lv);
  const dim3 gr((lv->ny + RB - 1) / RB, nv), gc((lv->nx + CB - 1) / CB, nv);
  const size_t shr = sizeof(C<T>) * ((size_t)RB * (lv->nx | 1) + lv->nx + RB);
  const size_t shc = sizeof(C<T>) * (size_t)CB * lv->ny + sizeof(T) * (lv->ny + CB);
  const int tc = CB * lv->ny / 8, bc = tc >= 1024 ? 1024 : tc >= 512 ? 512 : 256;
  hipLaunchKernelGGL((k_fft_rows<T, -1>), gr, dim3(TPB), shr, g_stream, *lv, *bl, px, twx, B, b.stride, X, x.stride, RB);
  LAUNCH_CHECK();
  hipLaunchKernelGGL(k_fft_cols<T>, gc, dim3(bc), shc, g_stream, *lv, *bl, px, py, twy, X, x.stride, CB);
  LAUNCH_CHECK();
  hipLaunchKernelGGL((k_fft_rows<T, 1>), gr, dim3(TPB), shr, g_stream, *lv, *bl, px, twx, (const C<T>*)X, x.stride, X,
                     x.stride, RB);
  LAUNCH_CHECK();
  return 0;
}
}  // extern "C++"

int mxh_lift(int prec, const mxh_level* lv, const mxh_bloch* bl, int nv, mxh_vecs e, mxh_vecs x, mxh_vecs bg,
             mxh_vecs xg, mxh_vecs u, mxh_vecs out, double alpha, const void* table, double* coef, double* work)
{
  if (!table || !coef || !work || !bg.p || !xg.p || !mxh_lift_supported(prec, lv)) return (int)hipErrorInvalidValue;
  double* csum = nullptr;
  const mxh_vecs none = {nullptr, 0, nullptr};
  int err = lift_rhs_launch(prec, lv, bl, nv, e, x, none, bg, none, coef, work, &csum);
  if (err) return err;
  hipLaunchKernelGGL(k_lift_coef, dim3(nblocks(nv, 64)), dim3(64), 0, g_stream, *lv, *bl, nv, csum, coef);
  LAUNCH_CHECK();
  err = prec == MXH_F64 ? node_direct<double>(prec, lv, bl, nv, bg, xg, (const C<double>*)table)
                        : node_direct<float>(prec, lv, bl, nv, bg, xg, (const C<float>*)table);
  if (err) return err;
  return lift_apply_launch(prec, lv, bl, nv, xg, u, x, out, alpha, coef, nullptr);
}

int mxh_gradient(int prec, const mxh_level* lv, const mxh_bloch* bl, int nv, mxh_vecs v, mxh_vecs e, double ar,
                 double ai)
{
  const long long N = (long long)lv->nx * lv->ny;
  dim3 grid(nblocks(N), nv);
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_gradient<double>, grid, dim3(TPB), 0, g_stream, *lv, *bl, (const C<double>*)v.p,
                       v.stride, (C<double>*)e.p, e.stride, ar, ai);
  else
    hipLaunchKernelGGL(k_gradient<float>, grid, dim3(TPB), 0, g_stream, *lv, *bl, (const C<float>*)v.p, v.stride,
                       (C<float>*)e.p, e.stride, ar, ai);
  LAUNCH_CHECK();
  return 0;
}

int mxh_adjgradient(int prec, const mxh_level* lv, const mxh_bloch* bl, int nv, mxh_vecs e, mxh_vecs v,
                    double ar, double ai)
{
  const long long N = (long long)lv->nx * lv->ny;
  dim3 grid(nblocks(N), nv);
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_adjgradient<double>, grid, dim3(TPB), 0, g_stream, *lv, *bl, (const C<double>*)e.p,
                       e.stride, (C<double>*)v.p, v.stride, ar, ai);
  else
    hipLaunchKernelGGL(k_adjgradient<float>, grid, dim3(TPB), 0, g_stream, *lv, *bl, (const C<float>*)e.p,
                       e.stride, (C<float>*)v.p, v.stride, ar, ai);
  LAUNCH_CHECK();
  return 0;
}

int mxh_scale(int prec, long long n, int nv, mxh_vecs x, double ar, double ai)
{
  dim3 grid(nblocks(n), nv);
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_scale<double>, grid, dim3(TPB), 0, g_stream, n, (C<double>*)x.p, x.stride, ar, ai);
  else
    hipLaunchKernelGGL(k_scale<float>, grid, dim3(TPB), 0, g_stream, n, (C<float>*)x.p, x.stride, ar, ai);
  LAUNCH_CHECK();
  return 0;
}

int mxh_axpy(int prec, long long n, int nv, mxh_vecs x, mxh_vecs y, double ar, double ai)
{
  dim3 grid(nblocks(n), nv);
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_axpy<double>, grid, dim3(TPB), 0, g_stream, n, (const C<double>*)x.p, x.stride,
                       (C<double>*)y.p, y.stride, ar, ai);
  else
    hipLaunchKernelGGL(k_axpy<float>, grid, dim3(TPB), 0, g_stream, n, (const C<float>*)x.p, x.stride,
                       (C<float>*)y.p, y.stride, ar, ai);
  LAUNCH_CHECK();
  return 0;
}

int mxh_dot(int prec, long long n, int nv, mxh_vecs x, mxh_vecs y, double* out, double* work)
{
  unsigned nb = red_blocks(n);
  dim3 grid(nb, nv);
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_dot<double>, grid, dim3(TPB), 0, g_stream, n, (const C<double>*)x.p, x.stride,
                       (const C<double>*)y.p, y.stride, work);
  else
    hipLaunchKernelGGL(k_dot<float>, grid, dim3(TPB), 0, g_stream, n, (const C<float>*)x.p, x.stride,
                       (const C<float>*)y.p, y.stride, work);
  LAUNCH_CHECK();
  hipLaunchKernelGGL(k_reduce_partials, dim3(reduce_blocks(2 * nv)), dim3(TPB), 0, g_stream, work, (int)nb, 2 * nv, out,
                     0);
  LAUNCH_CHECK();
  return 0;
}

static unsigned product_blocks(long long n)
{
  const long long b = (n + PRODUCT_TB - 1) / PRODUCT_TB;
  // up to four entries a thread one workgroup needs no second sum
  return (unsigned)(b <= 4 ? 1 : b < PRODUCT_BLOCKS ? b : PRODUCT_BLOCKS);
}

int mxh_product_edge(const mxh_level* lv, const mxh_bloch* bl, const void* x, const void* y, const double* eta,
                     const mxh_coef* cf, double* work, double* out, double mark)
{
  const long long N = (long long)lv->nx * lv->ny;
  hipLaunchKernelGGL(k_product<1>, dim3(product_blocks(N)), dim3(PRODUCT_TB), 0, g_stream, *lv, *bl, 2 * N,
                     (const C<double>*)x, (const C<double>*)y, eta, *cf, work, out, mark);
  LAUNCH_CHECK();
  return 0;
}

int mxh_product(long long n, const void* x, const void* y, double* work, double* out, double mark)
{
  hipLaunchKernelGGL(k_product<0>, dim3(product_blocks(n)), dim3(PRODUCT_TB), 0, g_stream, mxh_level(), mxh_bloch(), n,
                     (const C<double>*)x, (const C<double>*)y, (const double*)nullptr, mxh_coef(), work, out, mark);
  LAUNCH_CHECK();
  return 0;
}

int mxh_product_wait(const double* out, double mark, double limit_us)
{
  const volatile double* m = out + 2;
  auto look = [&](int times) {
    for (int k = 0; k < times; k++) {
      if (*m == mark) {
        __atomic_thread_fence(__ATOMIC_ACQUIRE);
        return true;
      }
      __builtin_ia32_pause();
    }
    return false;
  };
  // most marks come within the first 1024 looks (about 18 us), which the clock
  // would make 0.8 us longer
  if (look(1024)) return 1;
  timespec t0, t;
  clock_gettime(CLOCK_MONOTONIC, &t0);
  do {
    if (look(64)) return 1;
    clock_gettime(CLOCK_MONOTONIC, &t);
  } while (1e6 * (double)(t.tv_sec - t0.tv_sec) + 1e-3 * (double)(t.tv_nsec - t0.tv_nsec) < limit_us);
  return 0;
}

int mxh_norm(int prec, long long n, int nv, mxh_vecs x, int kind, double* out, double* work)
{
  unsigned nb = red_blocks(n);
  dim3 grid(nb, nv);
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_norm<double>, grid, dim3(TPB), 0, g_stream, n, (const C<double>*)x.p, x.stride, kind,
                       work);
  else
    hipLaunchKernelGGL(k_norm<float>, grid, dim3(TPB), 0, g_stream, n, (const C<float>*)x.p, x.stride, kind,
                       work);
  LAUNCH_CHECK();
  hipLaunchKernelGGL(k_reduce_partials, dim3(reduce_blocks(nv)), dim3(TPB), 0, g_stream, work, (int)nb, nv, out,
                     kind == 0 ? 0 : 1);
  LAUNCH_CHECK();
  return 0;
}

int mxh_center(int prec, long long half, int nv, mxh_vecs x, double* work)
{
  unsigned nb = red_blocks(half);
  dim3 grid(nb, nv);
  double* sums = work + (size_t)nb * nv * 4;
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_halfsums<double>, grid, dim3(TPB), 0, g_stream, half, (const C<double>*)x.p, x.stride,
                       work);
  else
    hipLaunchKernelGGL(k_halfsums<float>, grid, dim3(TPB), 0, g_stream, half, (const C<float>*)x.p, x.stride,
                       work);
  LAUNCH_CHECK();
  hipLaunchKernelGGL(k_reduce_partials, dim3(reduce_blocks(4 * nv)), dim3(TPB), 0, g_stream, work, (int)nb, 4 * nv,
                     sums, 0);
  LAUNCH_CHECK();
  dim3 g2(nblocks(half), nv);
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_center_apply<double>, g2, dim3(TPB), 0, g_stream, half, (C<double>*)x.p, x.stride, sums);
  else
    hipLaunchKernelGGL(k_center_apply<float>, g2, dim3(TPB), 0, g_stream, half, (C<float>*)x.p, x.stride, sums);
  LAUNCH_CHECK();
  return 0;
}

int mxh_convert(int dprec, int sprec, long long n, int nv, mxh_vecs dst, mxh_vecs src)
{
  dim3 grid(nblocks(n), nv);
  if (dprec == MXH_F64 && sprec == MXH_F32)
    hipLaunchKernelGGL((k_convert<double, float>), grid, dim3(TPB), 0, g_stream, n, (C<double>*)dst.p, dst.stride,
                       (const C<float>*)src.p, src.stride);
  else if (dprec == MXH_F32 && sprec == MXH_F64)
    hipLaunchKernelGGL((k_convert<float, double>), grid, dim3(TPB), 0, g_stream, n, (C<float>*)dst.p, dst.stride,
                       (const C<double>*)src.p, src.stride);
  else if (dprec == MXH_F64)
    hipLaunchKernelGGL((k_convert<double, double>), grid, dim3(TPB), 0, g_stream, n, (C<double>*)dst.p,
                       dst.stride, (const C<double>*)src.p, src.stride);
  else
    hipLaunchKernelGGL((k_convert<float, float>), grid, dim3(TPB), 0, g_stream, n, (C<float>*)dst.p, dst.stride,
                       (const C<float>*)src.p, src.stride);
  LAUNCH_CHECK();
  return 0;
}

int mxh_random(int prec, long long n, int nv, mxh_vecs x, unsigned long long seed, int first_vector)
{
  dim3 grid(nblocks(n), nv);
  if (prec == MXH_F64)
    hipLaunchKernelGGL(k_random<double>, grid, dim3(TPB), 0, g_stream, n, (C<double>*)x.p, x.stride, seed,
                       first_vector);
  else
    hipLaunchKernelGGL(k_random<float>, grid, dim3(TPB), 0, g_stream, n, (C<float>*)x.p, x.stride, seed,
                       first_vector);
  LAUNCH_CHECK();
  return 0;
}

int mxh_curl2(const mxh_level* lv, const mxh_bloch* bl, int nv, mxh_vecs e, const double* w, double* grad)
{
  hipLaunchKernelGGL(k_eta_grad<true>, dim3(nblocks((long long)lv->nx * lv->ny)), dim3(TPB), 0, g_stream, *lv, *bl, nv,
                     (const C<double>*)e.p, e.stride, w, grad);
  LAUNCH_CHECK();
  return 0;
}

int mxh_eta_grad(const mxh_level* lv, const mxh_bloch* bl, int nv, mxh_vecs e, const double* gram, double* out)
{
  hipLaunchKernelGGL(k_eta_grad<false>, dim3(nblocks((long long)lv->nx * lv->ny)), dim3(TPB), 0, g_stream, *lv, *bl, nv,
                     (const C<double>*)e.p, e.stride, gram, out);
  LAUNCH_CHECK();
  return 0;
}

int mxh_event_create(void** ev)
{
  hipEvent_t e;
  hipError_t r = hipEventCreate(&e);
  *ev = (void*)e;
  return (int)r;
}

int mxh_event_record(void* ev) { return (int)hipEventRecord((hipEvent_t)ev, g_stream); }

int mxh_event_elapsed_ms(void* start, void* stop, float* ms)
{
  hipError_t r = hipEventSynchronize((hipEvent_t)stop);
  if (r != hipSuccess) return (int)r;
  return (int)hipEventElapsedTime(ms, (hipEvent_t)start, (hipEvent_t)stop);
}

int mxh_event_destroy(void* ev) { return (int)hipEventDestroy((hipEvent_t)ev); }

// Stream capture into a reusable graph.  Capture is thread-local, so other
// host threads keep launching eagerly on their own streams; everything the
// library enqueues on its stream between begin and end becomes a node.
int mxh_capture_begin(void) { return (int)hipStreamBeginCapture(g_stream, hipStreamCaptureModeThreadLocal); }

void mxh_capture_abort(void)
{
  hipGraph_t g = nullptr;
  if (hipStreamEndCapture(g_stream, &g) == hipSuccess && g) (void)hipGraphDestroy(g);
  (void)hipGetLastError();
}

int mxh_capture_end(void** exec)
{
  hipGraph_t g = nullptr;
  hipError_t e = hipStreamEndCapture(g_stream, &g);
  if (e != hipSuccess) return (int)e;
  if (*exec) {
    // same topology (one node per launch, same kernels), other launch
    // shapes or arguments: update the instantiated graph in place
    hipGraphNode_t bad = nullptr;
    hipGraphExecUpdateResult res = hipGraphExecUpdateError;
    if (hipGraphExecUpdate((hipGraphExec_t)*exec, g, &bad, &res) == hipSuccess && res == hipGraphExecUpdateSuccess) {
      (void)hipGraphDestroy(g);
      return 0;
    }
    (void)hipGetLastError();
    (void)hipGraphExecDestroy((hipGraphExec_t)*exec);
    *exec = nullptr;
  }
  hipGraphExec_t x = nullptr;
  e = hipGraphInstantiate(&x, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  if (e != hipSuccess) return (int)e;
  *exec = (void*)x;
  return 0;
}

int mxh_graph_launch(void* exec) { return (int)hipGraphLaunch((hipGraphExec_t)exec, g_stream); }

void mxh_graph_destroy(void* exec)
{
  if (exec) (void)hipGraphExecDestroy((hipGraphExec_t)exec);
}

}  // extern "C"
