// Design-side kernels: density and maximum-length-scale filters (Filter.cpp:21-150,
// RecMesh.cpp:544,706-718), the material interpolation with its SIMP / SIMP_CUT /
// SIMP_LOGISTIC branches and the filter chain rule (Material_Interpolation.cpp:20-187), and
// compliance sensitivities (Compliance.cpp:37-46).
//
// These are HBM-bound element loops.  They reproduce the reference's floating-point
// operation order exactly (file-wide fp contract(off): no fused multiply-add), so the filter
// weights, rho, E, dE/dz and the element sensitivities are bit-identical to a
// sequential non-FMA evaluation of the reference formulas.
#include "k_common.hpp"

#include <algorithm>
#include <cstdlib>
#include <type_traits>

// Keep every multiply and add separately rounded (no fused multiply-add) in this file.
#pragma clang fp contract(off)

namespace tofe {
namespace {

constexpr int NT = 256;
constexpr int kMaxTpl = 1024;

__device__ inline bool tpl_valid(const FilterTemplate &t, int ex, int ey, int ez, int q,
                                 const int *off, int &nb)
{
  const int i = ex + off[3 * q], j = ey + off[3 * q + 1], k = ez + off[3 * q + 2];
  if (i < 0 || i >= t.nx || j < 0 || j >= t.ny || k < 0 || k >= t.nz) return false;
  nb = i + t.nx * (j + t.ny * k);
  return true;
}

#define TOFE_STAGE_TEMPLATE()                                              \
  __shared__ int soff[3 * kMaxTpl];                                        \
  __shared__ double sw[kMaxTpl];                                           \
  for (int v = threadIdx.x; v < t.ntpl; v += NT) {                         \
    soff[3 * v] = t.off[3 * v];                                            \
    soff[3 * v + 1] = t.off[3 * v + 1];                                    \
    soff[3 * v + 2] = t.off[3 * v + 2];                                    \
    sw[v] = t.w[v];                                                        \
  }                                                                        \
  __syncthreads();

// inv_e = 1 / (sequential sum of the row's weights in ascending column order)
// (MatGetRowSum + VecPointwiseDivide, Filter.cpp:136-147)
__global__ __launch_bounds__(NT) void k_filter_inv(FilterTemplate t, double *inv, int64_t ne)
{
  TOFE_STAGE_TEMPLATE();
  const int64_t el = (int64_t)blockIdx.x * NT + threadIdx.x;
  if (el >= ne) return;
  const int ex = (int)(el % t.nx), ey = (int)((el / t.nx) % t.ny), ez = (int)(el / ((int64_t)t.nx * t.ny));
  double s = 0.0;
  for (int q = 0; q < t.ntpl; ++q) {
    int nb;
    if (tpl_valid(t, ex, ey, ez, q, soff, nb)) s = (s + sw[q]);
  }
  inv[el] = 1.0 / s;
}

// rho_e = sum_j P_ej x_j, P_ej = w_q * inv_e, ascending columns (MatMult, Material_Interpolation.cpp:35)
__global__ __launch_bounds__(NT) void k_filter_apply(FilterTemplate t, const double *__restrict__ inv,
                                                     const double *__restrict__ x, double *rho,
                                                     int64_t ne)
{
  TOFE_STAGE_TEMPLATE();
  const int64_t el = (int64_t)blockIdx.x * NT + threadIdx.x;
  if (el >= ne) return;
  const int ex = (int)(el % t.nx), ey = (int)((el / t.nx) % t.ny), ez = (int)(el / ((int64_t)t.nx * t.ny));
  const double ie = inv[el];
  double s = 0.0;
  for (int q = 0; q < t.ntpl; ++q) {
    int nb;
    if (tpl_valid(t, ex, ey, ez, q, soff, nb)) s = s + (sw[q] * ie) * x[nb];
  }
  rho[el] = s;
}

// gx_j = sum_i P_ij g_i over rows i = j - off_q in ascending order, i.e. the template
// walked backwards (MatMultTranspose, Material_Interpolation.cpp:159-162, 180).
__global__ __launch_bounds__(NT) void k_filter_apply_T(FilterTemplate t,
                                                       const double *__restrict__ inv,
                                                       const double *__restrict__ g, double *gx,
                                                       int64_t ne)
{
  TOFE_STAGE_TEMPLATE();
  const int64_t el = (int64_t)blockIdx.x * NT + threadIdx.x;
  if (el >= ne) return;
  const int ex = (int)(el % t.nx), ey = (int)((el / t.nx) % t.ny), ez = (int)(el / ((int64_t)t.nx * t.ny));
  double s = 0.0;
  for (int q = t.ntpl - 1; q >= 0; --q) {
    const int i = ex - soff[3 * q], j = ey - soff[3 * q + 1], k = ez - soff[3 * q + 2];
    if (i < 0 || i >= t.nx || j < 0 || j >= t.ny || k < 0 || k >= t.nz) continue;
    const int64_t row = i + (int64_t)t.nx * (j + (int64_t)t.ny * k);
    s = s + (sw[q] * inv[row]) * g[row];
  }
  gx[el] = s;
}

__global__ __launch_bounds__(NT) void k_filter_count(FilterTemplate t, int64_t *cnt, int64_t ne)
{
  TOFE_STAGE_TEMPLATE();
  const int64_t el = (int64_t)blockIdx.x * NT + threadIdx.x;
  if (el >= ne) return;
  const int ex = (int)(el % t.nx), ey = (int)((el / t.nx) % t.ny), ez = (int)(el / ((int64_t)t.nx * t.ny));
  int64_t c = 0;
  for (int q = 0; q < t.ntpl; ++q) {
    int nb;
    if (tpl_valid(t, ex, ey, ez, q, soff, nb)) ++c;
  }
  cnt[el] = c;
}

__global__ __launch_bounds__(NT) void k_filter_fill(FilterTemplate t, const double *__restrict__ inv,
                                                    const int64_t *__restrict__ rowptr,
                                                    int32_t *col, double *w, int64_t ne)
{
  TOFE_STAGE_TEMPLATE();
  const int64_t el = (int64_t)blockIdx.x * NT + threadIdx.x;
  if (el >= ne) return;
  const int ex = (int)(el % t.nx), ey = (int)((el / t.nx) % t.ny), ez = (int)(el / ((int64_t)t.nx * t.ny));
  const double ie = inv[el];
  int64_t p = rowptr[el];
  for (int q = 0; q < t.ntpl; ++q) {
    int nb;
    if (tpl_valid(t, ex, ey, ez, q, soff, nb)) {
      col[p] = nb;
      w[p] = (sw[q] * ie);
      ++p;
    }
  }
}

// VecPow with PETSc's special exponents; pow() otherwise.
__device__ inline double vecpow1(double x, double p)
{
  if (p == 1.0) return x;
  if (p == 0.0) return 1.0;
  if (p == -1.0) return 1.0 / x;
  if (p == 0.5) return sqrt(x);
  if (p == -0.5) return 1.0 / sqrt(x);
  if (p == 2.0) return (x * x);
  if (p == -2.0) return 1.0 / (x * x);
  return pow(x, p);
}

// z = (1 - rho)^q after rho = min(rho, 1), in place on rho (Material_Interpolation.cpp:42-45)
__global__ void k_void_pre(double *rho, int64_t ne, double q, double *zt)
{
  for (int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x; i < ne; i += (int64_t)gridDim.x * NT) {
    double r = rho[i];
    if (r > 1.0) r = 1.0;
    rho[i] = r;
    zt[i] = vecpow1(1.0 + -1 * r, q);
  }
}

// y = min(1, (REdge + R z) / vdMin), R with unit weights summed in ascending columns
// after REdge (MatMultAdd, VecScale(1/vdMin), VecPointwiseMin; Material_Interpolation.cpp:46-52)
__global__ __launch_bounds__(NT) void k_rfilter_madd(FilterTemplate t, const double *__restrict__ REdge,
                                                     const double *__restrict__ zt, double inv_vdmin,
                                                     double *y, int64_t ne)
{
  TOFE_STAGE_TEMPLATE();
  const int64_t el = (int64_t)blockIdx.x * NT + threadIdx.x;
  if (el >= ne) return;
  const int ex = (int)(el % t.nx), ey = (int)((el / t.nx) % t.ny), ez = (int)(el / ((int64_t)t.nx * t.ny));
  double s = REdge[el];
  for (int q = 0; q < t.ntpl; ++q) {
    int nb;
    if (tpl_valid(t, ex, ey, ez, q, soff, nb)) s = s + 1.0 * zt[nb];
  }
  s = s * inv_vdmin;
  y[el] = s < 1.0 ? s : 1.0;
}

// R^T g with unit weights: rows i = j - off_q in ascending order (template walked backwards)
__global__ __launch_bounds__(NT) void k_rfilter_T(FilterTemplate t, const double *__restrict__ g,
                                                  double *gx, int64_t ne)
{
  TOFE_STAGE_TEMPLATE();
  const int64_t el = (int64_t)blockIdx.x * NT + threadIdx.x;
  if (el >= ne) return;
  const int ex = (int)(el % t.nx), ey = (int)((el / t.nx) % t.ny), ez = (int)(el / ((int64_t)t.nx * t.ny));
  double s = 0.0;
  for (int q = t.ntpl - 1; q >= 0; --q) {
    const int i = ex - soff[3 * q], j = ey - soff[3 * q + 1], k = ez - soff[3 * q + 2];
    if (i < 0 || i >= t.nx || j < 0 || j >= t.ny || k < 0 || k >= t.nz) continue;
    s = s + 1.0 * g[i + (int64_t)t.nx * (j + (int64_t)t.ny * k)];
  }
  gx[el] = s;
}

// MatIntFnc after the filters (Material_Interpolation.cpp:54-116): rhoq = (q/vdMin)(1-rho)^(q-1);
// z = rho y; dEsdz = z^(p-1); Es = dEsdz z; dEsdz *= p; dEdz = (1-eps) dEsdz;
// E = eps + (1-eps) Es; then SIMP_CUT / SIMP_LOGISTIC modify Es and dEsdz only.
__device__ inline void simp_one(int64_t i, double r, double y, const SimpParams &sp,
                                const SimpOut &o)
{
  const double sc = sp.vd_penal / sp.vd_min;
  o.rhoq[i] = vecpow1(1.0 + -1 * r, sp.vd_penal - 1) * sc;
  const double z = r * y;
  double d = vecpow1(z, sp.penal - 1);
  double es = d * z;
  d = d * sp.penal;
  const double e = sp.eps + (1 - sp.eps) * es;
  o.dEdz[i] = d * (1 - sp.eps);
  o.E[i] = e;
  if (o.E32) o.E32[i] = (float)e;
  if (sp.interp == TOFE_INTERP_SIMP_CUT) {
    const double cut = (z > sp.p0) ? 1.0 : 0.0;
    es = es * cut;
    d = d * cut;
  } else if (sp.interp == TOFE_INTERP_SIMP_LOGISTIC) {
    const double denom = 1 + exp(sp.p0 * (sp.p1 - z));
    es = es / denom;
    d = (d + (es * sp.p0) * (1 - 1 / denom)) / denom;
  }
  o.Es[i] = es;
  o.dEsdz[i] = d;
}

// y_in == nullptr means the plain density filter (y = 1, written to o.y).
__global__ void k_simp(const double *__restrict__ rho, const double *y_in, int64_t ne,
                       SimpParams sp, SimpOut o)
{
  for (int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x; i < ne; i += (int64_t)gridDim.x * NT) {
    const double y = y_in ? y_in[i] : 1.0;
    if (!y_in) o.y[i] = 1.0;
    simp_one(i, rho[i], y, sp, o);
  }
}

// Chain_Filter middle step (Material_Interpolation.cpp:168-179):
// out = dfdE .* y - rhoq .* ((y < 1) .* RtT), RtT = R^T(dfdE .* rho)
__device__ inline double chain_mid_one(double g, double y, double rhoq, double rt)
{
  const double b = g * y;
  const double mask = (y < 1.0) ? 1.0 : 0.0;
  double a = rt * mask;
  a = rhoq * a;
  return b - a;
}

__global__ void k_chain_mid(const double *__restrict__ dfdE, const double *__restrict__ y,
                            const double *__restrict__ rhoq, const double *__restrict__ RtT,
                            double *out, int64_t ne)
{
  for (int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x; i < ne; i += (int64_t)gridDim.x * NT)
    out[i] = chain_mid_one(dfdE[i], y[i], rhoq[i], RtT[i]);
}

__global__ void k_mul(const double *__restrict__ a, const double *__restrict__ b, double *c, int64_t n)
{
  for (int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x; i < n; i += (int64_t)gridDim.x * NT)
    c[i] = a[i] * b[i];
}

// Filters with a radius of up to kFilterTileMax elements, tiled through LDS.
//
// A block of 512 threads forms a tile of 32 x 8 x (2 RZ) outputs from one staged box of the
// source, H elements wider on every side (zero outside the mesh: a zero term leaves a partial
// sum as it is, for the sums start at +0 or at a value >= 0).  Every thread then walks the
// neighbour list once, in its ascending order, for RZ outputs: one scalar load of the entry's
// LDS offset and weight serves the wavefront, and a term costs one LDS read (two in the
// transpose, which scales by the source's row sum) and its separately rounded operations, in
// place of three LDS reads, three bounds checks and a gather.  The transpose visits the rows
// e - off in ascending order; the neighbour list is symmetric with equal weights, so that is
// the same walk.  Bound: the LDS reads, 8 bytes a term, and the staging loads ahead of them; the
// 32-wide rows are read without bank conflicts, and z is the axis of the RZ outputs because their
// offsets are then immediates (H is a template argument for the same reason).  Measured on
// 144x72x72 elements, us, untiled -> here: R of radius 4.5 (389 entries) with the interpolation 260
// -> 56, R^T with the chain rule's middle 256 -> 56, P of radius 3.5 (179) 134 -> 34, P^T 160 ->
// 57; 192x96x96, radius 1.5 (19): P with the interpolation 57 -> 33 (its 149 MB of fields at 4.5
// TB/s), P^T 45 -> 16.  Reading rows of entries as 16-byte pairs for two outputs measured the same
// (R^T 54, P 39, P^T 63), as did four planes per thread.
constexpr int FTX = 32, FTY = 8, FNT = 512;
enum FiltMode : int { FM_APPLY = 0, FM_T = 1, FM_RADD = 2, FM_RT = 3 };
// FE_PLAIN: out; FE_SIMP: rho (or y) and the interpolation; FE_VOID: rho and z = (1 - rho)^q
enum FiltEpi : int { FE_PLAIN = 0, FE_SIMP = 1, FE_VOID = 2 };

struct FilterArgs {
  FilterTemplate t;
  const double *src = nullptr;  // x; g; z = (1 - rho)^q; dfdE
  const double *inv = nullptr;  // reciprocal row sums (FM_APPLY, FM_T)
  const double *add = nullptr;  // FM_RADD: REdge
  double scale = 0;             // FM_RADD: 1 / vdMin
  const double *rho = nullptr;  // FM_RADD with FE_SIMP; FM_RT: the factor of dfdE
  const double *y = nullptr, *rhoq = nullptr;  // FM_RT
  double *out = nullptr;        // rho; P^T g; y; the chain rule's middle step
  double *copy = nullptr;       // FM_APPLY: where x itself is kept (null: nowhere)
  double *zt = nullptr;         // FE_VOID
  SimpParams sp;
  SimpOut so;
};

// planes of outputs per thread: two, or one where two would not fit the LDS
constexpr int filter_rz(int H, int mode) { return (mode == FM_T && H >= 5) ? 1 : 2; }

template <int H, int MODE, int EPI>
__global__ __launch_bounds__(FNT) void k_filter_tile(FilterArgs a)
{
  constexpr int RZ = filter_rz(H, MODE);
  constexpr int PX = FTX + 2 * H, PY = FTY + 2 * H, PZ = 2 * RZ + 2 * H, PL = PX * PY;
  __shared__ double sv[PL * PZ];
  __shared__ double si[MODE == FM_T ? PL * PZ : 1];
  const int nx = a.t.nx, ny = a.t.ny, nz = a.t.nz;
  const int bx = blockIdx.x * FTX, by = blockIdx.y * FTY, bz = blockIdx.z * (2 * RZ);
  // every load of the box is issued before the first value is used, without a branch (an element
  // outside the mesh reads element 0): waiting for them one by one cost R^T 6 of 64 us
  constexpr int NL = (PL * PZ + FNT - 1) / FNT;
  static_assert(NL <= 32, "one bit per staged element of a thread");
  double xv[NL], xi[MODE == FM_T || MODE == FM_RT ? NL : 1];
  unsigned inside = 0;
#pragma unroll
  for (int k = 0; k < NL; ++k) {
    const int v = (int)threadIdx.x + k * FNT;
    const int lz = v / PL, r = v - lz * PL, ly = r / PX, lx = r - ly * PX;
    const int gx = bx - H + lx, gy = by - H + ly, gz = bz - H + lz;
    const bool in = gx >= 0 && gx < nx && gy >= 0 && gy < ny && gz >= 0 && gz < nz && v < PL * PZ;
    const int n = in ? gx + nx * (gy + ny * gz) : 0;
    inside |= (in ? 1u : 0u) << k;
    xv[k] = a.src[n];
    if constexpr (MODE == FM_T) xi[k] = a.inv[n];
    if constexpr (MODE == FM_RT) xi[k] = a.rho[n];
  }
#pragma unroll
  for (int k = 0; k < NL; ++k) {
    const int v = (int)threadIdx.x + k * FNT;
    const bool in = (inside >> k) & 1u;
    if constexpr (MODE == FM_RT) xv[k] = xv[k] * xi[k];
    if (v < PL * PZ) {
      sv[v] = in ? xv[k] : 0.0;
      if constexpr (MODE == FM_T) si[v] = in ? xi[k] : 0.0;
    }
  }
  __syncthreads();
  const int tx = threadIdx.x % FTX, ty = (threadIdx.x / FTX) % FTY, tz = threadIdx.x / (FTX * FTY);
  const int gx = bx + tx, gy = by + ty, z0 = bz + tz * RZ;
  if (gx >= nx || gy >= ny || z0 >= nz) return;
  const int base = (tz * RZ * PY + ty) * PX + tx;  // the box corner of the first output
  int64_t el[RZ];
  double s[RZ], ie[RZ];
#pragma unroll
  for (int r = 0; r < RZ; ++r) {
    el[r] = gx + (int64_t)nx * (gy + (int64_t)ny * min(z0 + r, nz - 1));
    s[r] = 0.0;
    ie[r] = 0.0;
    if constexpr (MODE == FM_APPLY) ie[r] = a.inv[el[r]];
    if constexpr (MODE == FM_RADD) s[r] = a.add[el[r]];
  }
  const int *__restrict__ off = a.t.tile_off;
  const double *__restrict__ w = a.t.w;
#pragma unroll 8
  for (int q = 0; q < a.t.ntpl; ++q) {
    const double *p = sv + base + off[q];
    const double wq = (MODE == FM_APPLY || MODE == FM_T) ? w[q] : 1.0;
#pragma unroll
    for (int r = 0; r < RZ; ++r) {
      const double x = p[r * PL];
      if constexpr (MODE == FM_APPLY) s[r] = s[r] + (wq * ie[r]) * x;
      else if constexpr (MODE == FM_T) s[r] = s[r] + (wq * si[base + off[q] + r * PL]) * x;
      else s[r] = s[r] + x;
    }
  }
#pragma unroll 1
  for (int r = 0; r < RZ; ++r) {
    if (z0 + r >= nz) break;
    const int64_t e = gx + (int64_t)nx * (gy + (int64_t)ny * (z0 + r));
    double v = r ? s[RZ - 1] : s[0];
    if constexpr (MODE == FM_APPLY) {
      if (a.copy) a.copy[e] = sv[base + (H * PY + H) * PX + H + r * PL];
      if constexpr (EPI == FE_VOID) {  // as k_void_pre
        if (v > 1.0) v = 1.0;
        a.zt[e] = vecpow1(1.0 + -1 * v, a.sp.vd_penal);
      }
      a.out[e] = v;
      if constexpr (EPI == FE_SIMP) {
        a.so.y[e] = 1.0;
        simp_one(e, v, 1.0, a.sp, a.so);
      }
    } else if constexpr (MODE == FM_RADD) {
      v = v * a.scale;
      const double y = v < 1.0 ? v : 1.0;
      a.out[e] = y;
      simp_one(e, a.rho[e], y, a.sp, a.so);
    } else if constexpr (MODE == FM_RT) {
      a.out[e] = chain_mid_one(a.src[e], a.y[e], a.rhoq[e], v);
    } else {
      a.out[e] = v;
    }
  }
}

// g_e = -dEdz_e * u_e^T (KE u_e), sequential sums without contraction (Compliance.cpp:37-43)
__global__ __launch_bounds__(NT) void k_sensitivity(const double *__restrict__ U,
                                                    const double *__restrict__ dEdz,
                                                    const double *__restrict__ KE, int nx, int ny,
                                                    int nz, double *g)
{
  const int64_t ne = (int64_t)nx * ny * nz;
  const int64_t el = (int64_t)blockIdx.x * NT + threadIdx.x;
  if (el >= ne) return;
  const int ex = (int)(el % nx), ey = (int)((el / nx) % ny), ez = (int)(el / ((int64_t)nx * ny));
  const int Nx = nx + 1, Ny = ny + 1;
  double u[24];
#pragma unroll
  for (int l = 0; l < 8; ++l) {
    const int64_t n = (ex + lnx(l)) + (int64_t)Nx * ((ey + lny(l)) + (int64_t)Ny * (ez + lnz(l)));
#pragma unroll
    for (int c = 0; c < 3; ++c) u[3 * l + c] = U[3 * n + c];
  }
  double s = 0.0;
#pragma unroll
  for (int r = 0; r < 24; ++r) {
    double tr = 0.0;
#pragma unroll
    for (int c = 0; c < 24; ++c) tr = tr + KE[r * 24 + c] * u[c];
    s = s + u[r] * tr;
  }
  g[el] = (-dEdz[el] * s);
}

// Lumped mass diagonal (Frequency::DiagMassFnc, Dynamic.cpp:181-236): the element blocks
// V_e m0 I are added in ascending element order, then the lumped point masses
// (MatDiagonalSet ADD_VALUES, 233); Dirichlet DOFs get 1e-8 (MatZeroRowsColumns, 44-45).
__global__ __launch_bounds__(NT) void k_mass_diag(const double *__restrict__ V, int nx, int ny,
                                                  int nz, double m0, const double *__restrict__ mlump,
                                                  const uint8_t *__restrict__ fix, double *M)
{
  const int Nx = nx + 1, Ny = ny + 1, Nz = nz + 1;
  const int64_t nn = (int64_t)Nx * Ny * Nz;
  const int64_t n = (int64_t)blockIdx.x * NT + threadIdx.x;
  if (n >= nn) return;
  int i, j, k;
  node_ijk(n, Nx, Ny, i, j, k);
  double s = 0.0;
  for (int dz = -1; dz <= 0; ++dz)
    for (int dy = -1; dy <= 0; ++dy)
      for (int dx = -1; dx <= 0; ++dx) {
        const int ex = i + dx, ey = j + dy, ez = k + dz;
        if (ex < 0 || ex >= nx || ey < 0 || ey >= ny || ez < 0 || ez >= nz) continue;
        s = s + V[ex + (int64_t)nx * (ey + (int64_t)ny * ez)] * m0;
      }
  const uint8_t fm = fix ? fix[n] : 0;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    double v = mlump ? s + mlump[3 * n + c] : s;
    if ((fm >> c) & 1) v = 1e-8;
    M[3 * n + c] = v;
  }
}

__global__ void k_diag_mul(const double *__restrict__ d, const double *__restrict__ x, double *y,
                           int64_t n, int nrhs)
{
  const int64_t tot = n * nrhs;
  for (int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x; i < tot; i += (int64_t)gridDim.x * NT)
    y[i] = d[i % n] * x[i];
}

// Element quadratic forms of nvec vectors (the element terms of the eigenvalue
// sensitivities, Dynamic.cpp:113-154): kq = phi_e^T KE phi_e, mq = sum over the element's
// 24 DOFs of phi^2.  One thread per (element, vector).
// Consistent element mass over m0 = elemSize * density / 24 (the lumped matrix's per-DOF
// element mass): Q (x) I_3 with Q_ab = 24 prod_d (a_d == b_d ? 1/3 : 1/6) for element-local
// nodes a, b (the exact integral of N_a N_b over the box element, over elemSize / 24).
__device__ inline double mass_q(int a, int b)
{
  const int same = (lnx(a) == lnx(b)) + (lny(a) == lny(b)) + (lnz(a) == lnz(b));
  // 24 / 216 * 2^same
  return same == 3 ? 8.0 / 9.0 : same == 2 ? 4.0 / 9.0 : same == 1 ? 2.0 / 9.0 : 1.0 / 9.0;
}

__global__ __launch_bounds__(NT) void k_elem_quad(const double *__restrict__ phi,
                                                  const double *__restrict__ KE, int nx, int ny,
                                                  int nz, int64_t ndof, int nvec, double *kq,
                                                  double *mq, int consistent)
{
  const int64_t ne = (int64_t)nx * ny * nz;
  const int64_t t = (int64_t)blockIdx.x * NT + threadIdx.x;
  if (t >= ne * nvec) return;
  const int64_t el = t % ne;
  const int v = (int)(t / ne);
  const double *U = phi + (int64_t)v * ndof;
  const int ex = (int)(el % nx), ey = (int)((el / nx) % ny), ez = (int)(el / ((int64_t)nx * ny));
  const int Nx = nx + 1, Ny = ny + 1;
  double u[24];
#pragma unroll
  for (int l = 0; l < 8; ++l) {
    const int64_t n = (ex + lnx(l)) + (int64_t)Nx * ((ey + lny(l)) + (int64_t)Ny * (ez + lnz(l)));
#pragma unroll
    for (int c = 0; c < 3; ++c) u[3 * l + c] = U[3 * n + c];
  }
  double s = 0.0, m = 0.0;
#pragma unroll
  for (int r = 0; r < 24; ++r) {
    double tr = 0.0;
#pragma unroll
    for (int c = 0; c < 24; ++c) tr = tr + KE[r * 24 + c] * u[c];
    s = s + u[r] * tr;
    m = m + u[r] * u[r];
  }
  kq[t] = s;
  if (mq && consistent) {  // phi_e^T (Q (x) I_3) phi_e
    m = 0.0;
#pragma unroll
    for (int a = 0; a < 8; ++a)
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        const double w = mass_q(a, b);
#pragma unroll
        for (int c = 0; c < 3; ++c) m += w * u[3 * a + c] * u[3 * b + c];
      }
  }
  if (mq) mq[t] = m;
}

inline unsigned blocks_for(int64_t n) { return (unsigned)((n + NT - 1) / NT); }

}  // namespace

void filter_rowsum_inv(hipStream_t s, const FilterTemplate &t, double *inv)
{
  const int64_t ne = (int64_t)t.nx * t.ny * t.nz;
  k_filter_inv<<<dim3(blocks_for(ne)), dim3(NT), 0, s>>>(t, inv, ne);
  TOFE_LAUNCH_CHECK();
}

template <int MODE, int EPI>
static bool filter_tile(hipStream_t s, const FilterArgs &a)
{
  const auto go = [&](auto hc) {
    constexpr int H = decltype(hc)::value;
    constexpr int TZ = 2 * filter_rz(H, MODE);
    const dim3 grid((a.t.nx + FTX - 1) / FTX, (a.t.ny + FTY - 1) / FTY, (a.t.nz + TZ - 1) / TZ);
    if (grid.y > 65535 || grid.z > 65535) return false;
    k_filter_tile<H, MODE, EPI><<<grid, dim3(FNT), 0, s>>>(a);
    TOFE_LAUNCH_CHECK();
    return true;
  };
  switch (a.t.tile_h) {
    case 1: return go(std::integral_constant<int, 1>());
    case 2: return go(std::integral_constant<int, 2>());
    case 3: return go(std::integral_constant<int, 3>());
    case 4: return go(std::integral_constant<int, 4>());
    case 5: return go(std::integral_constant<int, 5>());
    default: return false;
  }
}

// The tiled kernels serve every filter whose neighbours lie within kFilterTileMax elements
// (LDS holds the staged box); the ones above walk larger neighbourhoods from global memory.
int filter_tile_h(const int *off, int n)
{
  int h = 1;
  for (int v = 0; v < 3 * n; ++v) h = std::max(h, std::abs(off[v]));
  return h <= kFilterTileMax ? h : 0;
}

void filter_tile_offsets(const int *off, int n, int h, int *out)
{
  const int px = FTX + 2 * h, py = FTY + 2 * h;
  for (int q = 0; q < n; ++q)
    out[q] = ((off[3 * q + 2] + h) * py + off[3 * q + 1] + h) * px + off[3 * q] + h;
}

void filter_apply(hipStream_t s, const FilterTemplate &t, const double *inv, const double *x,
                  double *rho)
{
  FilterArgs a;
  a.t = t;
  a.src = x;
  a.inv = inv;
  a.out = rho;
  if (filter_tile<FM_APPLY, FE_PLAIN>(s, a)) return;
  const int64_t ne = (int64_t)t.nx * t.ny * t.nz;
  k_filter_apply<<<dim3(blocks_for(ne)), dim3(NT), 0, s>>>(t, inv, x, rho, ne);
  TOFE_LAUNCH_CHECK();
}

void filter_apply_T(hipStream_t s, const FilterTemplate &t, const double *inv, const double *g,
                    double *gx)
{
  FilterArgs a;
  a.t = t;
  a.src = g;
  a.inv = inv;
  a.out = gx;
  if (filter_tile<FM_T, FE_PLAIN>(s, a)) return;
  const int64_t ne = (int64_t)t.nx * t.ny * t.nz;
  k_filter_apply_T<<<dim3(blocks_for(ne)), dim3(NT), 0, s>>>(t, inv, g, gx, ne);
  TOFE_LAUNCH_CHECK();
}

void filter_count(hipStream_t s, const FilterTemplate &t, int64_t *cnt)
{
  const int64_t ne = (int64_t)t.nx * t.ny * t.nz;
  k_filter_count<<<dim3(blocks_for(ne)), dim3(NT), 0, s>>>(t, cnt, ne);
  TOFE_LAUNCH_CHECK();
}

void filter_fill(hipStream_t s, const FilterTemplate &t, const double *inv, const int64_t *rowptr,
                 int32_t *col, double *w)
{
  const int64_t ne = (int64_t)t.nx * t.ny * t.nz;
  k_filter_fill<<<dim3(blocks_for(ne)), dim3(NT), 0, s>>>(t, inv, rowptr, col, w, ne);
  TOFE_LAUNCH_CHECK();
}

static unsigned stride_blocks(int64_t n)
{
  unsigned nb = blocks_for(n);
  return nb > 4096 ? 4096 : (nb ? nb : 1);
}

void design_fields(hipStream_t s, const FilterTemplate &t, const double *inv, const double *x,
                   double *xcopy, double *rho, const SimpParams &sp, const SimpOut &so)
{
  const int64_t ne = (int64_t)t.nx * t.ny * t.nz;
  FilterArgs a;
  a.t = t;
  a.src = x;
  a.inv = inv;
  a.out = rho;
  a.copy = xcopy;
  a.sp = sp;
  a.so = so;
  if (filter_tile<FM_APPLY, FE_SIMP>(s, a)) return;
  if (xcopy) TOFE_HIP(hipMemcpyAsync(xcopy, x, ne * sizeof(double), hipMemcpyDeviceToDevice, s));
  filter_apply(s, t, inv, x, rho);
  k_simp<<<dim3(stride_blocks(ne)), dim3(NT), 0, s>>>(rho, nullptr, ne, sp, so);
  TOFE_LAUNCH_CHECK();
}

void design_fields_void(hipStream_t s, const FilterTemplate &t, const FilterTemplate &tr,
                        const double *inv, const double *REdge, const double *x, double *xcopy,
                        double *rho, double *zt, const SimpParams &sp, const SimpOut &so)
{
  const int64_t ne = (int64_t)t.nx * t.ny * t.nz;
  FilterArgs a;
  a.t = t;
  a.src = x;
  a.inv = inv;
  a.out = rho;
  a.copy = xcopy;
  a.zt = zt;
  a.sp = sp;
  if (!filter_tile<FM_APPLY, FE_VOID>(s, a)) {
    if (xcopy) TOFE_HIP(hipMemcpyAsync(xcopy, x, ne * sizeof(double), hipMemcpyDeviceToDevice, s));
    filter_apply(s, t, inv, x, rho);
    k_void_pre<<<dim3(stride_blocks(ne)), dim3(NT), 0, s>>>(rho, ne, sp.vd_penal, zt);
    TOFE_LAUNCH_CHECK();
  }
  FilterArgs b;
  b.t = tr;
  b.src = zt;
  b.add = REdge;
  b.scale = 1 / sp.vd_min;
  b.rho = rho;
  b.out = so.y;
  b.sp = sp;
  b.so = so;
  if (filter_tile<FM_RADD, FE_SIMP>(s, b)) return;
  k_rfilter_madd<<<dim3(blocks_for(ne)), dim3(NT), 0, s>>>(tr, REdge, zt, b.scale, so.y, ne);
  TOFE_LAUNCH_CHECK();
  k_simp<<<dim3(stride_blocks(ne)), dim3(NT), 0, s>>>(rho, so.y, ne, sp, so);
  TOFE_LAUNCH_CHECK();
}

void chain_void(hipStream_t s, const FilterTemplate &tr, const double *dfdE, const double *rho,
                const double *y, const double *rhoq, double *out, double *t1, double *t2)
{
  const int64_t ne = (int64_t)tr.nx * tr.ny * tr.nz;
  FilterArgs a;
  a.t = tr;
  a.src = dfdE;
  a.rho = rho;
  a.y = y;
  a.rhoq = rhoq;
  a.out = out;
  if (filter_tile<FM_RT, FE_PLAIN>(s, a)) return;
  k_mul<<<dim3(stride_blocks(ne)), dim3(NT), 0, s>>>(dfdE, rho, t1, ne);
  TOFE_LAUNCH_CHECK();
  k_rfilter_T<<<dim3(blocks_for(ne)), dim3(NT), 0, s>>>(tr, t1, t2, ne);
  TOFE_LAUNCH_CHECK();
  k_chain_mid<<<dim3(stride_blocks(ne)), dim3(NT), 0, s>>>(dfdE, y, rhoq, t2, out, ne);
  TOFE_LAUNCH_CHECK();
}

void sensitivity(hipStream_t s, const double *U, const double *dEdz, const double *KE, int nx,
                 int ny, int nz, double *g)
{
  const int64_t ne = (int64_t)nx * ny * nz;
  k_sensitivity<<<dim3(blocks_for(ne)), dim3(NT), 0, s>>>(U, dEdz, KE, nx, ny, nz, g);
  TOFE_LAUNCH_CHECK();
}

void mass_diag(hipStream_t s, const double *V, int nx, int ny, int nz, double m0,
               const double *mlump, const uint8_t *fix, double *M)
{
  const int64_t nn = (int64_t)(nx + 1) * (ny + 1) * (nz + 1);
  k_mass_diag<<<dim3(blocks_for(nn)), dim3(NT), 0, s>>>(V, nx, ny, nz, m0, mlump, fix, M);
  TOFE_LAUNCH_CHECK();
}

void diag_mul(hipStream_t s, const double *d, const double *x, double *y, int64_t n, int nrhs)
{
  k_diag_mul<<<dim3(stride_blocks(n * nrhs)), dim3(NT), 0, s>>>(d, x, y, n, nrhs);
  TOFE_LAUNCH_CHECK();
}

void elem_quad(hipStream_t s, const double *phi, const double *KE, int nx, int ny, int nz,
               int64_t ndof, int nvec, double *kq, double *mq, bool consistent)
{
  const int64_t ne = (int64_t)nx * ny * nz;
  k_elem_quad<<<dim3(blocks_for(ne * nvec)), dim3(NT), 0, s>>>(phi, KE, nx, ny, nz, ndof, nvec,
                                                              kq, mq, consistent ? 1 : 0);
  TOFE_LAUNCH_CHECK();
}

}  // namespace tofe
