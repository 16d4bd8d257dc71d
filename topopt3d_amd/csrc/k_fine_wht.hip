// Matrix-free SIMP stiffness operator, element-centric in the Walsh-Hadamard basis.
//
// Same operator as k_fine_op (y = K(E) u with K = sum_e E_e KE, FEAnalysis.cpp:448-464, and
// the MatZeroRowsColumns rows and columns of FEAnalysis.cpp:473): fixed entries of u are
// zeroed on load and fixed rows return u itself.  Each element product is formed as
// KE u_e = H (M (H u_e)) (two 8-point Walsh-Hadamard transforms per displacement component
// and the 45 terms of the block-diagonal M, about 190 operations instead of 576
// multiply-adds), valid whenever KE has the reflection symmetry of the box element, which
// the host checks before it selects this kernel.
//
// A 256-thread block is a 16 x 16 tile of element columns marching up a chunk of z; thread
// (tx, ty) forms element (x0 - 1 + tx, y0 - 1 + ty) of each layer and owns the node at its
// (1, 1) corner, so the block owns 15 x 15 node columns.  A node's four elements of the
// layer are its own, its right neighbour's (lane + 1 in the same row of 16 lanes: DPP) and
// the two of the row above, whose partial sums come through LDS.  Node planes of u are
// staged in a ring of three LDS planes, loaded into registers one step ahead.
//
// The consistent mass (Dynamic.cpp:181-236's element mass as an exact integral) and the stress
// stiffness (Buckling.cpp:283-414) are sums of element matrices A_e (x) I_3 and take the same march
// with another middle: in the Walsh-Hadamard basis the mass is diagonal (four distinct values)
// and the stress matrix, whose rows sum to zero, is a symmetric 7 x 7 block, 28 stored values.
// A node-centric kernel gathering eight elements of eight nodes each took 1,783 us for M on 16
// vectors of the 160x80x80 mesh (380 us here) and 812 us for Ks on 10 vectors of 128x64x64 (64
// values per element read by every group of four vectors; 340 us here, bound by the stress matrices'
// 117 MB per vector at two wavefronts per SIMD).
#include "k_common.hpp"
#include "ke_wht.hpp"

namespace tofe {
namespace {

constexpr int WT = 16;          // element columns per tile edge, one thread each
constexpr int WN = WT - 1;      // owned node columns per tile edge
constexpr int NW = WT * WT;     // threads per block
constexpr int WP = WT + 1;      // staged node window edge
constexpr int WPL = WP * WP;    // nodes per staged plane

// coordinate index m = x + 2y + 4z of element-local node l
constexpr int mof(int l) { return lnx(l) + 2 * lny(l) + 4 * lnz(l); }

// unnormalised 8-point Walsh-Hadamard transform over the coordinate index
template <typename T>
__device__ inline void wht8(T (&v)[8])
{
#pragma unroll
  for (int b = 1; b < 8; b <<= 1)
#pragma unroll
    for (int m = 0; m < 8; ++m)
      if (!(m & b)) {
        const T a = v[m], c = v[m | b];
        v[m] = a + c;
        v[m | b] = a - c;
      }
}

// value held by lane + 1 of the same row of 16 lanes (0 for the last lane of a row)
template <typename T>
__device__ inline T from_next_lane(T x)
{
  if constexpr (sizeof(T) == 4) {
    return __builtin_bit_cast(T, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x101, 0xf, 0xf, true));
  } else {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, x);
    const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)b, 0x101, 0xf, 0xf, true);
    const unsigned hi = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), 0x101, 0xf, 0xf, true);
    return __builtin_bit_cast(T, ((unsigned long long)hi << 32) | lo);
  }
}

__device__ inline __amdgpu_buffer_rsrc_t wplane_rsrc(const void *base, int bytes)
{
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, bytes, 0x00020000);
}
template <typename T>
__device__ inline T wplane_load(__amdgpu_buffer_rsrc_t r, unsigned off)
{
  if constexpr (sizeof(T) == 4) return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
  else return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}

// what the march applies to an element's values: KE of a box, KE of a cube, the consistent mass,
// or the element's stress matrix
enum ElemForm : int { EF_BOX = 0, EF_CUBE = 1, EF_MASS = 2, EF_STRESS = 3 };

// stored value of block entry B_t[i][j] (cubic elements: its group value)
template <bool CUBE>
constexpr int wht_slot(int t, int i, int j)
{
  return CUBE ? kWhtCubeGroup[wht_index(t, i, j)] : wht_index(t, i, j);
}

// y = E * KE u for the element whose 24 values are v[c][m], in place.
template <typename T, bool CUBE, int NV>
__device__ inline void element_product(T (&v)[3][8], const T (&kb)[NV], T Ee)
{
  wht8(v[0]);
  wht8(v[1]);
  wht8(v[2]);
  // block t couples the entries (j, t ^ e_j), j = 0..2, and writes the same three
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    T x[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) x[j] = v[j][t ^ (1 << j)];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      T acc = 0;
#pragma unroll
      for (int j = 0; j < 3; ++j)
        if (wht_index(t, i, j) >= 0) acc += kb[wht_slot<CUBE>(t, i, j)] * x[j];
      v[i][t ^ (1 << i)] = Ee * acc;
    }
  }
  wht8(v[0]);
  wht8(v[1]);
  wht8(v[2]);
}

// y = Ee m0 (Q (x) I_3) u, in place: Q = 24 (x) [[1/3, 1/6], [1/6, 1/3]] per axis, whose eigenvalues
// on sums and differences are 1/2 and 1/6.
template <typename T>
__device__ inline void mass_product(T (&v)[3][8], T Ee)
{
  const T f[4] = {Ee * (T)(3.0 / 8), Ee * (T)(1.0 / 8), Ee * (T)(1.0 / 24), Ee * (T)(1.0 / 72)};
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    wht8(v[c]);
#pragma unroll
    for (int m = 0; m < 8; ++m) v[c][m] *= f[(m & 1) + ((m >> 1) & 1) + (m >> 2)];
    wht8(v[c]);
  }
}

// y = Ee (H (x) I_3) u, in place, from the 28 values of the stress matrix in this basis.
template <typename T>
__device__ inline void stress_product(T (&v)[3][8], const T (&h)[kStressVals], T Ee)
{
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    wht8(v[c]);
    T x[8];
#pragma unroll
    for (int m = 0; m < 8; ++m) x[m] = v[c][m];
    v[c][0] = 0;
#pragma unroll
    for (int r = 1; r < 8; ++r) {
      T acc = 0;
#pragma unroll
      for (int m = 1; m < 8; ++m) acc += h[stress_index(r, m)] * x[m];
      v[c][r] = Ee * acc;
    }
    wht8(v[c]);
  }
}

// One block of the operator: tile `bid` of the launch's `nblocks` (per vector), vector `vec`.
template <typename T, int EPI, int FORM>
__device__ __forceinline__ void fine_wht_block(const FineOp<T> &op, const T *u0, EpiArgs<T> ep,
                                               int tiles_x, int tiles_y, int nblocks, int zlen,
                                               int bid, int vec)
{
  // partial sums handed to the row below (lower, upper node): double-buffered in FP32; one
  // buffer and a second barrier per step in FP64, which keeps the block at 33 KB of LDS (four
  // resident blocks per CU instead of three)
  constexpr int NPB = sizeof(T) == 8 ? 1 : 2;
  __shared__ T su[3][3][WPL];     // ring of three node planes, one array per component
  __shared__ T sp[NPB][6][NW];
  __shared__ double sred[NW / 64];

  const int nx = op.nx, ny = op.ny, nz = op.nz;
  const int Nx = nx + 1, Ny = ny + 1, Nz = nz + 1;
  epi_offset(ep, vec, 3 * (int64_t)Nx * Ny * Nz, nblocks);
  const T *__restrict__ u = u0 + vec * (3 * (int64_t)Nx * Ny * Nz);
  const int txy = tiles_x * tiles_y;
  const int bz = bid / txy;
  const int rem = bid - bz * txy;
  const int by = rem / tiles_x, bx = rem - by * tiles_x;
  const int x0 = bx * WN, y0 = by * WN;  // first owned node column
  const int k0 = bz * zlen, k1 = min(k0 + zlen, Nz);
  const int t = threadIdx.x;
  const int tx = t % WT, ty = t / WT;
  const int ex = x0 - 1 + tx, ey = y0 - 1 + ty;  // element column of this thread
  const int i = x0 + tx, j = y0 + ty;            // owned node column
  const bool own = tx < WN && ty < WN && i < Nx && j < Ny;
  constexpr unsigned kNone = 0xffffffffu;
  const unsigned eidx = (ex >= 0 && ex < nx && ey >= 0 && ey < ny) ? unsigned(ex + nx * ey) : kNone;
  const T *__restrict__ E = op.E;
  const uint8_t *__restrict__ fix = op.fix;
  const int NxNy = Nx * Ny, nxny = nx * ny;

  constexpr bool CUBE = FORM == EF_CUBE, KEFORM = FORM == EF_BOX || FORM == EF_CUBE;
  constexpr int NV = !KEFORM ? 1 : CUBE ? kWhtCubeVals : kWhtVals;
  T kb[NV];
  if constexpr (KEFORM) {
#pragma unroll
    for (int k = 0; k < NV; ++k) kb[k] = op.KE[(CUBE ? kWhtCubeOffset : kWhtOffset) + k];
  }
  const int64_t ne = (int64_t)nxny * nz;

  // staging map: node slot q of this thread is node t + q * NW of the staged window
  // (x0 - 1 .. x0 + 15) x (y0 - 1 .. y0 + 15), its in-plane index or kNone
  constexpr int NU = (WPL + NW - 1) / NW;
  unsigned u_node[NU];
#pragma unroll
  for (int q = 0; q < NU; ++q) {
    const int nl = t + q * NW;
    const int ly = nl / WP, lx = nl - ly * WP;
    const int gx = x0 - 1 + lx, gy = y0 - 1 + ly;
    u_node[q] = (nl < WPL && gx >= 0 && gx < Nx && gy >= 0 && gy < Ny) ? unsigned(gx + Nx * gy) : kNone;
  }
  // EPI_CHEB_FIRST: pu holds b and pd D^-1 of the node, and the staged operand is c20 (D^-1 b)
  constexpr bool FIRST = EPI == EPI_CHEB_FIRST;
  constexpr int ND = FIRST ? NU : 1;
  const T *__restrict__ ub = FIRST ? ep.b : u;
  auto load_u = [&](T (&pu)[NU][3], T (&pd)[ND][3], unsigned (&pf)[NU], int gz) {
    const bool zin = gz >= 0 && gz < Nz;
    const int64_t z = zin ? gz : 0;
    const __amdgpu_buffer_rsrc_t ur = wplane_rsrc(ub + 3 * NxNy * z, 3 * NxNy * (int)sizeof(T));
    const __amdgpu_buffer_rsrc_t dr =
        wplane_rsrc(FIRST ? ep.dinv + 3 * NxNy * z : ub, FIRST ? 3 * NxNy * (int)sizeof(T) : 0);
    const __amdgpu_buffer_rsrc_t fr = wplane_rsrc(fix ? fix + NxNy * z : fix, NxNy);
#pragma unroll
    for (int q = 0; q < NU; ++q) {
      pu[q][0] = pu[q][1] = pu[q][2] = 0;
      if constexpr (FIRST) pd[q][0] = pd[q][1] = pd[q][2] = 0;
      pf[q] = 0;
      if (zin && u_node[q] != kNone) {
        const unsigned off = u_node[q] * (3 * sizeof(T));
#pragma unroll
        for (int c = 0; c < 3; ++c) pu[q][c] = wplane_load<T>(ur, off + c * sizeof(T));
        if constexpr (FIRST) {
#pragma unroll
          for (int c = 0; c < 3; ++c) pd[q][c] = wplane_load<T>(dr, off + c * sizeof(T));
        }
        if (fix) pf[q] = __builtin_amdgcn_raw_buffer_load_b8(fr, u_node[q], 0, 0);
      }
    }
  };
  // the fixed-DOF mask is applied at the store, after the arithmetic that hides the loads
  auto store_u = [&](const T (&pu)[NU][3], const T (&pd)[ND][3], const unsigned (&pf)[NU], int slot) {
#pragma unroll
    for (int q = 0; q < NU; ++q) {
      const int nl = t + q * NW;
      if (nl < WPL) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          T v = pu[q][c];
          if constexpr (FIRST) v = ep.c20 * (pd[q][c] * v);
          su[slot][c][nl] = ((pf[q] >> c) & 1u) ? T(0) : v;
        }
      }
    }
  };
  auto load_E = [&](int ez) -> T {
    if (!(ez >= 0 && ez < nz && eidx != kNone)) return T(0);
    const T e = E[eidx + (int64_t)nxny * ez];
    return KEFORM ? e : op.escale * e;
  };

  // stress matrix of this thread's element of layer ez (zero outside the mesh)
  constexpr int NH = FORM == EF_STRESS ? kStressVals : 1;
  T h[NH];
  auto load_H = [&](T (&hv)[NH], int ez) {
#pragma unroll
    for (int k = 0; k < NH; ++k) hv[k] = 0;
    if (ez >= 0 && ez < nz && eidx != kNone) {
      const T *__restrict__ H = op.H + (eidx + (int64_t)nxny * ez);
#pragma unroll
      for (int k = 0; k < NH; ++k) hv[k] = H[k * ne];
    }
  };

  T alo[3], ahi[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) ahi[c] = 0;
  double dsum = 0, dsum2 = 0;

  T Ecur;
  {
    T pu[NU][3], pd[ND][3];
    unsigned pf[NU];
    load_u(pu, pd, pf, k0 - 1);
    store_u(pu, pd, pf, 0);
    load_u(pu, pd, pf, k0);
    store_u(pu, pd, pf, 1);
    Ecur = load_E(k0 - 1);
    if constexpr (FORM == EF_STRESS) load_H(h, k0 - 1);
  }
  __syncthreads();
  // Step st (element layer ez = k0 - 1 + st) reads node planes ez and ez + 1 from ring slots
  // st % 3 and (st + 1) % 3, writes partial sums to sp[st % 2] and node plane ez + 2 to slot
  // (st + 2) % 3, then passes the step's barrier.  Those two were last read before the
  // barrier of step st - 1 (FP32); with the single sp buffer of FP64 a second barrier ahead
  // of the sp writes orders them after the previous step's reads.
  int st = 0;
  for (int ez = k0 - 1; ez < k1; ++ez, ++st) {
    const int slo = st % 3, shi = (st + 1) % 3, pb = NPB == 2 ? (st & 1) : 0;
    const bool more = ez + 1 < k1;
    T pu[NU][3], pd[ND][3];
    unsigned pf[NU];
    T Enext = 0;
    if (more) {
      load_u(pu, pd, pf, ez + 2);
      Enext = load_E(ez + 1);
    }
    // this step's epilogue inputs, loaded ahead of the element arithmetic
    const bool emit = own && ez >= k0;
    const int64_t n = i + (int64_t)Nx * (j + (int64_t)Ny * ez);
    EpiIn<T, EPI> ein;
    if (emit) epi_load<T, EPI>(ep, u, fix, n, ein);
    T hn[NH];
    if constexpr (FORM == EF_STRESS) load_H(hn, more ? ez + 1 : -1);
    T v[3][8];
#pragma unroll
    for (int l = 0; l < 8; ++l) {
      const int nl = (ty + lny(l)) * WP + tx + lnx(l);
#pragma unroll
      for (int c = 0; c < 3; ++c) v[c][mof(l)] = su[lnz(l) ? shi : slo][c][nl];
    }
    if constexpr (FORM == EF_MASS) mass_product<T>(v, Ecur);
    else if constexpr (FORM == EF_STRESS) stress_product<T>(v, h, Ecur);
    else element_product<T, CUBE, NV>(v, kb, Ecur);
    // node (i, j): own element's corner (1, 1) [m = 3 lower, 7 upper] + right element's
    // corner (0, 1) [m = 2, 6]; the row above contributes corners (1, 0) and (0, 0)
    // [m = 1, 5 and 0, 4] of its two elements, summed there and passed through LDS
    T plo[3], phi[3];
    if constexpr (NPB == 1) __syncthreads();  // the previous step's readers of sp are done
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      plo[c] = v[c][3] + from_next_lane(v[c][2]);
      phi[c] = v[c][7] + from_next_lane(v[c][6]);
      sp[pb][c][t] = v[c][1] + from_next_lane(v[c][0]);
      sp[pb][3 + c][t] = v[c][5] + from_next_lane(v[c][4]);
    }
    if (more) store_u(pu, pd, pf, (st + 2) % 3);
    __syncthreads();
    const int tb = min(t + WT, NW - 1);  // thread (tx, ty + 1); ty = 15 owns no node
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      alo[c] = ahi[c] + (plo[c] + sp[pb][c][tb]);
      ahi[c] = phi[c] + sp[pb][3 + c][tb];
    }
    if (emit) {
      if (op.spk) {  // spring supports (point masses): + diag(spk) on free DOFs
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const T uv = FIRST ? ep.c20 * (ein.dinv[c] * ein.b[c]) : ein.u[c];
          alo[c] += op.spk[3 * n + c] * uv;
        }
      }
      if constexpr (KEFORM) {
        epi_store<T, EPI>(ep, n, ein, alo, dsum, dsum2);
      } else {
#pragma unroll
        for (int c = 0; c < 3; ++c)
          ep.y[3 * n + c] = ((ein.fm >> c) & 1) ? op.fixval * ein.u[c] : alo[c];
      }
    }
    Ecur = Enext;
    if constexpr (FORM == EF_STRESS) {
#pragma unroll
      for (int k = 0; k < NH; ++k) h[k] = hn[k];
    }
  }
  if constexpr (EPI == EPI_APPLY_DOT || EPI == EPI_APPLY_DOT2 || EPI == EPI_CHEB_OUT) {
    __syncthreads();
    const double s1 = block_sum<NW>(dsum, sred);
    if (t == 0) ep.partial[bid] = s1;
    if constexpr (EPI == EPI_APPLY_DOT2) {
      __syncthreads();
      const double s2 = block_sum<NW>(dsum2, sred);
      if (t == 0) ep.partial2[bid] = s2;
    }
  }
}

// Vectors are the launch's second axis.  (Blocks of a tile's vectors next to one another on one XCD,
// so that E and D^-1 or the stress matrices come from its L2, measured slower: a Chebyshev step on
// 16 vectors of the 160x80x80 mesh 702 against 670 us, Ks on 10 of 128x64x64 363 against 340 us.)
template <typename T, int EPI, int FORM>
__global__ __launch_bounds__(NW) void k_fine_wht(FineOp<T> op, const T *u0, EpiArgs<T> ep,
                                                 int tiles_x, int tiles_y, int nblocks, int zlen)
{
  fine_wht_block<T, EPI, FORM>(op, u0, ep, tiles_x, tiles_y, nblocks, zlen,
                               xcd_remap(blockIdx.x, gridDim.x), blockIdx.y);
}

// The operator of several instances in one grid: entry e of the table owns blocks
// [b0[e], b0[e + 1]).  (Cubic and general elements take separate launches: one kernel holding
// both bodies would hold both bodies' LDS arrays.)
template <typename T, int EPI, int FORM>
__global__ __launch_bounds__(NW) void k_fine_wht_batch(const FineLaunch<T> *__restrict__ tab,
                                                       const int *__restrict__ b0, int n)
{
  const int e = batch_entry(b0, n, blockIdx.x);
  const FineLaunch<T> L = tab[e];
  fine_wht_block<T, EPI, FORM>(L.op, L.u, L.ep, L.tiles_x, L.tiles_y, L.nblocks, L.zlen,
                               xcd_remap(blockIdx.x - b0[e], L.nblocks), blockIdx.y);
}

struct WhtGrid {
  int tiles_x, tiles_y, nblocks;
};

template <typename T>
WhtGrid wht_grid(const FineOp<T> &op)
{
  if (op.zlen < 1) throw Error(TOFE_ERR_ARG, "fine operator: invalid z-chunk length");
  if ((int64_t)3 * (op.nx + 1) * (op.ny + 1) * (int64_t)sizeof(T) >= (int64_t(1) << 31))
    throw Error(TOFE_ERR_ARG, "fine operator: node plane of 2 GiB or more");
  WhtGrid g;
  g.tiles_x = (op.nx + 1 + WN - 1) / WN;
  g.tiles_y = (op.ny + 1 + WN - 1) / WN;
  g.nblocks = g.tiles_x * g.tiles_y * ((op.nz + 1 + op.zlen - 1) / op.zlen);
  return g;
}

}  // namespace

int fine_wht_zlen(int nx, int ny, int nz, int ncu, int hide, int nvec, int zmax)
{
  // A block lasts a fixed start (the first two planes and the launch itself, about two and a
  // half steps) and zlen + 1 steps, since the chunk's lowest element layer is formed too; with m
  // blocks on the busiest CU the launch takes a time proportional to m + hide, `hide` being the
  // blocks whose latencies overlap for free.  Measured on MI355X over 24x12x12 to 192x96x96
  // elements (us per apply, FP64 / FP32): one step more costs 1.33 / 1.15 on a grid of one block
  // per CU; 24x12x12 5.1 / 4.6 at zlen 1 and 9.1 / 8.0 at 4; 96x48x48 13.5 / 9.3 at 1, 11.2 / 8.4
  // at 2, 13.0 / 9.8 at 4; 128x64x64 17.0 / 12.3 at 3; 192x96x96 fastest at 7.  The larger chunk
  // wins ties.
  const int tiles = ((nx + 1 + WN - 1) / WN) * ((ny + 1 + WN - 1) / WN);
  int best = 8;
  double best_cost = 1e300;
  ncu = std::max(ncu, 1);
  for (int zl = 1; zl <= zmax; ++zl) {
    const int nb = tiles * ((nz + 1 + zl - 1) / zl);
    const double cost = (zl + 3.0) * (((int64_t)nb * nvec + ncu - 1) / ncu + hide);
    if (cost < best_cost - 1e-9 || (cost < best_cost + 1e-9 && zl > best)) {
      best_cost = cost;
      best = zl;
    }
  }
  return best;
}

template <typename T>
int fine_wht_blocks(const FineOp<T> &op)
{
  return wht_grid(op).nblocks;
}

// Several vectors, or the instances of a batch, fill the CUs with longer chunks, which form fewer
// extra element layers: the rule's best of up to eight planes for K and M (six, seven, eight and ten
// measured alike over 48x24x24 to 160x80x80, 2 to 16 vectors; the best of all lengths cut at six lost 5 to
// 10% where that is seven: K on 16 vectors of 61x33x27 42.8 and 38.8 us, on 2 of 200x40x40 33.7 and
// 32.5) and of up to six for the kernels with further fields, the V-cycle's and Ks (a Chebyshev step on
// 16 vectors of 160x80x80 670 us at 6, 717 at 14; V-cycle on 16 of 130x50x46 1,323 at up to 6, 1,374 at
// up to 8; Ks, K and V-cycle on 10 of 128x64x64 1,367 and 1,398).  A merged solve of 32 instances of 16 to 96 elements along x, ms: with their own lengths 57.5
// for four load cases each and 35.3 for one, this way 54.1 and 34.4.  The chunk length does not show in
// the outputs, only in the partial sums of the dot products, where each vector's stay those of its
// own launch.
constexpr int kSharedZlenApply = 8, kSharedZlenFields = 6;
template <typename T>
int fine_wht_shared_zlen(const FineOp<T> &op, Epi epi, int nvec)
{
  const bool sums = epi == EPI_APPLY_DOT || epi == EPI_APPLY_DOT2 || epi == EPI_CHEB_OUT;
  const int zmax = epi == EPI_APPLY && !op.H ? kSharedZlenApply : kSharedZlenFields;
  if (sums || nvec <= 1 || op.ncu <= 0 || op.zlen >= zmax) return op.zlen;
  return fine_wht_zlen(op.nx, op.ny, op.nz, op.ncu, sizeof(T) == 8 ? kWhtHide64 : kWhtHide32, nvec, zmax);
}

template <typename T, int EPI, int FORM>
void launch_form(hipStream_t s, FineOp<T> op, const T *u, const EpiArgs<T> &ep)
{
  op.zlen = fine_wht_shared_zlen(op, (Epi)EPI, ep.nvec);
  const WhtGrid g = wht_grid(op);
  k_fine_wht<T, EPI, FORM><<<dim3(g.nblocks, ep.nvec), dim3(NW), 0, s>>>(op, u, ep, g.tiles_x, g.tiles_y,
                                                                        g.nblocks, op.zlen);
}
template <typename T, int EPI>
void launch_wht(hipStream_t s, const FineOp<T> &op, const T *u, const EpiArgs<T> &ep)
{
  if (op.wht_cube) launch_form<T, EPI, EF_CUBE>(s, op, u, ep);
  else launch_form<T, EPI, EF_BOX>(s, op, u, ep);
}

void fine_mass(hipStream_t s, const FineOp<double> &op, const double *u, const EpiArgs<double> &ep)
{
  launch_form<double, EPI_APPLY, EF_MASS>(s, op, u, ep);
  TOFE_LAUNCH_CHECK();
}

void fine_stress(hipStream_t s, const FineOp<double> &op, const double *u, const EpiArgs<double> &ep)
{
  launch_form<double, EPI_APPLY, EF_STRESS>(s, op, u, ep);
  TOFE_LAUNCH_CHECK();
}

template <typename T>
void fine_wht(hipStream_t s, const FineOp<T> &op, const T *u, Epi epi, const EpiArgs<T> &ep)
{
  switch (epi) {
    case EPI_APPLY: launch_wht<T, EPI_APPLY>(s, op, u, ep); break;
    case EPI_APPLY_DOT: launch_wht<T, EPI_APPLY_DOT>(s, op, u, ep); break;
    case EPI_APPLY_DOT2: launch_wht<T, EPI_APPLY_DOT2>(s, op, u, ep); break;
    case EPI_RESID: launch_wht<T, EPI_RESID>(s, op, u, ep); break;
    case EPI_CHEB: launch_wht<T, EPI_CHEB>(s, op, u, ep); break;
    case EPI_CHEB_OUT: launch_wht<T, EPI_CHEB_OUT>(s, op, u, ep); break;
    case EPI_CHEB_FIRST: launch_wht<T, EPI_CHEB_FIRST>(s, op, u, ep); break;
  }
  TOFE_LAUNCH_CHECK();
}

template <typename T>
int fine_wht_grid(const FineOp<T> &op, int *tiles_x, int *tiles_y)
{
  const WhtGrid g = wht_grid(op);
  *tiles_x = g.tiles_x;
  *tiles_y = g.tiles_y;
  return g.nblocks;
}

template <typename T, int EPI>
void launch_wht_batch(hipStream_t s, bool cube, const FineLaunch<T> *tab, const int *b0, int n,
                      int nblocks_total, int nvec)
{
  dim3 grid(nblocks_total, nvec), block(NW);
  if (cube) k_fine_wht_batch<T, EPI, EF_CUBE><<<grid, block, 0, s>>>(tab, b0, n);
  else k_fine_wht_batch<T, EPI, EF_BOX><<<grid, block, 0, s>>>(tab, b0, n);
}

template <typename T>
void fine_wht_batch(hipStream_t s, Epi epi, bool cube, const FineLaunch<T> *tab, const int *b0,
                    int n, int nblocks_total, int nvec)
{
  switch (epi) {
    case EPI_APPLY: launch_wht_batch<T, EPI_APPLY>(s, cube, tab, b0, n, nblocks_total, nvec); break;
    case EPI_APPLY_DOT: launch_wht_batch<T, EPI_APPLY_DOT>(s, cube, tab, b0, n, nblocks_total, nvec); break;
    case EPI_APPLY_DOT2: launch_wht_batch<T, EPI_APPLY_DOT2>(s, cube, tab, b0, n, nblocks_total, nvec); break;
    case EPI_RESID: launch_wht_batch<T, EPI_RESID>(s, cube, tab, b0, n, nblocks_total, nvec); break;
    case EPI_CHEB: launch_wht_batch<T, EPI_CHEB>(s, cube, tab, b0, n, nblocks_total, nvec); break;
    case EPI_CHEB_OUT: launch_wht_batch<T, EPI_CHEB_OUT>(s, cube, tab, b0, n, nblocks_total, nvec); break;
    case EPI_CHEB_FIRST: launch_wht_batch<T, EPI_CHEB_FIRST>(s, cube, tab, b0, n, nblocks_total, nvec); break;
  }
  TOFE_LAUNCH_CHECK();
}

template int fine_wht_grid<double>(const FineOp<double> &, int *, int *);
template int fine_wht_grid<float>(const FineOp<float> &, int *, int *);
template void fine_wht_batch<double>(hipStream_t, Epi, bool, const FineLaunch<double> *, const int *,
                                     int, int, int);
template void fine_wht_batch<float>(hipStream_t, Epi, bool, const FineLaunch<float> *, const int *,
                                    int, int, int);
template int fine_wht_shared_zlen<double>(const FineOp<double> &, Epi, int);
template int fine_wht_shared_zlen<float>(const FineOp<float> &, Epi, int);
template int fine_wht_blocks<double>(const FineOp<double> &);
template int fine_wht_blocks<float>(const FineOp<float> &);
template void fine_wht<double>(hipStream_t, const FineOp<double> &, const double *, Epi, const EpiArgs<double> &);
template void fine_wht<float>(hipStream_t, const FineOp<float> &, const float *, Epi, const EpiArgs<float> &);

}  // namespace tofe
