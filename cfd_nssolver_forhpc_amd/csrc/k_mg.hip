// k_mg.hip -- cell-centred geometric multigrid V-cycle used as a
// preconditioner of the pressure solve (an addition: the reference solves
// with Jacobi-scaled BiCGSTAB only).
//
// The Jacobi-scaled operator is A = J L with J = diag(jp) and L the
// finite-volume Laplacian of createPressureMatrix (inc/matrix/
// PressureMatrix.hpp:5-117): per axis, the coefficient to the -/+ neighbour
// is 1/(D[i] Ds[i-1]) / 1/(D[i] Ds[i]), Neumann faces drop theirs, Dirichlet
// faces keep theirs in the diagonal.  M^-1 r = V-cycle(L, r / jp) is a cheap
// approximation of A^-1 r.
//
// Every level is matrix-free: the grids are tensor products, so a level is
// its extents plus per-axis arrays (coefficients to the -/+ neighbour, their
// diagonal share, cell widths); a smoothing sweep streams only x and b.
// Coarse levels halve every axis that is even and at least 4 cells long;
// their coefficients are rediscretised from the merged cell widths (a
// Dirichlet face keeps its mirror-ghost coefficient).  With periodic z every
// level wraps in z like the operator (the first and last planes are
// neighbours across the seam); z is halved only while its length stays even,
// so the red-black colouring stays consistent across the seam.  Restriction is the
// volume-weighted sum of the children's residuals, prolongation adds the
// parent's correction.  Smoother: red-black Gauss-Seidel, nu sweeps before
// and after.  Levels of at most MG_SMALL cells run inside one workgroup (one
// launch for the whole bottom of the cycle, mg_bottom_kernel; mg_small_kernel
// where the coarsest level has more cells); the coarsest is solved by its dense
// inverse or smoothed MG_COARSE_SWEEPS times.
//
// The finest level keeps x and b colour-split (ColourSplit), and so does every
// next level while the level above halves every axis and it is not part of
// the one-workgroup bottom (split_levels).  Their sweeps run up to four
// half-sweeps in one pass over the level (mg_fused_kernel), the first pass
// after the coarse correction with the prolongation folded in, the last one
// writing the result; the restriction reads the children as colour pairs.
// What a pass cannot take (one sweep, the odd sweep of an odd count, lines of
// more than 128 cells, whose z its tiles do not split) runs as single colour sweeps whose threads walk
// MG_PLANES planes and load each other-colour entry once for its three uses.
// Each does the arithmetic of the generic per-cell functions term for term,
// so the cycle's result is the same bit for bit in either layout.
//
// Every kernel returns at once when the Krylov solver's `done` flag is set,
// so preconditioned iterations can be launched in batches like the plain
// ones.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "dev_common.h"
#include "pred_tiled.h"

namespace cfd {

constexpr int MG_MAX_LEVELS = 16;
constexpr int64_t MG_SMALL = 4096;
constexpr int MG_COARSE_SWEEPS = 48;
// per-level device view: ax = cm[nx] cp[nx] dd[nx] w[nx] (and ay, az)
struct MGView {
  int nx, ny, nz, fx, fy, fz;
  int wz;  // periodic z: k = 0 and k = nz - 1 are neighbours (nz even)
  int64_t n;
  const double *ax, *ay, *az;
};

struct MGLevel {
  MGView v{};
  double *coef = nullptr;               // ax | ay | az
  double *x64 = nullptr, *b64 = nullptr;
  float *x32 = nullptr, *b32 = nullptr;
  // a colour-split level below the finest: its x in natural layout, written
  // by its last post-smoothing half-sweep for the prolongation above it
  double *xn64 = nullptr;
  float *xn32 = nullptr;
  // the second x of a level with fused passes: mg_fused_kernel reads one and writes the other
  double *xb64 = nullptr;
  float *xb32 = nullptr;
};

struct MGState {
  std::vector<MGLevel> lv;
  int small_from = 0;   // first level handled by the one-workgroup kernel
  int nu = 2;
  std::string shape;
  int split_levels = 0; // levels 0 .. split_levels - 1 are colour-split (they run the split kernels)
  int dense_n = 0;      // > 0: the coarsest level (dense_n cells) is solved by its dense inverse
  double *cinv64 = nullptr;
  float *cinv32 = nullptr;
};

namespace {

template <typename T>
int mg_alloc(T **p, size_t n) {
  *p = nullptr;
  hipError_t e = hipMalloc((void **)p, (n ? n : 1) * sizeof(T));
  if (e != hipSuccess) {
    *p = nullptr;
    return fail(CFD_ERR_NOMEM, std::string("multigrid: hipMalloc failed: ") + hipGetErrorString(e));
  }
  return CFD_OK;
}

template <typename T>
void mg_free(T *&p) {
  if (p) (void)hipFree((void *)p);
  p = nullptr;
}

__device__ inline int64_t idx3(const MGView &L, int i, int j, int k) { return ((int64_t)i * L.ny + j) * L.nz + k; }

// the z index one step down / up, across the seam with periodic z (meaningful
// where that neighbour exists)
__device__ inline int kdn(const MGView &L, int k) { return k > 0 ? k - 1 : L.nz - 1; }
__device__ inline int kup(const MGView &L, int k) { return k < L.nz - 1 ? k + 1 : 0; }

// a cell's own index and its neighbours' (meaningful where the neighbour exists)
struct Nb {
  int64_t c, xm, xp, ym, yp, zm, zp;
};

// Layouts of a level's x and b.  Natural: (i ny + j) nz + k.
struct Natural {
  __device__ static int64_t at(const MGView &L, int i, int j, int k) { return idx3(L, i, j, k); }
  __device__ static Nb nbrs(const MGView &L, int i, int j, int k) {
    const int64_t c = idx3(L, i, j, k), sx = (int64_t)L.ny * L.nz, sy = L.nz;
    return Nb{c, c - sx, c + sx, c - sy, c + sy, k > 0 ? c - 1 : c + (L.nz - 1), k < L.nz - 1 ? c + 1 : c - (L.nz - 1)};
  }
};

// ColourSplit (the finest level of a multi-level cycle): the red cells
// (i + j + k even) first, then the black ones, each colour at
// (i ny + j) hz + k/2 with hz = ceil(nz / 2).  A colour sweep streams its
// own half and reads the other at unit stride instead of touching every line
// of both at stride 2.  For odd nz one colour has an unused last slot per
// row.  The six neighbours of a cell are the other colour's entries at
// h -+ ny hz, h -+ hz and, along k, h or h -+ 1 by the parity of k.
struct ColourSplit {
  __device__ static int64_t half(const MGView &L) { return (int64_t)L.nx * L.ny * ((L.nz + 1) >> 1); }
  __device__ static int64_t at(const MGView &L, int i, int j, int k) {
    const int hz = (L.nz + 1) >> 1;
    const int64_t h = ((int64_t)i * L.ny + j) * hz + (k >> 1);
    return ((i + j + k) & 1) ? half(L) + h : h;
  }
  __device__ static Nb nbrs(const MGView &L, int i, int j, int k) {
    const int hz = (L.nz + 1) >> 1;
    const int64_t h = ((int64_t)i * L.ny + j) * hz + (k >> 1), ns = half(L);
    const bool black = (i + j + k) & 1;
    const int64_t own = black ? ns + h : h, oth = black ? h : ns + h, sx = (int64_t)L.ny * hz;
    // across the periodic seam (nz even): k = 0's -z neighbour is k = nz - 1
    // at k/2 = hz - 1, and k = nz - 1's +z neighbour k = 0 at k/2 = 0
    const int64_t zm = k > 0 ? oth - ((k & 1) ? 0 : 1) : oth + (hz - 1);
    const int64_t zp = k < L.nz - 1 ? oth + (k & 1) : oth - (hz - 1);
    return Nb{own, oth - sx, oth + sx, oth - hz, oth + hz, zm, zp};
  }
};

template <typename T>
__device__ inline T mg_diag(const MGView &L, int i, int j, int k) {
  return (T)(L.ax[2 * L.nx + i] + L.ay[2 * L.ny + j] + L.az[2 * L.nz + k]);
}

// which of the six neighbours exist
struct Has {
  bool xm, xp, ym, yp, zm, zp;
};
__device__ inline Has has6(const MGView &L, int i, int j, int k) {
  return Has{i > 0, i < L.nx - 1, j > 0, j < L.ny - 1, L.wz || k > 0, L.wz || k < L.nz - 1};
}

// the six neighbour coefficients (an absent neighbour's entry is 0 and in range)
template <typename T>
struct Coef6 {
  T xm, xp, ym, yp, zm, zp;
};
template <typename T>
__device__ inline Coef6<T> coef6(const MGView &L, int i, int j, int k) {
  return Coef6<T>{(T)L.ax[i], (T)L.ax[L.nx + i], (T)L.ay[j], (T)L.ay[L.ny + j], (T)L.az[k], (T)L.az[L.nz + k]};
}

// sum over the neighbours of coefficient * x, in the order -x +x -y +y -z
// +z.  Every load is issued before the sum (an absent neighbour reads the
// cell itself and is left out by a select), so a wave has all of them in
// flight at once instead of one exec-masked load and wait per neighbour.
template <typename T>
__device__ inline T mg_off(const MGView &L, const T *__restrict__ x, int i, int j, int k, const Nb &n) {
  const Has h = has6(L, i, j, k);
  const T vxm = x[h.xm ? n.xm : n.c], vxp = x[h.xp ? n.xp : n.c], vym = x[h.ym ? n.ym : n.c];
  const T vyp = x[h.yp ? n.yp : n.c], vzm = x[h.zm ? n.zm : n.c], vzp = x[h.zp ? n.zp : n.c];
  const Coef6<T> a = coef6<T>(L, i, j, k);
  T s = (T)0;
  s = h.xm ? s + a.xm * vxm : s;
  s = h.xp ? s + a.xp * vxp : s;
  s = h.ym ? s + a.ym * vym : s;
  s = h.yp ? s + a.yp * vyp : s;
  s = h.zm ? s + a.zm * vzm : s;
  s = h.zp ? s + a.zp * vzp : s;
  return s;
}

template <typename T>
__device__ inline double mg_vol(const MGView &L, int i, int j, int k) {
  return L.ax[3 * L.nx + i] * L.ay[3 * L.ny + j] * L.az[3 * L.nz + k];
}

// one colour of a red-black Gauss-Seidel sweep at (i, j, k2), k = 2 k2 +
// parity (colour 0 = red: i + j + k even)
template <typename T, typename Lay>
__device__ inline void rb_at(const MGView &L, int i, int j, int k2, int colour, const T *__restrict__ b,
                             T *__restrict__ x) {
  const int k = 2 * k2 + ((i + j + colour) & 1);
  if (k >= L.nz) return;
  const Nb n = Lay::nbrs(L, i, j, k);
  x[n.c] = (b[n.c] + mg_off<T>(L, x, i, j, k, n)) / mg_diag<T>(L, i, j, k);
}

// parent of fine cell (i, j, k) on the next coarser level
__device__ inline int64_t parent(const MGView &F, const MGView &C, int i, int j, int k) {
  return idx3(C, F.fx == 2 ? i >> 1 : i, F.fy == 2 ? j >> 1 : j, F.fz == 2 ? k >> 1 : k);
}

// the first red sweep after the coarse correction, with the prolongation
// folded in: the black neighbours are read as x + xc[parent].  Red cells are
// overwritten here and black cells by the black sweep that follows, so the
// corrected values are only ever needed as neighbours.
template <typename T, typename Lay>
__device__ inline void rb_prolong_at(const MGView &F, const MGView &C, int i, int j, int k2, const T *__restrict__ b,
                                     T *__restrict__ x, const T *__restrict__ xc) {
  const int k = 2 * k2 + ((i + j) & 1);
  if (k >= F.nz) return;
  const Nb n = Lay::nbrs(F, i, j, k);
  const Has h = has6(F, i, j, k);
  // all loads first (absent neighbours read the cell and its parent), as in mg_off
  const T vxm = x[h.xm ? n.xm : n.c] + xc[parent(F, C, h.xm ? i - 1 : i, j, k)];
  const T vxp = x[h.xp ? n.xp : n.c] + xc[parent(F, C, h.xp ? i + 1 : i, j, k)];
  const T vym = x[h.ym ? n.ym : n.c] + xc[parent(F, C, i, h.ym ? j - 1 : j, k)];
  const T vyp = x[h.yp ? n.yp : n.c] + xc[parent(F, C, i, h.yp ? j + 1 : j, k)];
  const T vzm = x[h.zm ? n.zm : n.c] + xc[parent(F, C, i, j, h.zm ? kdn(F, k) : k)];
  const T vzp = x[h.zp ? n.zp : n.c] + xc[parent(F, C, i, j, h.zp ? kup(F, k) : k)];
  const Coef6<T> a = coef6<T>(F, i, j, k);
  T s = (T)0;
  s = h.xm ? s + a.xm * vxm : s;
  s = h.xp ? s + a.xp * vxp : s;
  s = h.ym ? s + a.ym * vym : s;
  s = h.yp ? s + a.yp * vyp : s;
  s = h.zm ? s + a.zm * vzm : s;
  s = h.zp ? s + a.zp * vzp : s;
  x[n.c] = (b[n.c] + s) / mg_diag<T>(F, i, j, k);
}

// a new right-hand side at cell (i, j, k) and the first red half-sweep from x = 0
template <typename T, typename Lay>
__device__ inline void set_rhs(const MGView &L, int i, int j, int k, T bv, T *__restrict__ b, T *__restrict__ x) {
  const int64_t c = Lay::at(L, i, j, k);
  b[c] = bv;
  x[c] = ((i + j + k) & 1) == 0 ? bv / mg_diag<T>(L, i, j, k) : (T)0;
}

// residual of the children of coarse cell (I, J, K), volume-weighted into
// the coarse right-hand side (which starts its own first red half-sweep);
// the coarse level is always in natural layout
template <typename T, typename Lay>
__device__ inline double child_res(const MGView &F, int i, int j, int k, const T *__restrict__ bf,
                                   const T *__restrict__ xf) {
  const Nb n = Lay::nbrs(F, i, j, k);
  const T r = bf[n.c] - (mg_diag<T>(F, i, j, k) * xf[n.c] - mg_off<T>(F, xf, i, j, k, n));
  return mg_vol<T>(F, i, j, k) * (double)r;
}

template <typename T, typename Lay>
__device__ inline void restrict_at(const MGView &F, const MGView &C, int I, int J, int K, const T *__restrict__ bf,
                                   const T *__restrict__ xf, T *__restrict__ bc, T *__restrict__ xc) {
  double acc = 0.0;
  if (F.fx == 2 && F.fy == 2 && F.fz == 2) {
#pragma unroll
    for (int d = 0; d < 8; ++d)
      acc += child_res<T, Lay>(F, 2 * I + (d >> 2), 2 * J + ((d >> 1) & 1), 2 * K + (d & 1), bf, xf);
  } else {
    for (int di = 0; di < F.fx; ++di)
      for (int dj = 0; dj < F.fy; ++dj)
        for (int dk = 0; dk < F.fz; ++dk)
          acc += child_res<T, Lay>(F, I * F.fx + di, J * F.fy + dj, K * F.fz + dk, bf, xf);
  }
  set_rhs<T, Natural>(C, I, J, K, (T)(acc / mg_vol<T>(C, I, J, K)), bc, xc);
}

// b = r / jp on the finest level (r and jp in natural layout, b and x in Lay)
template <typename T, typename V, typename Lay>
__global__ void __launch_bounds__(256) mg_scale_kernel(MGView L, const V *__restrict__ r, const double *__restrict__ jp,
                                                       T *__restrict__ b, T *__restrict__ x, const KrylovScalars *ks) {
  if (ks && ks->done) return;
  const int k = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y * blockDim.y + threadIdx.y, i = blockIdx.z;
  if (k >= L.nz || j >= L.ny) return;
  const int64_t c = idx3(L, i, j, k);
  set_rhs<T, Lay>(L, i, j, k, (T)((double)r[c] / jp[c]), b, x);
}

template <typename T, typename V>
__global__ void __launch_bounds__(256) mg_widen_kernel(int64_t n, const T *__restrict__ x, V *__restrict__ out,
                                                       const KrylovScalars *ks) {
  if (ks && ks->done) return;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) out[t] = (V)x[t];
}

// 3-D launches (x: k or k2, y: j, z: i): no 64-bit index division per thread
template <typename T, typename Lay>
__global__ void __launch_bounds__(256) mg_rb_kernel(MGView L, int colour, const T *__restrict__ b, T *__restrict__ x,
                                                    const KrylovScalars *ks) {
  if (ks && ks->done) return;
  const int k2 = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y * blockDim.y + threadIdx.y, i = blockIdx.z;
  if (k2 >= (L.nz + 1) / 2 || j >= L.ny) return;
  rb_at<T, Lay>(L, i, j, k2, colour, b, x);
}

// planes of a colour-split level that one thread of a single sweep walks:
// at 4 the FP64 sweeps hold 72-112 VGPRs (4-7 waves a SIMD; 8 planes: 112-182,
// 2-4 waves), and the 512x256x64 multigrid steps ran 1-1.5% faster than at 8
// (2 planes: 5% slower)
constexpr int MG_PLANES = 4;

enum SplitSweep { SWEEP_PLAIN, SWEEP_PROLONG, SWEEP_OUT };

// One colour of a red-black sweep of the colour-split finest level.  Thread
// (k2, j) walks the planes i0 .. i0 + MG_PLANES - 1 (i0 = MG_PLANES
// blockIdx.z) and updates the cell of the colour at (i, j, k2) of each.  The
// other colour's entry at (i', j, k2), cen(i'), is loaded once: it is the -x
// neighbour of plane i' + 1, the +x neighbour of plane i' - 1 and one of the
// two k neighbours of plane i' (the other is the entry at k2 -+ 1).  The y
// and z coefficients are loaded once per thread (the z ones for both
// parities of k, which alternate from plane to plane), the x ones are
// plane-uniform.  The arithmetic is rb_at's, term for term.
//   SWEEP_PROLONG: the first red half-sweep after the coarse correction: the
//     neighbours are read as x + xc[parent], as in rb_prolong_at.
//   SWEEP_OUT: the last black half-sweep of the finest level (or of a
//     colour-split coarse level, whose natural copy the prolongation above
//     reads); it writes the new black value and the red one (its cen) to
//     out in natural layout, precision V.
template <typename T, typename V, int MODE, typename CLay = Natural>
__global__ void __launch_bounds__(256) mg_split_sweep_kernel(MGView L, MGView C, int colour, const T *__restrict__ b,
                                                             T *__restrict__ x, const T *__restrict__ xc,
                                                             V *__restrict__ out, const KrylovScalars *ks) {
  if (ks && ks->done) return;
  const int k2 = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y * blockDim.y + threadIdx.y;
  const int hz = (L.nz + 1) >> 1;
  if (k2 >= hz || j >= L.ny) return;
  const int i0 = blockIdx.z * MG_PLANES;
  const int64_t ns = (int64_t)L.nx * L.ny * hz, sx = (int64_t)L.ny * hz;
  T *__restrict__ own = x + (colour ? ns : 0);
  const T *__restrict__ oth = x + (colour ? 0 : ns);
  const T *__restrict__ bown = b + (colour ? ns : 0);
  const int64_t col = (int64_t)j * hz + k2;  // position of (0, j, k2) in a colour
  const bool hym = j > 0, hyp = j < L.ny - 1;
  const T cym = (T)L.ay[j], cyp = (T)L.ay[L.ny + j];
  const double dy = L.ay[2 * L.ny + j];
  T czm[2], czp[2];
  double dz[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int k = min(2 * k2 + e, L.nz - 1);  // the clamped entry of an absent cell is never used
    czm[e] = (T)L.az[k];
    czp[e] = (T)L.az[L.nz + k];
    dz[e] = L.az[2 * L.nz + k];
  }
  // the parent's indices along y and z of a neighbour at (j', k'); x is per plane
  auto par = [&](int ip, int jp, int kp) -> int64_t {
    return CLay::at(C, L.fx == 2 ? ip >> 1 : ip, L.fy == 2 ? jp >> 1 : jp, L.fz == 2 ? kp >> 1 : kp);
  };
  T cen[MG_PLANES + 2];
#pragma unroll
  for (int p = 0; p < MG_PLANES + 2; ++p) {
    const int ip = min(max(i0 - 1 + p, 0), L.nx - 1);  // clamped planes are never used
    cen[p] = oth[ip * sx + col];
    if (MODE == SWEEP_PROLONG) {
      // the other colour's cell at (ip, j, k2)
      const int kb = 2 * k2 + ((ip + j + colour + 1) & 1);
      cen[p] += xc[par(ip, j, min(kb, L.nz - 1))];
    }
  }
  // every plane's loads are issued before any result is stored (planes past
  // the grid and the padding slot of odd nz load clamped entries and store
  // nothing), so the wave has them all in flight at once
  T vym[MG_PLANES], vyp[MG_PLANES], side[MG_PLANES], bv[MG_PLANES];
#pragma unroll
  for (int p = 0; p < MG_PLANES; ++p) {
    const int i = min(i0 + p, L.nx - 1);
    const int e = (i + j + colour) & 1;
    const int k = min(2 * k2 + e, L.nz - 1);
    const int64_t h = i * sx + col;
    // the k neighbour that is not cen: k2 - 1 below an even k, k2 + 1 above
    // an odd one; across the periodic seam k2 = hz - 1 below k = 0 and
    // k2 = 0 above k = nz - 1
    const bool hside = L.wz || (e ? k < L.nz - 1 : k > 0);
    const int64_t hs = e ? (k < L.nz - 1 ? h + 1 : h - (hz - 1)) : (k > 0 ? h - 1 : h + (hz - 1));
    vym[p] = oth[hym ? h - hz : h];
    vyp[p] = oth[hyp ? h + hz : h];
    side[p] = oth[hside ? hs : h];
    bv[p] = bown[h];
    if (MODE == SWEEP_PROLONG) {
      vym[p] += xc[par(i, hym ? j - 1 : j, k)];
      vyp[p] += xc[par(i, hyp ? j + 1 : j, k)];
      side[p] += xc[par(i, j, hside ? (e ? kup(L, k) : kdn(L, k)) : k)];
    }
  }
#pragma unroll
  for (int p = 0; p < MG_PLANES; ++p) {
    const int i = i0 + p;
    const int e = (i + j + colour) & 1;
    const int k = 2 * k2 + e;
    if (MODE == SWEEP_OUT && i < L.nx && 2 * k2 + 1 - e < L.nz) out[idx3(L, i, j, 2 * k2 + 1 - e)] = (V)cen[p + 1];
    if (i >= L.nx || k >= L.nz) continue;
    const bool hxm = i > 0, hxp = i < L.nx - 1, hzm = L.wz || k > 0, hzp = L.wz || k < L.nz - 1;
    const T vzm = e ? cen[p + 1] : side[p], vzp = e ? side[p] : cen[p + 1];
    const T cxm = (T)L.ax[i], cxp = (T)L.ax[L.nx + i];
    T s = (T)0;
    s = hxm ? s + cxm * cen[p] : s;
    s = hxp ? s + cxp * cen[p + 2] : s;
    s = hym ? s + cym * vym[p] : s;
    s = hyp ? s + cyp * vyp[p] : s;
    s = hzm ? s + czm[e] * vzm : s;
    s = hzp ? s + czp[e] * vzp : s;
    const T v = (bv[p] + s) / (T)(L.ax[2 * L.nx + i] + dy + dz[e]);
    if (MODE == SWEEP_OUT)
      out[idx3(L, i, j, k)] = (V)v;
    else
      own[i * sx + col] = v;
  }
}

// ---- several half-sweeps of a colour-split level in one pass ---------------
//
// A half-sweep alone streams 12 B a cell (FP64) and, on the small levels, is
// a launch of 3-6 us whatever its size.  mg_fused_kernel runs NS of them in
// one pass: a workgroup owns a tile of rows (all of z) and a run of planes,
// marches along i, and at step t applies half-sweep 1 to plane t, half-sweep
// 2 to plane t - 1, ... NS to plane t - NS + 1.  Thread (row, k2) holds the
// column's entries of both colours; its x- and same-k2 neighbours are its
// own registers, the other three come from LDS, where every stage leaves its
// half-plane for the next step (two buffers, one barrier a step).  Tiles
// overlap by NS rows and planes: the overlap is computed twice instead of
// exchanged, so x is read from one buffer and written to another.  Loads run
// two (FP64: registers) or three planes ahead; the loop is unrolled by the length of the register
// rings, so their positions are fixed.  The arithmetic is rb_at's, term for
// term (an absent neighbour's coefficient is 0).
//
// What bounds a pass is latency on the small levels (8-14 us for 4
// half-sweeps, 4 launches of 3.5-6 us before) and, on the finest, the stages'
// chain of LDS reads and divisions: four half-sweeps of 512x256x64 take
// 40-51 us FP64 and 29-32 us FP32 (4 x 21 and 4 x 15 as single sweeps), at 30 B
// a cell 6.1 TB/s of FP64 traffic.  With a branch per stage the compiler
// drained every load before its use and an FP64 pass took 59-68 us.  One
// workgroup a CU: tiles of 24 rows and 23 planes at that size, each computing
// 32 x 29 instead, 1.7 times its cells (2.05 at 1024x512x128, 3.1 at
// 256x128x32, 3.5 at 200x104x40, 6 at 128x64x16), are what 256 CUs leave (two
// workgroups a CU, with twice the overlap: a cycle of 490 us against 422).
// Choosing tiles by waves and steps (fused_shape) instead of the fewest tiles of rows: 396 -> 386 us a
// cycle there, 159 -> 152 at 256x128x32, 151 -> 139 at 200x104x40.  Three timesteps
// there went from 73.9 to 57.2 ms (FP64; mixed 65.5 to 50.8), the 256x128x32
// adjoint from 110 to 83 ms.
//
// The cycle's first pass (SCL) forms the right-hand side r / jp from the
// natural-order vectors on the way in and starts from x = 0, so that neither a
// kernel that scales nor the first red half-sweep touches memory on its own:
// at 512x256x64 48 + 34 -> 66 us FP64, 46 + 25 -> 41 FP32, a cycle 422 -> 400
// and 303 -> 278.  It reads pairs of cells, so nz has to be even.
constexpr int FUSED_THREADS = 1024;
constexpr int FUSED_RING = 6;     // planes of x and b a thread holds
constexpr int FUSED_WAVES = 16, FUSED_START = 3;  // fused_shape's cost
constexpr int FUSED_CHUNK = 512;  // planes of a run at most (its coefficients sit in LDS)

struct FusedShape {
  int hz, R, TJ, njt, chunk, nci, halo;  // halo: rows beside a tile (0: one tile spans y)
};

// n / d, split so that the reciprocal of d is shared by the two divisions a cell
// of a pass makes.  FP64: the compiler's own operations on the same operands
// without its rescaling, so correctly rounded while d, 1 / d and n 2^-53 are
// normal numbers.  (Past that a grid's cells are shorter than 2^-510 or longer
// than 2^510, or n is below 2^-969, where the Krylov solver's dot products are
// zero.)
__device__ inline double div_recip(double d) {
  double y = __builtin_amdgcn_rcp(d);
  double e = fma(-d, y, 1.0);
  y = fma(y, e, y);
  e = fma(-d, y, 1.0);
  return fma(y, e, y);
}
__device__ inline double div_by(double n, double d, double y) {
  const double q = n * y;
  const double r = fma(-d, q, n);
  return __builtin_amdgcn_div_fixup(fma(r, y, q), d, n);
}
// FP32: reciprocal and product in FP64 are off by 2^-51 at most, and a quotient
// of two floats is at least 2^-49 away from the middle between two floats: the
// correctly rounded quotient over the whole exponent range.  (Split in FP32 like
// the other one it lost diagonals past 2^126 and below 2^-126, with a cycle of
// 270 us at 512x256x64 for 278 now; three timesteps there 43.3 -> 43.8 ms.)
__device__ inline double div_recip(float d) { return __builtin_amdgcn_div_fixup(div_recip((double)d), (double)d, 1.0); }
__device__ inline float div_by(float n, float, double y) { return (float)((double)n * y); }

// the column a thread of mg_fused_kernel owns and what it carries
// SCL: the pass forms the right-hand side r / jp itself (natural order, nz
// even), from x = 0, and leaves it in b
template <typename T, typename V>
struct FusedRhs {
  const V *r;
  const double *jp;
  T *b;
};

template <typename T, int NS>
struct FusedCol {
  T in[FUSED_RING], bA[FUSED_RING], bB[FUSED_RING];  // other colour before the pass; right-hand sides
  T st[NS][3];                                       // stage results of the last three planes
  double yA[3], yB[3];                               // 1 / diagonal of both colours
  T cym, cyp, czm[2], czp[2];
  double dy, dz[2];
  int side[2];  // LDS position of the k neighbour beside k2, by plane parity
  bool up[2];   // that neighbour is the +z one
};

template <typename T>
struct alignas(2 * sizeof(T)) CoefX {
  T m, p;  // to the -x and +x neighbour
};

template <typename T, typename V, int NS, int START, bool PRO, bool OUT, bool SCL = false>
__global__ void __launch_bounds__(FUSED_THREADS) mg_fused_kernel(MGView L, MGView C, FusedShape S,
                                                                 const T *__restrict__ b, const T *__restrict__ xin,
                                                                 T *__restrict__ xout, const T *__restrict__ xc,
                                                                 V *__restrict__ out, FusedRhs<T, V> R,
                                                                 const KrylovScalars *ks) {
  if (ks && ks->done) return;
  constexpr int PD = sizeof(T) == 8 || SCL ? 2 : 3;
  __shared__ T half[2][NS][FUSED_THREADS];
  __shared__ CoefX<T> cxl[FUSED_CHUNK + 2 * NS];
  __shared__ double dxl[FUSED_CHUNK + 2 * NS];
  const int tid = threadIdx.x, hz = S.hz;
  const int blk = pt_xcd_order((int)blockIdx.x, S.njt * S.nci);
  const int jt = blk % S.njt, ci = blk / S.njt;
  const int row = tid / hz, k2 = tid - row * hz;
  const int j = jt * S.TJ - S.halo + row;
  const int jc = min(max(j, 0), L.ny - 1);
  const bool store = row < S.R && j >= jt * S.TJ && j < min((jt + 1) * S.TJ, L.ny);
  const int i0 = ci * S.chunk, i1 = min(i0 + S.chunk, L.nx);
  const int ta = max(i0 - (NS - 1), 0), te = i1 - 1 + (NS - 1);
  const int64_t ns = (int64_t)L.nx * L.ny * hz;
  const int sx = L.ny * hz, at = jc * hz + k2;
  const T *__restrict__ xo = xin + (START ? 0 : ns);  // the colour the first half-sweep reads
  const T *__restrict__ bA = b + (START ? ns : 0), *__restrict__ bB = b + (START ? 0 : ns);
  // a plane's base is uniform, a thread's place in it 32 bits
  const unsigned atb = (unsigned)at * (unsigned)sizeof(T);
  auto in_plane = [&](const T *p, int plane) {
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(p + (int64_t)plane * sx) + atb);
  };
  // per-plane coefficients ta .. min(te, nx - 1)
  const int npl = min(te, L.nx - 1) - ta + 1;
  for (int q = tid; q < npl; q += (int)blockDim.x) {
    cxl[q] = CoefX<T>{(T)L.ax[ta + q], (T)L.ax[L.nx + ta + q]};
    dxl[q] = L.ax[2 * L.nx + ta + q];
  }
  FusedCol<T, NS> c;
  c.cym = (T)L.ay[jc];
  c.cyp = (T)L.ay[L.ny + jc];
  c.dy = L.ay[2 * L.ny + jc];
  // the START colour at plane ta + n has k = 2 k2 + e, e = (ta + n + j + START) & 1;
  // index q of the parity arrays: n & 1 for that colour, the other for the other
  bool pad[2];  // k is past an odd nz (never read: the entry is 0 and its result unused)
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int e = (ta + q + jc + START) & 1;
    const int k = min(2 * k2 + e, L.nz - 1);
    pad[q] = 2 * k2 + e >= L.nz;
    c.czm[q] = (T)L.az[k];
    c.czp[q] = (T)L.az[L.nz + k];
    c.dz[q] = L.az[2 * L.nz + k];
    c.up[q] = e;
    const int ks2 = e ? (k2 + 1 < hz ? k2 + 1 : (L.wz ? 0 : k2)) : (k2 > 0 ? k2 - 1 : (L.wz ? hz - 1 : k2));
    c.side[q] = tid + (ks2 - k2);
  }
  if (row >= S.R) c.side[0] = c.side[1] = tid;
  const int im = row > 0 ? tid - hz : tid, ip = row + 1 < S.R ? tid + hz : tid;
  // SCL: the right-hand side's pair of cells at a plane, r and jp as they come
  typedef V V2 __attribute__((ext_vector_type(2)));
  typedef double D2 __attribute__((ext_vector_type(2)));
  V2 rr[3];
  D2 rj[3];
  const unsigned pair = (unsigned)(jc * L.nz + 2 * k2);
  auto load_pair = [&](int s, int plane) {
    const int64_t o = (int64_t)min(max(plane, 0), L.nx - 1) * L.ny * L.nz;
    rr[s] = *reinterpret_cast<const V2 *>(reinterpret_cast<const char *>(R.r + o) + pair * (unsigned)sizeof(V));
    rj[s] = *reinterpret_cast<const D2 *>(reinterpret_cast<const char *>(R.jp + o) + pair * 8u);
  };
  auto load_in = [&](int plane, int q) -> T {  // q: parity index of the other colour at that plane
    if (SCL) return (T)0;
    plane = min(max(plane, 0), L.nx - 1);
    T v = in_plane(xo, plane);
    if (PRO) {
      const int k = min(2 * k2 + (c.up[q] ? 1 : 0), L.nz - 1);
      const unsigned pb = (unsigned)((L.fy == 2 ? jc >> 1 : jc) * C.nz + (L.fz == 2 ? k >> 1 : k)) * (unsigned)sizeof(T);
      const T *pl = xc + (int64_t)(L.fx == 2 ? plane >> 1 : plane) * C.ny * C.nz;
      v += *reinterpret_cast<const T *>(reinterpret_cast<const char *>(pl) + pb);
    }
    return pad[q] ? (T)0 : v;
  };
  auto load_b = [&](const T *__restrict__ p, int plane, int q) -> T {
    const T v = in_plane(p, min(max(plane, 0), L.nx - 1));
    return pad[q] ? (T)0 : v;
  };
  // ring positions: plane ta + m of x at (m + 1) mod 6, of b at m mod 6
#pragma unroll
  for (int m = -1; m <= PD; ++m) c.in[m + 1] = load_in(ta + m, (m + 1) & 1);
  if (SCL) {
#pragma unroll
    for (int m = 0; m < FUSED_RING; ++m) c.bA[m] = c.bB[m] = (T)0;
#pragma unroll
    for (int m = 0; m < PD; ++m) load_pair(m, ta + m);
  } else {
#pragma unroll
    for (int m = 0; m < PD; ++m) c.bA[m] = load_b(bA, ta + m, m & 1);
#pragma unroll
    for (int m = 0; m < PD - 1; ++m) c.bB[m] = load_b(bB, ta + m, (m + 1) & 1);
#pragma unroll
    for (int m = PD; m < FUSED_RING; ++m) c.bA[m] = c.bB[m] = (T)0;
    c.bB[PD - 1] = (T)0;
  }
#pragma unroll
  for (int m = PD + 2; m < FUSED_RING; ++m) c.in[m] = (T)0;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    c.yA[q] = c.yB[q] = 1.0;
#pragma unroll
    for (int s = 0; s < NS; ++s) c.st[s][q] = (T)0;
  }
  half[1][0][tid] = c.in[1];  // plane ta, as if left by the step before the first
#pragma unroll
  for (int s = 1; s < NS; ++s) half[1][s][tid] = (T)0;  // planes before ta: read, never needed
  __syncthreads();

  // A step has no branches: every stage runs, on planes it need not do as
  // well (they feed only such planes, and values finite but unused: a
  // coefficient across the grid's end is 0), and every load is issued with
  // its plane clamped, so that the waits count loads instead of draining
  // them and the stages' LDS reads overlap.
  const int ilast = npl - 1;
  const unsigned outb = (unsigned)(jc * L.nz + 2 * k2) * (unsigned)sizeof(V);
  auto step = [&](auto uc, int n) {
    constexpr int u = decltype(uc)::value;  // n mod 6
    constexpr int q = u & 1;                // parity index of every stage's colour at its plane
    const T(*prev)[FUSED_THREADS] = half[(u + 1) & 1];
    T(*cur)[FUSED_THREADS] = half[u & 1];
    // loads of the planes PD ahead of their first use
    c.in[(u + 2 + PD) % 6] = load_in(min(ta + n + 1 + PD, te + 1), (u + PD) & 1);
    if (SCL) {
      load_pair((u + PD) % 3, min(ta + n + PD, te));
      // b of plane ta + n, mg_scale_kernel's
      const T b0 = (T)((double)rr[u % 3].x / rj[u % 3].x), b1 = (T)((double)rr[u % 3].y / rj[u % 3].y);
      c.bA[u] = c.up[q] ? b1 : b0;
      c.bB[u] = c.up[q] ? b0 : b1;
      if (ta + n >= i0 && ta + n < i1 && store) {
        char *o = reinterpret_cast<char *>(R.b + (int64_t)(ta + n) * sx);
        *reinterpret_cast<T *>(o + (START ? ns * (int64_t)sizeof(T) : 0) + atb) = c.bA[u];
        *reinterpret_cast<T *>(o + (START ? 0 : ns * (int64_t)sizeof(T)) + atb) = c.bB[u];
      }
      if (sizeof(T) == 8) __builtin_amdgcn_sched_barrier(0);
    } else {
      c.bA[(u + PD) % 6] = load_b(bA, min(ta + n + PD, te), (u + PD) & 1);
      c.bB[(u + PD - 1) % 6] = load_b(bB, min(ta + n + PD - 1, te), (u + PD) & 1);
    }
    // a stage's LDS reads are issued before the stage ahead of it is computed,
    // and not earlier (all at once they take registers that FP64 lacks)
    T vym[NS], vyp[NS], vs[NS];
    CoefX<T> cx[NS];
    auto fetch = [&](int s) {  // stage s works on plane ta + n - s
      vym[s] = prev[s][im];
      vyp[s] = prev[s][ip];
      vs[s] = prev[s][c.side[q]];
      cx[s] = cxl[min(max(n - s, 0), ilast)];
    };
    if (!SCL) fetch(0);  // SCL: the first stage's neighbours are zero
    const double dx0 = dxl[min(n, ilast)], dx1 = dxl[min(max(n - 1, 0), ilast)];
    double dx2 = 0.0, dx3 = 0.0;
    if (sizeof(T) == 8) {  // div_by's diagonal, added again instead of held
      dx2 = dxl[min(max(n - 2, 0), ilast)];
      if (NS > 3) dx3 = dxl[min(max(n - 3, 0), ilast)];
    }
    c.yA[u % 3] = div_recip((T)(dx0 + c.dy + c.dz[q]));
    c.yB[(u + 2) % 3] = div_recip((T)(dx1 + c.dy + c.dz[q]));
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      if (s + 1 < NS) fetch(s + 1 < NS ? s + 1 : 0);
      if (sizeof(T) == 8) __builtin_amdgcn_sched_barrier(0);
      // ring positions mod 3 of the planes ta + n - s - 1, ta + n - s, ta + n - s + 1
      const int r0 = (u + 6 - s) % 3, rm = (u + 5 - s) % 3, rp = (u + 7 - s) % 3;
      const T xm = s == 0 ? c.in[u % 6] : c.st[s > 0 ? s - 1 : 0][rm];
      const T x0 = s == 0 ? c.in[(u + 1) % 6] : c.st[s > 0 ? s - 1 : 0][r0];
      const T xp = s == 0 ? c.in[(u + 2) % 6] : c.st[s > 0 ? s - 1 : 0][rp];
      const T bv = (s & 1) ? c.bB[(u + 6 - s) % 6] : c.bA[(u + 6 - s) % 6];
      const T d = (T)((s == 0 ? dx0 : s == 1 ? dx1 : s == 2 ? dx2 : dx3) + c.dy + c.dz[q]);
      const double y = (s & 1) ? c.yB[r0] : c.yA[r0];
      T v = (T)0;
      if (!SCL || s > 0) {
        v = fma(cx[s].m, xm, (T)0);
        v = fma(cx[s].p, xp, v);
        v = fma(c.cym, vym[s], v);
        v = fma(c.cyp, vyp[s], v);
        const T v1 = c.up[q] ? x0 : vs[s], v2 = c.up[q] ? vs[s] : x0;  // -z, +z
        v = fma(c.czm[q], v1, v);
        v = fma(c.czp[q], v2, v);
      }
      c.st[s][r0] = div_by(bv + v, d, y);
      if (s + 1 < NS) cur[s + 1 < NS ? s + 1 : 0][tid] = c.st[s][r0];
    }
    if (!SCL) cur[0][tid] = c.in[(u + 2) % 6];
    // the pass's result of plane ta + n - NS + 1: the last half-sweep's colour and the other
    const int p = ta + n - (NS - 1);
    if (p >= i0 && p < i1 && store) {
      constexpr int rf = (u + 6 - (NS - 1)) % 3;
      const T last = c.st[NS - 1][rf], other = c.st[NS - 2][rf];
      if (OUT) {
        char *o = reinterpret_cast<char *>(out + (int64_t)p * L.ny * L.nz) + outb;
        reinterpret_cast<V *>(o)[0] = (V)(c.up[q] ? other : last);
        if (2 * k2 + 1 < L.nz) reinterpret_cast<V *>(o)[1] = (V)(c.up[q] ? last : other);
      } else {
        constexpr int lastc = (NS & 1) ? START : 1 - START;
        char *o = reinterpret_cast<char *>(xout + (int64_t)p * sx);
        *reinterpret_cast<T *>(o + (lastc ? ns * (int64_t)sizeof(T) : 0) + atb) = last;
        *reinterpret_cast<T *>(o + (lastc ? 0 : ns * (int64_t)sizeof(T)) + atb) = other;
      }
    }
    __syncthreads();
  };
  const int nst = te - ta + 1;
  for (int n = 0; n < nst; n += 6) {
    step(std::integral_constant<int, 0>{}, n);
    if (n + 1 < nst) step(std::integral_constant<int, 1>{}, n + 1);
    if (n + 2 < nst) step(std::integral_constant<int, 2>{}, n + 2);
    if (n + 3 < nst) step(std::integral_constant<int, 3>{}, n + 3);
    if (n + 4 < nst) step(std::integral_constant<int, 4>{}, n + 4);
    if (n + 5 < nst) step(std::integral_constant<int, 5>{}, n + 5);
  }
}

// Restriction from the colour-split finest level when every axis is halved.
// The children of (I, J, K) are the entries at position K of the four (i, j)
// columns 2I..2I+1 x 2J..2J+1, one of each colour per column (k = 2K and
// 2K + 1).  The kernel loads those pairs, the pairs of the eight columns
// beside them and the single entries below (2K - 1) and above (2K + 2) each
// column (40 loads for 8 children, with b), and sums the children's
// residuals in restrict_at's order with child_res's arithmetic.  Bound by its
// instructions (three quarters of the VALU's cycles in FP32): with the 40
// addresses formed from uniform plane bases and six offsets 512x256x64 takes
// 33.8 us FP64 and 20.9 FP32, from indexes of their own 36.7 and 25.  Four
// waves a SIMD instead of three spill (49.5 and 43.6 us).
template <typename T, typename CLay = Natural>
__global__ void __launch_bounds__(256) mg_restrict_split_kernel(MGView F, MGView C, const T *__restrict__ bf,
                                                                const T *__restrict__ xf, T *__restrict__ bc,
                                                                T *__restrict__ xc, const KrylovScalars *ks) {
  if (ks && ks->done) return;
  const int K = blockIdx.x * blockDim.x + threadIdx.x, J = blockIdx.y * blockDim.y + threadIdx.y, I = blockIdx.z;
  if (K >= C.nz || J >= C.ny) return;
  const int hz = F.nz >> 1;  // nz is even where z is halved
  const int64_t ns = (int64_t)F.nx * F.ny * hz;
  // The entry at k = 2 KK + m of column (2I - 1 + a, 2J - 1 + c) is in colour
  // half (a + c + m) & 1: a plane's base is uniform, a thread's place in it one
  // of six 32-bit offsets.  Columns outside the grid are clamped into it (KK
  // wraps across the periodic seam); what they load is not used.
  const int Km = K > 0 ? K - 1 : F.wz ? hz - 1 : 0, Kp = K < hz - 1 ? K + 1 : F.wz ? 0 : hz - 1;
  unsigned row[4], rkm[2], rkp[2];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int j = min(max(2 * J - 1 + c, 0), F.ny - 1);
    row[c] = (unsigned)(j * hz + K) * (unsigned)sizeof(T);
    if (c == 1 || c == 2) {
      rkm[c - 1] = (unsigned)(j * hz + Km) * (unsigned)sizeof(T);
      rkp[c - 1] = (unsigned)(j * hz + Kp) * (unsigned)sizeof(T);
    }
  }
  auto ld = [&](const T *f, int a, int half, unsigned off) -> T {
    const int i = min(max(2 * I - 1 + a, 0), F.nx - 1);
    const T *base = f + ((half & 1) ? ns : 0) + (int64_t)i * F.ny * hz;
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + off);
  };
  // X[a][c] = the pair of column (2I - 1 + a, 2J - 1 + c): the four children's
  // columns (a, c in 1..2) and the eight beside them (no corners)
  T X[4][4][2], B[2][2][2], xkm[2][2], xkp[2][2];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int m = 0; m < 2; ++m)
        X[a][c][m] = ((a == 0 || a == 3) && (c == 0 || c == 3)) ? (T)0 : ld(xf, a, a + c + m, row[c]);
#pragma unroll
  for (int di = 0; di < 2; ++di)
#pragma unroll
    for (int dj = 0; dj < 2; ++dj) {
      B[di][dj][0] = ld(bf, di + 1, di + dj, row[dj + 1]);
      B[di][dj][1] = ld(bf, di + 1, di + dj + 1, row[dj + 1]);
      xkm[di][dj] = ld(xf, di + 1, di + dj + 1, rkm[dj]);  // k = 2K - 1
      xkp[di][dj] = ld(xf, di + 1, di + dj, rkp[dj]);      // k = 2K + 2
    }
  double acc = 0.0;
#pragma unroll
  for (int d = 0; d < 8; ++d) {
    const int di = d >> 2, dj = (d >> 1) & 1, m = d & 1;
    const int i = 2 * I + di, j = 2 * J + dj, k = 2 * K + m;
    const Has h = has6(F, i, j, k);
    const Coef6<T> a = coef6<T>(F, i, j, k);
    const T xv = X[di + 1][dj + 1][m];
    const T vzm = m ? X[di + 1][dj + 1][0] : xkm[di][dj], vzp = m ? xkp[di][dj] : X[di + 1][dj + 1][1];
    T s = (T)0;
    s = h.xm ? s + a.xm * X[di][dj + 1][m] : s;
    s = h.xp ? s + a.xp * X[di + 2][dj + 1][m] : s;
    s = h.ym ? s + a.ym * X[di + 1][dj][m] : s;
    s = h.yp ? s + a.yp * X[di + 1][dj + 2][m] : s;
    s = h.zm ? s + a.zm * vzm : s;
    s = h.zp ? s + a.zp * vzp : s;
    const T r = B[di][dj][m] - (mg_diag<T>(F, i, j, k) * xv - s);
    acc += mg_vol<T>(F, i, j, k) * (double)r;
  }
  set_rhs<T, CLay>(C, I, J, K, (T)(acc / mg_vol<T>(C, I, J, K)), bc, xc);
}

template <typename T, typename Lay>
__global__ void __launch_bounds__(256) mg_rb_prolong_kernel(MGView F, MGView C, const T *__restrict__ b,
                                                            T *__restrict__ x, const T *__restrict__ xc,
                                                            const KrylovScalars *ks) {
  if (ks && ks->done) return;
  const int k2 = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y * blockDim.y + threadIdx.y, i = blockIdx.z;
  if (k2 >= (F.nz + 1) / 2 || j >= F.ny) return;
  rb_prolong_at<T, Lay>(F, C, i, j, k2, b, x, xc);
}

template <typename T, typename Lay>
__global__ void __launch_bounds__(256) mg_restrict_kernel(MGView F, MGView C, const T *__restrict__ bf,
                                                          const T *__restrict__ xf, T *__restrict__ bc,
                                                          T *__restrict__ xc, const KrylovScalars *ks) {
  if (ks && ks->done) return;
  const int K = blockIdx.x * blockDim.x + threadIdx.x, J = blockIdx.y * blockDim.y + threadIdx.y, I = blockIdx.z;
  if (K >= C.nz || J >= C.ny) return;
  restrict_at<T, Lay>(F, C, I, J, K, bf, xf, bc, xc);
}

// ---- the bottom of the V-cycle (levels of at most MG_SMALL cells) ----------
//
// One workgroup, one launch; __syncthreads separates the half-sweeps.  What
// bounds it is the length of a half-sweep's chain: about 35 of them follow
// each other whatever the levels' sizes.  So a thread keeps what a half-sweep
// needs of its cells (at most BOTTOM_CELLS of each colour: neighbour
// positions, coefficients, diagonal and its reciprocal, right-hand side) in
// registers for as long as the workgroup works on a level; the levels' x, the
// right-hand sides handed down, the residuals and the axis arrays are in LDS.
// A half-sweep is then six LDS reads, their sum, a division and a barrier.
// 512x256x64's bottom (2048, 256 and 64 cells, 30 half-sweeps and a dense
// solve) takes 21.9 us FP64 against 48.8 for the cell-by-cell form that
// read coefficients from memory and split indices by division in every
// half-sweep; 96 half-sweeps of a 1625-cell coarsest level 26.3 against 110.
constexpr int BOTTOM_THREADS = 1024;
constexpr int BOTTOM_CELLS = (int)(MG_SMALL / 2 / BOTTOM_THREADS);
static_assert(BOTTOM_CELLS * 2 * BOTTOM_THREADS == MG_SMALL, "a thread's cells");
constexpr size_t BOTTOM_LDS = 156 * 1024;  // of a CU's 160 KB
constexpr int DENSE_PF = 4;  // dense-inverse entries a thread prefetches: a 64-cell inverse

template <typename T>
struct SmallArgs {
  int nlev, nu, coarse_sweeps, dense;
  // the bottom kernel's LDS: doubles, then elements of T
  int coef_off[MG_MAX_LEVELS];  // level l's axis arrays
  int x_off[MG_MAX_LEVELS];     // its x, its b behind it
  int t_base, res_off, stage_off, staged;
  MGView v[MG_MAX_LEVELS];
  T *x[MG_MAX_LEVELS];
  T *b[MG_MAX_LEVELS];
  const T *cinv;  // dense inverse of the coarsest operator, column-major, when dense
};

// fills the LDS positions; the bytes to launch the bottom kernel with (0: the
// levels do not fit a workgroup)
template <typename T>
size_t bottom_layout(SmallArgs<T> &S) {
  if (S.v[0].n > MG_SMALL) return 0;
  size_t dbl = 0, elems = 0;
  for (int l = 0; l < S.nlev; ++l) {
    S.coef_off[l] = (int)dbl;
    dbl += 4 * (size_t)(S.v[l].nx + S.v[l].ny + S.v[l].nz);
    S.x_off[l] = (int)elems;
    elems += 2 * (size_t)S.v[l].n;
    // an odd nz leaves threads without a cell: more of them than there are
    if ((int64_t)S.v[l].nx * S.v[l].ny * ((S.v[l].nz + 1) / 2) > BOTTOM_CELLS * BOTTOM_THREADS) return 0;
  }
  S.t_base = (int)dbl;
  S.res_off = (int)elems;
  if (S.nlev > 1) elems += (size_t)S.v[0].n;
  S.stage_off = (int)elems;
  S.staged = 0;
  if (dbl * sizeof(double) + elems * sizeof(T) > BOTTOM_LDS) return 0;
  const size_t nn = (size_t)(S.v[S.nlev - 1].n * S.v[S.nlev - 1].n);
  if (S.dense && nn <= (size_t)DENSE_PF * BOTTOM_THREADS &&
      dbl * sizeof(double) + (elems + nn) * sizeof(T) <= BOTTOM_LDS) {
    S.staged = 1;
    elems += nn;
  }
  return dbl * sizeof(double) + elems * sizeof(T);
}

// a level as the bottom kernel sees it: axis arrays in LDS
struct BottomLevel {
  int nx, ny, nz, n, wz;
  const double *ax, *ay, *az;
  __device__ double diag(int i, int j, int k) const { return ax[2 * nx + i] + ay[2 * ny + j] + az[2 * nz + k]; }
  __device__ double vol(int i, int j, int k) const { return ax[3 * nx + i] * ay[3 * ny + j] * az[3 * nz + k]; }
};

// one cell of a thread: LDS positions (two to a register), coefficients in
// rb_at's order (an absent neighbour is the cell itself with coefficient 0)
template <typename T>
struct BottomCell {
  unsigned cn, x, y, z;  // own position | parent's; -x | +x; -y | +y; -z | +z
  T a[6], d, b;          // coefficients, diagonal, right-hand side
  double r;              // the diagonal's reciprocal
  bool on;

  __device__ T off(const T *xl) const {
    const T vxm = xl[x & 0xffff], vxp = xl[x >> 16], vym = xl[y & 0xffff], vyp = xl[y >> 16], vzm = xl[z & 0xffff],
            vzp = xl[z >> 16];
    T s = fma(a[0], vxm, (T)0);
    s = fma(a[1], vxp, s);
    s = fma(a[2], vym, s);
    s = fma(a[3], vyp, s);
    s = fma(a[4], vzm, s);
    return fma(a[5], vzp, s);
  }
};

template <typename T>
__global__ void __launch_bounds__(BOTTOM_THREADS) mg_bottom_kernel(SmallArgs<T> S, const KrylovScalars *ks) {
  if (ks && ks->done) return;
  extern __shared__ __align__(16) double bottom_lds[];
  const int tid = threadIdx.x;
  T *const lds = reinterpret_cast<T *>(bottom_lds + S.t_base);
  T *const res = lds + S.res_off;
  auto X = [&](int l) { return lds + S.x_off[l]; };
  auto B = [&](int l) { return lds + S.x_off[l] + (int)S.v[l].n; };
  auto level = [&](int l) {
    const MGView &v = S.v[l];
    const double *c = bottom_lds + S.coef_off[l];
    return BottomLevel{v.nx, v.ny, v.nz, (int)v.n, v.wz, c, c + 4 * v.nx, c + 4 * (v.nx + v.ny)};
  };
  // the first level's x and b, the axis arrays and a small dense inverse: one
  // round trip to memory for all of them
  constexpr int CP = (int)(MG_SMALL / BOTTOM_THREADS);
  const int n0 = (int)S.v[0].n, last = S.nlev - 1;
  T xv[CP], bv[CP], pf[DENSE_PF];
#pragma unroll
  for (int u = 0; u < CP; ++u) {
    const int t = tid + u * BOTTOM_THREADS;
    xv[u] = t < n0 ? S.x[0][t] : (T)0;
    bv[u] = t < n0 ? S.b[0][t] : (T)0;
  }
  const int nn = S.staged ? (int)(S.v[last].n * S.v[last].n) : 0;
#pragma unroll
  for (int u = 0; u < DENSE_PF; ++u) {
    const int e = tid + u * BOTTOM_THREADS;
    pf[u] = e < nn ? S.cinv[e] : (T)0;
  }
  for (int l = 0; l < S.nlev; ++l) {
    const int nc = 4 * (S.v[l].nx + S.v[l].ny + S.v[l].nz);
    for (int q = tid; q < nc; q += BOTTOM_THREADS) bottom_lds[S.coef_off[l] + q] = S.v[l].ax[q];
  }
#pragma unroll
  for (int u = 0; u < CP; ++u) {
    const int t = tid + u * BOTTOM_THREADS;
    if (t < n0) {
      X(0)[t] = xv[u];
      B(0)[t] = bv[u];
    }
  }
#pragma unroll
  for (int u = 0; u < DENSE_PF; ++u) {
    const int e = tid + u * BOTTOM_THREADS;
    if (e < nn) lds[S.stage_off + e] = pf[u];
  }
  __syncthreads();

  // nsw sweeps of level l.  skip_red0: the first red half-sweep is done;
  // correct: level l + 1's correction goes into the black cells first (the red
  // ones are overwritten); restrict_to: the residual into res at the end.
  // C: cells of a colour a thread owns.
  auto visit = [&](auto cc, int l, int nsw, bool skip_red0, bool correct, bool residual)
                   __attribute__((always_inline)) {
    constexpr int C = decltype(cc)::value;
    const BottomLevel L = level(l);
    T *const xl = X(l);
    const T *const bl = B(l);
    const int hz = (L.nz + 1) / 2, sx = L.ny * L.nz, cnt = L.nx * L.ny * hz;
    const MGView &F = S.v[l];
    BottomCell<T> cell[2][C];
#pragma unroll
    for (int m = 0; m < C; ++m) {
      const int t = tid + m * BOTTOM_THREADS;
      const int q = min(t, cnt - 1) / hz, k2 = min(t, cnt - 1) - q * hz, i = q / L.ny, j = q - i * L.ny;
#pragma unroll
      for (int colour = 0; colour < 2; ++colour) {
        BottomCell<T> &e = cell[colour][m];
        const int kk = 2 * k2 + ((i + j + colour) & 1), k = min(kk, L.nz - 1);
        e.on = t < cnt && kk < L.nz;
        const int o = (i * L.ny + j) * L.nz + k;
        const int zm = k > 0 ? o - 1 : L.wz ? o + (L.nz - 1) : o, zp = k < L.nz - 1 ? o + 1 : L.wz ? o - (L.nz - 1) : o;
        int par = 0;
        if (correct)
          par = ((F.fx == 2 ? i >> 1 : i) * S.v[l + 1].ny + (F.fy == 2 ? j >> 1 : j)) * S.v[l + 1].nz +
                (F.fz == 2 ? k >> 1 : k);
        e.cn = (unsigned)o | (unsigned)par << 16;
        e.x = (unsigned)(i > 0 ? o - sx : o) | (unsigned)(i < L.nx - 1 ? o + sx : o) << 16;
        e.y = (unsigned)(j > 0 ? o - L.nz : o) | (unsigned)(j < L.ny - 1 ? o + L.nz : o) << 16;
        e.z = (unsigned)zm | (unsigned)zp << 16;
        e.a[0] = (T)L.ax[i];
        e.a[1] = (T)L.ax[L.nx + i];
        e.a[2] = (T)L.ay[j];
        e.a[3] = (T)L.ay[L.ny + j];
        e.a[4] = (T)L.az[k];
        e.a[5] = (T)L.az[L.nz + k];
        e.d = (T)L.diag(i, j, k);
        e.r = div_recip(e.d);
        e.b = bl[o];
      }
    }
    if (correct) {
#pragma unroll
      for (int m = 0; m < C; ++m)
        if (cell[1][m].on) xl[cell[1][m].cn & 0xffff] += X(l + 1)[cell[1][m].cn >> 16];
      __syncthreads();
    }
    for (int s = 0; s < nsw; ++s) {
#pragma unroll
      for (int colour = 0; colour < 2; ++colour) {
        if (s == 0 && colour == 0 && skip_red0) continue;
#pragma unroll
        for (int m = 0; m < C; ++m) {
          const BottomCell<T> &e = cell[colour][m];
          const T v = div_by(e.b + e.off(xl), e.d, e.r);
          if (e.on) xl[e.cn & 0xffff] = v;
        }
        __syncthreads();
      }
    }
    if (residual) {
#pragma unroll
      for (int colour = 0; colour < 2; ++colour)
#pragma unroll
        for (int m = 0; m < C; ++m) {
          const BottomCell<T> &e = cell[colour][m];
          const T r = e.b - fma(e.d, xl[e.cn & 0xffff], -e.off(xl));
          if (e.on) res[e.cn & 0xffff] = r;
        }
      __syncthreads();
    }
  };
  // down to the coarsest level and up again
#pragma unroll 1
  for (int ph = 0; ph <= 2 * last; ++ph) {
    const bool down = ph < last, up = ph > last;
    const int l = up ? 2 * last - ph : ph;
    if (ph == last && S.dense) {
      // x = A^-1 b, a row a thread, summed over the columns in order
      const int n = (int)S.v[last].n;
      const T *const bl = B(last);
      T *const xl = X(last);
      if (tid < n) {
        double acc = 0.0;
        if (S.staged) {
          const T *const inv = lds + S.stage_off + tid;
          for (int q = 0; q < n; ++q) acc += (double)inv[q * n] * (double)bl[q];
        } else {
          for (int q = 0; q < n; ++q) acc += (double)S.cinv[(int64_t)q * n + tid] * (double)bl[q];
        }
        xl[tid] = (T)acc;
      }
      __syncthreads();
      continue;
    }
    const int nsw = ph == last ? S.coarse_sweeps : S.nu;
    if (S.v[l].nx * S.v[l].ny * ((S.v[l].nz + 1) / 2) <= BOTTOM_THREADS)
      visit(std::integral_constant<int, 1>{}, l, nsw, !up, up, down);
    else
      visit(std::integral_constant<int, BOTTOM_CELLS>{}, l, nsw, !up, up, down);
    if (!down) continue;
    // the children's residuals, volume-weighted, and the first red half-sweep (set_rhs)
    const BottomLevel F = level(l), C = level(l + 1);
    const int fx = S.v[l].fx, fy = S.v[l].fy, fz = S.v[l].fz;
    for (int t = tid; t < C.n; t += BOTTOM_THREADS) {
      const int K = t % C.nz, q = t / C.nz, J = q % C.ny, I = q / C.ny;
      double acc = 0.0;
      for (int di = 0; di < fx; ++di)
        for (int dj = 0; dj < fy; ++dj)
          for (int dk = 0; dk < fz; ++dk) {
            const int i = I * fx + di, j = J * fy + dj, k = K * fz + dk;
            acc = fma(F.vol(i, j, k), (double)res[(i * F.ny + j) * F.nz + k], acc);
          }
      const T bc = (T)(acc / C.vol(I, J, K));
      B(l + 1)[t] = bc;
      X(l + 1)[t] = ((I + J + K) & 1) == 0 ? bc / (T)C.diag(I, J, K) : (T)0;
    }
    __syncthreads();
  }
  for (int t = tid; t < n0; t += BOTTOM_THREADS) S.x[0][t] = X(0)[t];
}

// The same on levels that a workgroup's LDS does not hold (a coarsest level
// that never halves below MG_SMALL cells): cell by cell, x and b in memory.
constexpr int MG_SMALL_THREADS = 512;

template <typename T>
__global__ void __launch_bounds__(MG_SMALL_THREADS) mg_small_kernel(SmallArgs<T> S, const KrylovScalars *ks) {
  if (ks && ks->done) return;
  const int nt = MG_SMALL_THREADS;
  // nsw sweeps of level l; skip_red0: the first red half-sweep is done;
  // prolong_from >= 0: the first red half-sweep folds in that level's correction
  auto sweep = [&](int l, int nsw, bool skip_red0, int prolong_from) {
    const MGView &L = S.v[l];
    const int half = (L.nz + 1) / 2;
    const int cnt = L.nx * L.ny * half;
    for (int s = 0; s < nsw; ++s)
      for (int colour = 0; colour < 2; ++colour) {
        if (s == 0 && colour == 0 && skip_red0) continue;
        const bool fold = s == 0 && colour == 0 && prolong_from >= 0;
        for (int t = threadIdx.x; t < cnt; t += nt) {
          const int k2 = t % half, r = t / half;
          if (fold)
            rb_prolong_at<T, Natural>(L, S.v[prolong_from], r / L.ny, r % L.ny, k2, S.b[l], S.x[l], S.x[prolong_from]);
          else
            rb_at<T, Natural>(L, r / L.ny, r % L.ny, k2, colour, S.b[l], S.x[l]);
        }
        __syncthreads();
      }
  };
  const int last = S.nlev - 1;
  for (int l = 0; l < last; ++l) {
    sweep(l, S.nu, true, -1);
    const MGView &C = S.v[l + 1];
    for (int t = threadIdx.x; t < (int)C.n; t += nt) {
      const int K = t % C.nz, r = t / C.nz;
      restrict_at<T, Natural>(S.v[l], C, r / C.ny, r % C.ny, K, S.b[l], S.x[l], S.b[l + 1], S.x[l + 1]);
    }
    __syncthreads();
  }
  if (S.dense) {
    // consecutive threads read consecutive entries of a column
    const int n = (int)S.v[last].n;
    for (int t = threadIdx.x; t < n; t += nt) {
      double acc = 0.0;
      for (int q = 0; q < n; ++q) acc += (double)S.cinv[(int64_t)q * n + t] * (double)S.b[last][q];
      S.x[last][t] = (T)acc;
    }
    __syncthreads();
  } else {
    sweep(last, S.coarse_sweeps, true, -1);
  }
  for (int l = last - 1; l >= 0; --l) sweep(l, S.nu, false, l + 1);
}

// launch shape of a 3-D kernel over (nk, ny, nx) with 256-thread blocks
struct Shape3 {
  dim3 grid, block;
};
Shape3 shape3(int nk, int ny, int nx) {
  int bx = 1;
  while (bx < nk && bx < 64) bx <<= 1;
  const int by = 256 / bx;
  Shape3 s;
  s.block = dim3(bx, by, 1);
  s.grid = dim3((nk + bx - 1) / bx, (ny + by - 1) / by, nx);
  return s;
}

// tiles of mg_fused_kernel on a level; R = 0 where a line is too long for a
// workgroup to hold rows beside each other (nz > 128)
FusedShape fused_shape(const MGView &v, int ns) {
  FusedShape s{};
  s.hz = (v.nz + 1) / 2;
  const int rmax = FUSED_THREADS / s.hz;
  if (rmax < 4 * ns) return s;
  // As many tiles as leave one workgroup a CU, split between rows and planes
  // for the least time: a step takes about FUSED_WAVES + the waves of a
  // workgroup (latency and instructions; fitted to the passes of 512x256x64,
  // its levels, 256x128x32 and 200x104x40), and a run of `chunk` planes takes
  // chunk + 2 (ns - 1) steps and some for its start.
  const int fewest = v.ny <= rmax ? 1 : (v.ny + rmax - 2 * ns - 1) / (rmax - 2 * ns);
  int64_t best = INT64_MAX;
  for (int njt = fewest; njt < fewest + 64 && njt <= v.ny; ++njt) {
    FusedShape t = s;
    t.njt = njt;
    t.TJ = (v.ny + njt - 1) / njt;
    t.halo = njt > 1 ? ns : 0;
    t.R = t.TJ + 2 * t.halo;
    if (t.R > rmax || (njt - 1) * t.TJ >= v.ny) continue;
    const int runs = std::max(1, 256 / njt);
    t.chunk = std::min((v.nx + runs - 1) / runs, FUSED_CHUNK);
    t.nci = (v.nx + t.chunk - 1) / t.chunk;
    const int64_t rounds = ((int64_t)njt * t.nci + 255) / 256;
    const int64_t cost = rounds * ((t.R * t.hz + 63) / 64 + FUSED_WAVES) * (t.chunk + 2 * (ns - 1) + FUSED_START);
    if (cost < best) {
      best = cost;
      s = t;
    }
  }
  return s;
}

// whether the sweeps of a colour-split level run as fused passes
bool fused_passes(const MGView &v, int nu) { return nu >= 2 && fused_shape(v, 4).R > 0; }

template <typename T, typename V, int NS, int START, bool PRO, bool OUT>
void launch_fused(const MGView &v, const MGView &C, const T *b, const T *xin, T *xout, const T *xc, V *out,
                  const KrylovScalars *ks, hipStream_t st) {
  const FusedShape s = fused_shape(v, NS);
  const int threads = (s.R * s.hz + 63) / 64 * 64;
  mg_fused_kernel<T, V, NS, START, PRO, OUT>
      <<<s.njt * s.nci, threads, 0, st>>>(v, C, s, b, xin, xout, xc, out, FusedRhs<T, V>{}, ks);
}

// the first four half-sweeps from x = 0 with the right-hand side r / jp
template <typename T, typename V>
void launch_fused_scaled(const MGView &v, const V *r, const double *jp, T *b, T *xout, const KrylovScalars *ks,
                         hipStream_t st) {
  const FusedShape s = fused_shape(v, 4);
  const int threads = (s.R * s.hz + 63) / 64 * 64;
  mg_fused_kernel<T, V, 4, 0, false, false, true><<<s.njt * s.nci, threads, 0, st>>>(
      v, v, s, b, nullptr, xout, nullptr, nullptr, FusedRhs<T, V>{r, jp, b}, ks);
}

int nblk(int64_t n) { return blocks_for(n, 256, 1 << 30); }

template <typename T>
T *lx(MGLevel &L);
template <>
double *lx<double>(MGLevel &L) { return L.x64; }
template <>
float *lx<float>(MGLevel &L) { return L.x32; }
template <typename T>
T *lxn(MGLevel &L);
template <>
double *lxn<double>(MGLevel &L) { return L.xn64; }
template <>
float *lxn<float>(MGLevel &L) { return L.xn32; }
template <typename T>
T *lxb(MGLevel &L);
template <>
double *lxb<double>(MGLevel &L) { return L.xb64; }
template <>
float *lxb<float>(MGLevel &L) { return L.xb32; }
template <typename T>
T *lb(MGLevel &L);
template <>
double *lb<double>(MGLevel &L) { return L.b64; }
template <>
float *lb<float>(MGLevel &L) { return L.b32; }

// level l's kernels in layout Lay
template <typename T, typename Lay>
struct LevelOps {
  template <typename V>
  static void scale_from(const MGView &v, const V *r, const double *jp, T *b, T *x, const KrylovScalars *ks,
                         hipStream_t st) {
    const Shape3 sh = shape3(v.nz, v.ny, v.nx);
    mg_scale_kernel<T, V, Lay><<<sh.grid, sh.block, 0, st>>>(v, r, jp, b, x, ks);
  }
  static void rb(const MGView &v, int colour, const T *b, T *x, const KrylovScalars *ks, hipStream_t st) {
    const Shape3 sh = shape3((v.nz + 1) / 2, v.ny, v.nx);
    mg_rb_kernel<T, Lay><<<sh.grid, sh.block, 0, st>>>(v, colour, b, x, ks);
  }
  static void rb_prolong(const MGView &v, const MGView &C, const T *b, T *x, const T *xc, const KrylovScalars *ks,
                         hipStream_t st) {
    const Shape3 sh = shape3((v.nz + 1) / 2, v.ny, v.nx);
    mg_rb_prolong_kernel<T, Lay><<<sh.grid, sh.block, 0, st>>>(v, C, b, x, xc, ks);
  }
  static void restrict_to(const MGView &v, const MGView &C, const T *b, const T *x, T *bc, T *xc,
                          const KrylovScalars *ks, hipStream_t st) {
    const Shape3 sh = shape3(C.nz, C.ny, C.nx);
    mg_restrict_kernel<T, Lay><<<sh.grid, sh.block, 0, st>>>(v, C, b, x, bc, xc, ks);
  }
};

// out = V-cycle(L, r / jp): the cycle runs in T, the vectors r and out are V
// (an FP32 cycle inside an FP64 Krylov solve widens its result at the end).
// When the finest level is smoothed by the level kernels (the cycle has more
// than the one-workgroup bottom), its x and b are colour-split and its last
// black half-sweep writes out; otherwise the bottom kernel works on out
// directly (or on x, widened into out).
template <typename T, typename V>
int mg_apply(Ctx &c, const V *r, V *out, const KrylovScalars *ks) {
  MGState &M = *c.mg;
  const int nl = (int)M.lv.size();
  const int ls = M.small_from;
  const bool split = ls > 0;
  T *b0 = lb<T>(M.lv[0]);
  constexpr bool same = std::is_same<T, V>::value;
  T *x0 = (same && !split) ? reinterpret_cast<T *>(out) : lx<T>(M.lv[0]);
  if (!b0 || !x0) return fail(CFD_ERR_STATE, "multigrid buffers of this precision are not allocated");
  auto X = [&](int l) { return l == 0 ? x0 : lx<T>(M.lv[l]); };
  const MGView &v0 = M.lv[0].v;
  const bool scaled = split && v0.nz % 2 == 0 && fused_passes(v0, M.nu) &&
                      reinterpret_cast<uintptr_t>(r) % (2 * sizeof(V)) == 0;
  if (scaled)
    launch_fused_scaled<T, V>(v0, r, c.f[CFD_JP], b0, x0, ks, c.stream);
  else if (split)
    LevelOps<T, ColourSplit>::scale_from(M.lv[0].v, r, c.f[CFD_JP], b0, x0, ks, c.stream);
  else
    LevelOps<T, Natural>::scale_from(M.lv[0].v, r, c.f[CFD_JP], b0, x0, ks, c.stream);
  // nu sweeps of level l: pre-smoothing skips the red half-sweep its
  // right-hand side's producer did; post-smoothing folds the prolongation
  // into its first red half-sweep, and on a colour-split level ends in the
  // half-sweep that writes out (or the level's natural copy)
  T *xs[MG_MAX_LEVELS] = {};  // the buffer that holds a colour-split level's x
  for (int l = 0; l < M.split_levels; ++l) xs[l] = X(l);
  auto correction = [&](int l) { return l + 1 < M.split_levels ? lxn<T>(M.lv[l + 1]) : X(l + 1); };
  auto single = [&](int l, int colour, int mode) {
    const MGView &v = M.lv[l].v, &C = M.lv[l + 1].v;
    Shape3 sh = shape3((v.nz + 1) / 2, v.ny, v.nx);
    sh.grid.z = (v.nx + MG_PLANES - 1) / MG_PLANES;
    T *bl = l == 0 ? b0 : lb<T>(M.lv[l]);
    if (mode == SWEEP_PROLONG)
      mg_split_sweep_kernel<T, T, SWEEP_PROLONG><<<sh.grid, sh.block, 0, c.stream>>>(v, C, 0, bl, xs[l], correction(l),
                                                                                    nullptr, ks);
    else if (mode == SWEEP_OUT && l > 0)  // the natural copy the level above reads
      mg_split_sweep_kernel<T, T, SWEEP_OUT><<<sh.grid, sh.block, 0, c.stream>>>(v, C, 1, bl, xs[l], nullptr,
                                                                                lxn<T>(M.lv[l]), ks);
    else if (mode == SWEEP_OUT)
      mg_split_sweep_kernel<T, V, SWEEP_OUT><<<sh.grid, sh.block, 0, c.stream>>>(v, C, 1, bl, xs[l], nullptr, out, ks);
    else
      mg_split_sweep_kernel<T, T, SWEEP_PLAIN><<<sh.grid, sh.block, 0, c.stream>>>(v, C, colour, bl, xs[l], nullptr,
                                                                                  nullptr, ks);
  };
  // passes of up to four half-sweeps (mg_fused_kernel); what is left over
  // (one before, two after for an odd nu) runs as single half-sweeps
  auto smooth_fused = [&](int l, bool pre) {
    const MGView &v = M.lv[l].v, &C = M.lv[l + 1].v;
    const T *bl = l == 0 ? b0 : lb<T>(M.lv[l]);
    T *other = xs[l] == X(l) ? lxb<T>(M.lv[l]) : X(l);
    auto swap = [&] { std::swap(xs[l], other); };
    T *const none = nullptr;
    if (pre && l == 0 && scaled) {
      int left = 2 * M.nu - 4;  // red first
      for (; left >= 4; left -= 4) {
        launch_fused<T, T, 4, 0, false, false>(v, C, bl, xs[l], other, none, none, ks, c.stream);
        swap();
      }
      if (left == 2) {
        single(l, 0, SWEEP_PLAIN);
        single(l, 1, SWEEP_PLAIN);
      }
      return;
    }
    if (pre) {
      int left = 2 * M.nu - 1;  // black first
      for (; left >= 4; left -= 4) {
        launch_fused<T, T, 4, 1, false, false>(v, C, bl, xs[l], other, none, none, ks, c.stream);
        swap();
      }
      if (left == 3) {
        launch_fused<T, T, 3, 1, false, false>(v, C, bl, xs[l], other, none, none, ks, c.stream);
        swap();
      } else if (left == 1) {
        single(l, 1, SWEEP_PLAIN);
      }
      return;
    }
    const T *xc = correction(l);
    int left = 2 * M.nu - 4;
    if (left == 0) {  // nu = 2: prolongation to result in one pass
      if (l > 0)
        launch_fused<T, T, 4, 0, true, true>(v, C, bl, xs[l], other, xc, lxn<T>(M.lv[l]), ks, c.stream);
      else
        launch_fused<T, V, 4, 0, true, true>(v, C, bl, xs[l], other, xc, out, ks, c.stream);
      return;
    }
    launch_fused<T, T, 4, 0, true, false>(v, C, bl, xs[l], other, xc, none, ks, c.stream);
    swap();
    for (; left > 4; left -= 4) {
      launch_fused<T, T, 4, 0, false, false>(v, C, bl, xs[l], other, none, none, ks, c.stream);
      swap();
    }
    if (left == 4) {
      if (l > 0)
        launch_fused<T, T, 4, 0, false, true>(v, C, bl, xs[l], other, none, lxn<T>(M.lv[l]), ks, c.stream);
      else
        launch_fused<T, V, 4, 0, false, true>(v, C, bl, xs[l], other, none, out, ks, c.stream);
    } else {
      single(l, 0, SWEEP_PLAIN);
      single(l, 1, SWEEP_OUT);
    }
  };
  auto smooth = [&](int l, bool pre) {
    const MGView &v = M.lv[l].v;
    if (l < M.split_levels && fused_passes(v, M.nu)) {
      smooth_fused(l, pre);
      return;
    }
    for (int s = 0; s < M.nu; ++s)
      for (int colour = 0; colour < 2; ++colour) {
        const bool first = s == 0 && colour == 0, last = s == M.nu - 1 && colour == 1;
        if (first && pre) continue;
        if (l < M.split_levels) {
          single(l, colour, first ? SWEEP_PROLONG : last && !pre ? SWEEP_OUT : SWEEP_PLAIN);
        } else {
          using Ops = LevelOps<T, Natural>;
          if (first)
            Ops::rb_prolong(v, M.lv[l + 1].v, lb<T>(M.lv[l]), X(l), X(l + 1), ks, c.stream);
          else
            Ops::rb(v, colour, lb<T>(M.lv[l]), X(l), ks, c.stream);
        }
      }
  };
  for (int l = 0; l < ls; ++l) {
    smooth(l, true);
    const MGView &F = M.lv[l].v;
    const bool fsplit = l < M.split_levels;
    T *bf = l == 0 ? b0 : lb<T>(M.lv[l]);
    if (fsplit && F.fx == 2 && F.fy == 2 && F.fz == 2) {
      const MGView &C = M.lv[l + 1].v;
      const Shape3 sh = shape3(C.nz, C.ny, C.nx);
      if (l + 1 < M.split_levels)  // the coarse right-hand side in its colour-split layout
        mg_restrict_split_kernel<T, ColourSplit><<<sh.grid, sh.block, 0, c.stream>>>(
            F, C, bf, xs[l], lb<T>(M.lv[l + 1]), X(l + 1), ks);
      else
        mg_restrict_split_kernel<T><<<sh.grid, sh.block, 0, c.stream>>>(F, C, bf, xs[l], lb<T>(M.lv[l + 1]),
                                                                        X(l + 1), ks);
    } else if (fsplit)  // a colour-split level into a natural one, cell by cell
      LevelOps<T, ColourSplit>::restrict_to(F, M.lv[l + 1].v, bf, xs[l], lb<T>(M.lv[l + 1]), X(l + 1), ks, c.stream);
    else
      LevelOps<T, Natural>::restrict_to(M.lv[l].v, M.lv[l + 1].v, lb<T>(M.lv[l]), X(l), lb<T>(M.lv[l + 1]),
                                        X(l + 1), ks, c.stream);
  }
  SmallArgs<T> S;
  std::memset(&S, 0, sizeof(S));
  S.nlev = nl - ls;
  S.nu = M.nu;
  S.coarse_sweeps = MG_COARSE_SWEEPS;
  S.dense = M.dense_n > 0 ? 1 : 0;
  S.cinv = std::is_same<T, double>::value ? reinterpret_cast<const T *>(M.cinv64) : reinterpret_cast<const T *>(M.cinv32);
  for (int l = ls; l < nl; ++l) {
    S.v[l - ls] = M.lv[l].v;
    S.x[l - ls] = X(l);
    S.b[l - ls] = lb<T>(M.lv[l]);
  }
  const size_t lds_bytes = bottom_layout(S);
  if (lds_bytes) {  // at most BOTTOM_LDS, which mg_ensure has asked for
    mg_bottom_kernel<T><<<1, BOTTOM_THREADS, lds_bytes, c.stream>>>(S, ks);
  } else {
    mg_small_kernel<T><<<1, MG_SMALL_THREADS, 0, c.stream>>>(S, ks);
  }
  for (int l = ls - 1; l >= 0; --l) smooth(l, false);
  if (!same && !split) mg_widen_kernel<T, V><<<nblk(c.g.N), 256, 0, c.stream>>>(c.g.N, x0, out, ks);
  CFD_HIP(hipGetLastError());
  return CFD_OK;
}

// per-axis level arrays from widths w (n) and the centre distances of the
// finest level (ds_lo: centre of cell i-1 to i, for i = 0 the ghost
// distance; ds_hi: centre of i to i+1, for i = n-1 the ghost distance)
// (periodic: the end cells keep their coefficient to the neighbour across
// the seam, whose distances dlo[0] and dhi[n-1] give)
void axis_arrays(const std::vector<double> &w, const std::vector<double> &dlo, const std::vector<double> &dhi,
                 bool dir_lo, bool dir_hi, std::vector<double> &out, bool periodic = false) {
  const size_t n = w.size();
  out.assign(4 * n, 0.0);
  for (size_t i = 0; i < n; ++i) {
    const double xm = 1.0 / w[i] / dlo[i], xp = 1.0 / w[i] / dhi[i];
    out[i] = (i > 0 || periodic) ? xm : 0.0;
    out[n + i] = (i + 1 < n || periodic) ? xp : 0.0;
    out[2 * n + i] = ((i > 0 || dir_lo || periodic) ? xm : 0.0) + ((i + 1 < n || dir_hi || periodic) ? xp : 0.0);
    out[3 * n + i] = w[i];
  }
}

}  // namespace

void mg_release(Ctx &c) {
  if (!c.mg) return;
  for (auto &L : c.mg->lv) {
    mg_free(L.coef);
    mg_free(L.x64);
    mg_free(L.b64);
    mg_free(L.x32);
    mg_free(L.b32);
    mg_free(L.xn64);
    mg_free(L.xn32);
    mg_free(L.xb64);
    mg_free(L.xb32);
  }
  mg_free(c.mg->cinv64);
  mg_free(c.mg->cinv32);
  delete c.mg;
  c.mg = nullptr;
  mg_free(c.ph64);
  mg_free(c.sh64);
  mg_free(c.ph32);
  mg_free(c.sh32);
}

// builds the hierarchy (once) and the buffers of the requested precision
int mg_ensure(Ctx &c, bool fp32) {
  if (!c.mg) {
    for (const void *k : {reinterpret_cast<const void *>(mg_bottom_kernel<double>),
                          reinterpret_cast<const void *>(mg_bottom_kernel<float>)})
      CFD_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)BOTTOM_LDS));
    MGState *M = new MGState();
    c.mg = M;
    const int nc[3] = {c.g.nxc, c.g.nyc, c.g.nzc};
    const std::vector<double> *Dh[3] = {&c.hDx, &c.hDy, &c.hDz}, *Dsh[3] = {&c.hDxs, &c.hDys, &c.hDzs};
    std::vector<double> w[3], dlo[3], dhi[3];
    for (int a = 0; a < 3; ++a) {
      for (int q = 0; q < nc[a]; ++q) {
        const int I = q + GC;
        w[a].push_back((*Dh[a])[I]);
        dlo[a].push_back((*Dsh[a])[I - 1]);
        dhi[a].push_back((*Dsh[a])[I]);
      }
    }
    // periodic z: every level wraps in z (the fine level's seam coefficient
    // is the operator's, from the ghost distances Dzs)
    const bool pz = c.prm.periodic_z != 0;
    const bool dl[3] = {c.prm.p_dirichlet[0] != 0, c.prm.p_dirichlet[2] != 0, !pz && c.prm.p_dirichlet[4] != 0};
    const bool dh[3] = {c.prm.p_dirichlet[1] != 0, c.prm.p_dirichlet[3] != 0, !pz && c.prm.p_dirichlet[5] != 0};
    std::vector<double> last_arr[3];
    for (;;) {
      MGLevel L;
      L.v.nx = (int)w[0].size();
      L.v.ny = (int)w[1].size();
      L.v.nz = (int)w[2].size();
      L.v.n = (int64_t)L.v.nx * L.v.ny * L.v.nz;
      L.v.wz = pz ? 1 : 0;
      std::vector<double> arr[3], all;
      for (int a = 0; a < 3; ++a) {
        axis_arrays(w[a], dlo[a], dhi[a], dl[a], dh[a], arr[a], a == 2 && pz);
        all.insert(all.end(), arr[a].begin(), arr[a].end());
        last_arr[a] = arr[a];
      }
      int rc = mg_alloc(&L.coef, all.size());
      if (rc) return rc;
      CFD_HIP(hipMemcpy(L.coef, all.data(), all.size() * sizeof(double), hipMemcpyHostToDevice));
      L.v.ax = L.coef;
      L.v.ay = L.coef + 4 * L.v.nx;
      L.v.az = L.coef + 4 * L.v.nx + 4 * L.v.ny;
      int f[3];
      for (int a = 0; a < 3; ++a) f[a] = (w[a].size() % 2 == 0 && w[a].size() >= 4) ? 2 : 1;
      if (pz && (w[2].size() / 2) % 2 != 0) f[2] = 1;  // periodic z stays even
      const bool more = (f[0] > 1 || f[1] > 1 || f[2] > 1) && L.v.n > 64 && (int)M->lv.size() < MG_MAX_LEVELS - 1;
      L.v.fx = more ? f[0] : 1;
      L.v.fy = more ? f[1] : 1;
      L.v.fz = more ? f[2] : 1;
      M->lv.push_back(L);
      if (!more) break;
      // merged widths; centre distances from the widths, mirror ghosts at Dirichlet faces
      for (int a = 0; a < 3; ++a) {
        if (f[a] == 1) continue;
        std::vector<double> wc;
        for (size_t q = 0; q < w[a].size(); q += 2) wc.push_back(w[a][q] + w[a][q + 1]);
        const size_t n = wc.size();
        std::vector<double> lo(n), hi(n);
        const double seam = 0.5 * (wc[n - 1] + wc[0]);  // centre distance across a periodic seam
        for (size_t q = 0; q < n; ++q) {
          lo[q] = q > 0 ? 0.5 * (wc[q - 1] + wc[q]) : (a == 2 && pz ? seam : wc[q]);
          hi[q] = q + 1 < n ? 0.5 * (wc[q] + wc[q + 1]) : (a == 2 && pz ? seam : wc[q]);
        }
        w[a] = wc;
        dlo[a] = lo;
        dhi[a] = hi;
      }
    }
    M->small_from = (int)M->lv.size() - 1;
    while (M->small_from > 0 && M->lv[M->small_from - 1].v.n <= MG_SMALL) M->small_from--;
    // the finest level is colour-split whenever it has level kernels; each
    // next one is too while the level above halves every axis (its split
    // restriction then writes the coarse right-hand side in that layout)
    M->split_levels = M->small_from > 0 ? 1 : 0;
    while (M->split_levels < M->small_from) {
      const MGView &P = M->lv[M->split_levels - 1].v;
      if (!(P.fx == 2 && P.fy == 2 && P.fz == 2)) break;
      M->split_levels++;
    }
    // exact coarsest solve: the dense inverse of the coarsest operator when a
    // Dirichlet face makes it nonsingular (all-Neumann keeps the sweeps)
    const MGView &Lc = M->lv.back().v;
    const bool any_dir = dl[0] || dl[1] || dl[2] || dh[0] || dh[1] || dh[2];
    if (any_dir && Lc.n <= 512) {
      const int n = (int)Lc.n, nx = Lc.nx, ny = Lc.ny, nz = Lc.nz;
      std::vector<double> A((size_t)n * n, 0.0), Inv((size_t)n * n, 0.0);
      const std::vector<double> &ax = last_arr[0], &ay = last_arr[1], &az = last_arr[2];
      for (int i = 0; i < nx; ++i)
        for (int j = 0; j < ny; ++j)
          for (int k = 0; k < nz; ++k) {
            const int r = (i * ny + j) * nz + k;
            A[(size_t)r * n + r] = ax[2 * nx + i] + ay[2 * ny + j] + az[2 * nz + k];
            if (i > 0) A[(size_t)r * n + r - ny * nz] -= ax[i];
            if (i < nx - 1) A[(size_t)r * n + r + ny * nz] -= ax[nx + i];
            if (j > 0) A[(size_t)r * n + r - nz] -= ay[j];
            if (j < ny - 1) A[(size_t)r * n + r + nz] -= ay[ny + j];
            // z neighbours, across the seam with periodic z (with nz = 2 both
            // couplings of a cell reach the same neighbour and add)
            if (k > 0 || Lc.wz) A[(size_t)r * n + r - k + (k > 0 ? k - 1 : nz - 1)] -= az[k];
            if (k < nz - 1 || Lc.wz) A[(size_t)r * n + r - k + (k < nz - 1 ? k + 1 : 0)] -= az[nz + k];
          }
      for (int r = 0; r < n; ++r) Inv[(size_t)r * n + r] = 1.0;
      bool ok = true;
      for (int col = 0; col < n && ok; ++col) {  // Gauss-Jordan with partial pivoting
        int piv = col;
        for (int r = col + 1; r < n; ++r)
          if (std::fabs(A[(size_t)r * n + col]) > std::fabs(A[(size_t)piv * n + col])) piv = r;
        if (!(std::fabs(A[(size_t)piv * n + col]) > 0.0)) { ok = false; break; }
        if (piv != col)
          for (int q = 0; q < n; ++q) {
            std::swap(A[(size_t)piv * n + q], A[(size_t)col * n + q]);
            std::swap(Inv[(size_t)piv * n + q], Inv[(size_t)col * n + q]);
          }
        const double d = A[(size_t)col * n + col];
        for (int q = 0; q < n; ++q) { A[(size_t)col * n + q] /= d; Inv[(size_t)col * n + q] /= d; }
        for (int r = 0; r < n; ++r) {
          if (r == col) continue;
          const double f = A[(size_t)r * n + col];
          if (f == 0.0) continue;
          for (int q = 0; q < n; ++q) {
            A[(size_t)r * n + q] -= f * A[(size_t)col * n + q];
            Inv[(size_t)r * n + q] -= f * Inv[(size_t)col * n + q];
          }
        }
      }
      if (ok) {
        // column-major: the kernel's threads (one per row) read a column together
        std::vector<double> InvT((size_t)n * n);
        for (int r = 0; r < n; ++r)
          for (int q = 0; q < n; ++q) InvT[(size_t)q * n + r] = Inv[(size_t)r * n + q];
        Inv.swap(InvT);
        std::vector<float> inv32(Inv.begin(), Inv.end());
        int rc = mg_alloc(&M->cinv64, Inv.size());
        if (!rc) rc = mg_alloc(&M->cinv32, inv32.size());
        if (rc) return rc;
        CFD_HIP(hipMemcpy(M->cinv64, Inv.data(), Inv.size() * sizeof(double), hipMemcpyHostToDevice));
        CFD_HIP(hipMemcpy(M->cinv32, inv32.data(), inv32.size() * sizeof(float), hipMemcpyHostToDevice));
        M->dense_n = n;
      }
    }
    M->nu = c.prm.mg_nu > 0 ? c.prm.mg_nu : 4;
    for (auto &L : M->lv) M->shape += std::to_string(L.v.nx) + "x" + std::to_string(L.v.ny) + "x" +
                                      std::to_string(L.v.nz) + " ";
  }
  MGState &M = *c.mg;
  M.nu = c.prm.mg_nu > 0 ? c.prm.mg_nu : 4;
  for (size_t l = 0; l < M.lv.size(); ++l) {
    MGLevel &L = M.lv[l];
    // colour-split vectors hold nx ny ceil(nz / 2) cells per colour
    const bool sp = (int)l < M.split_levels;
    const size_t n = sp ? (size_t)L.v.nx * L.v.ny * (2 * ((L.v.nz + 1) / 2)) : (size_t)L.v.n;
    const bool nat = sp && l > 0;  // a split level below the finest keeps a natural copy of x
    const bool second = sp && fused_passes(L.v, M.nu);
    int rc = CFD_OK;
    if (fp32) {
      if (!L.b32 && (rc = mg_alloc(&L.b32, n))) return rc;
      if (!L.x32 && (rc = mg_alloc(&L.x32, n))) return rc;
      if (nat && !L.xn32 && (rc = mg_alloc(&L.xn32, (size_t)L.v.n))) return rc;
      if (second && !L.xb32 && (rc = mg_alloc(&L.xb32, n))) return rc;
    } else {
      if (!L.b64 && (rc = mg_alloc(&L.b64, n))) return rc;
      if (!L.x64 && (rc = mg_alloc(&L.x64, n))) return rc;
      if (nat && !L.xn64 && (rc = mg_alloc(&L.xn64, (size_t)L.v.n))) return rc;
      if (second && !L.xb64 && (rc = mg_alloc(&L.xb64, n))) return rc;
    }
  }
  const size_t N = (size_t)c.g.N;
  int rc = CFD_OK;
  if (fp32) {
    if ((!c.ph32 && (rc = mg_alloc(&c.ph32, N))) || (!c.sh32 && (rc = mg_alloc(&c.sh32, N)))) return rc;
  } else {
    if ((!c.ph64 && (rc = mg_alloc(&c.ph64, N))) || (!c.sh64 && (rc = mg_alloc(&c.sh64, N)))) return rc;
  }
  return CFD_OK;
}

int mg_apply64(Ctx &c, const double *r, double *out, const KrylovScalars *ks) {
  return mg_apply<double, double>(c, r, out, ks);
}
int mg_apply32(Ctx &c, const float *r, float *out, const KrylovScalars *ks) { return mg_apply<float, float>(c, r, out, ks); }
int mg_apply64_fp32cycle(Ctx &c, const double *r, double *out, const KrylovScalars *ks) {
  return mg_apply<float, double>(c, r, out, ks);
}

const char *mg_shape(const Ctx &c) { return c.mg ? c.mg->shape.c_str() : ""; }

}  // namespace cfd
