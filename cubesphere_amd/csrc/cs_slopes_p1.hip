// cs_slopes_p1.hip -- the reference's second-order zone reconstruction
// LIMIT_ALL_SLOPES_P1 (cubesphere/400riemann_integrate/410limit_all_slopes_p1.f:9)
// for one patch on the GPU, FP64, behind cs_limit_all_slopes_p1.
//
// The patch arrays keep the reference's column-major layouts (first index
// fastest), so a thread per zone or face reads consecutive addresses along x.
// Each kernel is one dependency level of the routine:
//   k_prim        steps 2 and 5: constants, higher modes cleared, tri-corner
//                 zones made safe, CONS_TO_PRIM, magnetosonic speed
//   k_face_zero   step 2 (faces): face B between two inactive zones cleared
//   k_tricorner   step 3: face B synchronised at the tri-corners
//   k_flat_a/b/c  step 6.a-c: velocity-divergence flattener, its pressure-
//                 ratio extension, its spread to the six neighbours
//   k_weno9       step 7.a: multi-D WENO of the 8 primitives and the entropy,
//                 one thread per three fields of a zone
//   k_pos         step 7.b: ENFORCE_PRESSURE_POSITIVITY_PRIM (440...f)
//   k_face_pts    step 8.a-c: normal B at the five B-field points of each face
//   k_clsq_e      step 8.d and 9.a: ADP constrained least squares for the 12
//                 linear B coefficients; zone E = -v x B
//   k_weno9       step 9.b: WENO of E (the same kernel, three fields)
//   k_diag(+final) step 10: min/max of the primitives, face-B divergence
//
// The constrained least squares of 8.d (the reference assembles the 18 x 18
// KKT matrix and factors it with Numerical Recipes' LU) is adp_clsq, with six
// of the twelve unknowns eliminated.
//
// The positivity limiter of the reference runs in loop order and, when a zone
// fails every reduction, also zeroes its entropy mean (440...f:553-600), which
// later zones of the loop then see in their entropy range.  k_pos runs all
// zones with the incoming entropy means and flags the zones that fail
// completely; when any do, the zones with such a neighbour earlier in the
// loop order (k_cands) are recomputed (k_replay) with the means of the flagged
// earlier zones taken as zero, repeating until the flags no longer change; a
// zone flagged for the first time in a sweep brings its later neighbours onto
// the list before the next sweep (the dependence only runs forward in the
// loop order, so this reaches the sequential result), and the flagged means
// are then cleared.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <type_traits>
#include <vector>

#include "cs_physics.h"
#include "cs_p1_common.h"
#include "../../include/cubesphere_hip.h"

namespace cs {
void set_error(const char* fmt, ...);
}

using namespace csp;

namespace csp1 {

struct P1 {
  cs_p1_patch a;
  int N, NR, g, nz, nzr, nf, nfr;
  int64_t NZ, NXF, NZF, NFC;

  __device__ __forceinline__ int64_t zi(int i, int j, int k) const {
    return (int64_t)(i - 1 + g) + (int64_t)nz * ((j - 1 + g) + (int64_t)nz * (k - 1 + g));
  }
  __device__ __forceinline__ int64_t fci(int i, int j, int k) const {
    return (int64_t)(i + g) + (int64_t)nf * ((j + g) + (int64_t)nf * (k + g));
  }
  __device__ __forceinline__ int64_t xfi(int i, int j, int k) const {
    return (int64_t)(i + g) + (int64_t)nf * ((j - 1 + g) + (int64_t)nz * (k - 1 + g));
  }
  __device__ __forceinline__ int64_t yfi(int i, int j, int k) const {
    return (int64_t)(i - 1 + g) + (int64_t)nz * ((j + g) + (int64_t)nf * (k - 1 + g));
  }
  __device__ __forceinline__ int64_t zfi(int i, int j, int k) const {
    return (int64_t)(i - 1 + g) + (int64_t)nz * ((j - 1 + g) + (int64_t)nz * (k + g));
  }
  // stencil entry n (R L U D RR LL UU DD RU LU LD RD) of zone column (i, j),
  // clamped to the zone range so that no table entry can address outside it
  __device__ __forceinline__ void nbr(int i, int j, int n, int& ni, int& nj) const {
    const int64_t s = (int64_t)(i - 1 + g) + (int64_t)nz * (j - 1 + g), plane = (int64_t)nz * nz;
    ni = min(max(a.stencil[s + plane * (2 * n)], 1 - g), N + g);
    nj = min(max(a.stencil[s + plane * (2 * n + 1)], 1 - g), N + g);
  }
  __device__ __forceinline__ bool active(int i, int j, int k) const { return a.mask[zi(i, j, k)] == 1; }
  __device__ __forceinline__ double V(int c, int m, int64_t z) const { return a.V[z + NZ * (c + 8 * m)]; }
  __device__ __forceinline__ double& Vr(int c, int m, int64_t z) const { return a.V[z + NZ * (c + 8 * m)]; }
  __device__ __forceinline__ double& Ur(int c, int m, int64_t z) const { return a.U[z + NZ * (c + 8 * m)]; }
  __device__ __forceinline__ double obl(int64_t z) const { return 1.0 / fmax(a.scale[z], a.smallnum); }
  __device__ __forceinline__ double cen(int64_t z, int c) const { return a.v_centroid[z + NZ * c]; }
};

// a box of zone or face indices, decoded from a flat thread index
struct Box {
  int i0, j0, k0, ni, nj, nk;
  __device__ __forceinline__ bool decode(int64_t t, int& i, int& j, int& k) const {
    if (t >= (int64_t)ni * nj * nk) return false;
    i = i0 + (int)(t % ni);
    j = j0 + (int)((t / ni) % nj);
    k = k0 + (int)(t / ((int64_t)ni * nj));
    return true;
  }
  __host__ __device__ int64_t count() const { return (int64_t)ni * nj * nk; }
};
static Box make_box(int i0, int i1, int j0, int j1, int k0, int k1) {
  return Box{i0, j0, k0, i1 - i0 + 1, j1 - j0 + 1, k1 - k0 + 1};
}

__device__ __forceinline__ int64_t tid() { return (int64_t)blockIdx.x * blockDim.x + threadIdx.x; }

// ---------------------------------------------------------------------------
// step 7.b, the positivity limiter (pos_zone)
// sweep < 0: every zone of the range with the incoming entropy means; sets its
// flags and counts the zones whose slopes were removed.
// sweep >= 0: a zone of the replay list (those with a flagged zone earlier in
// the loop order among their 27), taking the entropy means of the earlier
// zones flagged by the sweep before as zero; sets its flag for the next sweep
// and counts the zones whose flag changed.
constexpr int kMaxSweeps = 256;  // the replay has to settle within these
constexpr int kSweepBatch = 4;   // sweeps put on the stream between two looks of the host
struct Flags {
  uint8_t* fl[2];          // [zone]: sweep n reads fl[n % 2] and writes fl[(n + 1) % 2]
  uint8_t *ever, *inlist;  // [zone]: flagged in the first pass or any sweep; on the list
  int64_t* list;
  // [0] zones whose slopes the first pass removed, [1] list length, [2] and
  // [3] of step 9.c, [4 + n] flag changes of sweep n
  unsigned int* ctr;
  // a sweep after one that changed no flag has nothing to do; its own change
  // count, zero from the start, passes that on
  __device__ __forceinline__ bool done(int sweep) const {
    return ctr[0] == 0 || (sweep > 0 && ctr[4 + sweep - 1] == 0);
  }
};
constexpr int kCtrWords = 4 + kMaxSweeps;

// ---------------------------------------------------------------------------
// steps 2 and 5
// and the positivity limiter's flags and counters start clear
__global__ void __launch_bounds__(256) k_prim(const P1 P, const Box b, const Flags F) {
  int i, j, k;
  if (blockIdx.x == 0)
    for (int q = threadIdx.x; q < kCtrWords; q += blockDim.x) F.ctr[q] = 0;
  if (!b.decode(tid(), i, j, k)) return;
  const cs_p1_patch& a = P.a;
  const int64_t z = P.zi(i, j, k);
  F.fl[0][z] = F.fl[1][z] = F.ever[z] = F.inlist[z] = 0;
  const double gam = a.gamma;
  a.gamma_eos[z] = gam;
  a.gamma_sound[z] = gam;
  a.mean_mol_wt[z] = a.molewt;
#pragma unroll
  for (int c = 0; c < 8; ++c)
#pragma unroll
    for (int m = 1; m < 4; ++m) {
      P.Ur(c, m, z) = 0.0;
      P.Vr(c, m, z) = 0.0;
    }
#pragma unroll
  for (int m = 1; m < 4; ++m) a.ent[z + P.NZ * m] = 0.0;
  double U[8], was[8], V[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) was[c] = P.Ur(c, 0, z);
  if (a.mask[z] == 0) {
#pragma unroll
    for (int c = 0; c < 8; ++c) U[c] = 0.0;
    U[0] = a.rhofloor;
    U[4] = a.prsfloor / (gam - 1.0);
    a.scale[z] = a.smallnum;
  } else {
#pragma unroll
    for (int c = 0; c < 8; ++c) U[c] = was[c];
  }
  double e = a.ent[z];
  Gas<double> gs{gam, gam - 1.0, a.rhofloor, a.prsfloor, 1.0 / (gam - 1.0)};
  V[4] = 0.0;
  cons_to_prim(gs, U, V, e);
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    P.Vr(c, 0, z) = V[c];
    put_changed(P.Ur(c, 0, z), U[c], was[c]);
  }
  a.ent[z] = e;
  const double b2 = (V[5] * V[5] + V[6] * V[6] + V[7] * V[7]) * C<double>::ob4pi;
  a.msonic[z] = sqrt((gam * V[4] + b2) / V[0]);
}

// step 2, faces: blockIdx.y = family
__global__ void __launch_bounds__(256) k_face_zero(const P1 P) {
  const int fam = blockIdx.y;
  const int n = P.nf;
  const int64_t t = tid();
  if (t >= P.NFC) return;
  const int i = (int)(t % n) - P.g, j = (int)((t / n) % n) - P.g, k = (int)(t / ((int64_t)n * n)) - P.g;
  const int lo = 1 - P.g, hi = P.N + P.g, hr = P.NR + P.g;
  if (fam == 0) {
    if (j < lo || k < lo || k > hr) return;
    if (!P.active(max(i, lo), j, k) && !P.active(min(i + 1, hi), j, k)) P.a.Bxf[t] = 0.0;
  } else if (fam == 1) {
    if (i < lo || k < lo || k > hr) return;
    if (!P.active(i, max(j, lo), k) && !P.active(i, min(j + 1, hi), k)) P.a.Byf[t] = 0.0;
  } else {
    if (i < lo || j < lo) return;
    if (!P.active(i, j, 1)) P.a.Bzf[t] = 0.0;
  }
}

// step 3: one thread per (corner, ghost column, radial layer)
__global__ void __launch_bounds__(256) k_tricorner(const P1 P) {
  const int64_t t = tid();
  const int g = P.g, nzr = P.nzr;
  if (t >= 4 * (int64_t)g * nzr) return;
  const int corner = (int)(t / ((int64_t)g * nzr)), ii = (int)((t / nzr) % g), k = (int)(t % nzr) + 1 - g;
  if (!P.a.itri[corner]) return;
  const bool left = corner == 0 || corner == 3, down = corner < 2;
  const int i = left ? 1 - g + ii : P.N + 1 + ii, jj = down ? 1 : P.N;
  int a, b;
  P.nbr(i, jj, down ? 3 : 2, a, b);
  double& by = P.a.Byf[P.fci(i, down ? jj - 1 : jj, k)];
  double& bx = P.a.Bxf[P.fci(left ? a - 1 : a, b, k)];
  if (corner == 0 || corner == 2) {
    const double s = 0.5 * (by - bx);
    by = s;
    bx = -s;
  } else {
    const double s = 0.5 * (by + bx);
    by = s;
    bx = s;
  }
}

// ---------------------------------------------------------------------------
// step 6
__device__ __forceinline__ void six(const P1& P, int i, int j, int k, int64_t* z6) {
  int a, b;
  P.nbr(i, j, 0, a, b);
  z6[0] = P.zi(a, b, k);
  P.nbr(i, j, 1, a, b);
  z6[1] = P.zi(a, b, k);
  P.nbr(i, j, 2, a, b);
  z6[2] = P.zi(a, b, k);
  P.nbr(i, j, 3, a, b);
  z6[3] = P.zi(a, b, k);
  z6[4] = P.zi(i, j, k + 1);
  z6[5] = P.zi(i, j, k - 1);
}

__device__ __forceinline__ bool in_flat_range(const P1& P, int i, int j, int k) {
  const int lo = 2 - P.g, hx = P.N + P.g - 1, hr = P.NR + P.g - 1;
  return i >= lo && i <= hx && j >= lo && j <= hx && k >= lo && k <= hr;
}

__global__ void __launch_bounds__(256) k_flat_a(const P1 P, const Box b) {
  int i, j, k;
  if (!b.decode(tid(), i, j, k)) return;
  const cs_p1_patch& a = P.a;
  const int64_t z = P.zi(i, j, k);
  if (!in_flat_range(P, i, j, k)) {
    a.flatten[z] = 0.0;
    return;
  }
  int64_t z6[6];
  six(P, i, j, k, z6);
  const double obl = P.obl(z);
  double wmin = a.msonic[z];
#pragma unroll
  for (int q = 0; q < 6; ++q) wmin = fmin(wmin, a.msonic[z6[q]]);
  // the unit radial direction of the top z-face serves both z-faces
  double nzv[3];
  {
    const int64_t f = P.zfi(i, j, k);
    double s = 0.0;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      nzv[c] = a.zf_centroid[f + P.NZF * c];
    }
    s = 1.0 / fmax(sqrt(nzv[0] * nzv[0] + nzv[1] * nzv[1] + nzv[2] * nzv[2]), a.smallnum);
#pragma unroll
    for (int c = 0; c < 3; ++c) nzv[c] = nzv[c] * s;
  }
  double dv = 0.0;
#pragma unroll
  for (int q = 0; q < 6; ++q) {
    const bool up = (q % 2) == 0;
    const int64_t zo = up ? z6[q] : z, zn = up ? z : z6[q];
    double r[3], n[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) r[c] = (P.cen(zo, c) - P.cen(zn, c)) * obl;
    const double a11 = 0.5 / fmax(sqrt(r[0] * r[0] + r[1] * r[1] + r[2] * r[2]), a.smallnum);
    if (q < 2) {
      const int64_t f = P.xfi(q == 0 ? i : i - 1, j, k);
#pragma unroll
      for (int c = 0; c < 3; ++c) n[c] = a.xf_normal[f + P.NXF * c];
    } else if (q < 4) {
      const int64_t f = P.yfi(i, q == 2 ? j : j - 1, k);
#pragma unroll
      for (int c = 0; c < 3; ++c) n[c] = a.yf_normal[f + P.NXF * c];
    } else {
#pragma unroll
      for (int c = 0; c < 3; ++c) n[c] = nzv[c];
    }
    dv = dv + n[0] * a11 * (P.V(1, 0, zo) - P.V(1, 0, zn)) + n[1] * a11 * (P.V(2, 0, zo) - P.V(2, 0, zn)) +
         n[2] * a11 * (P.V(3, 0, zo) - P.V(3, 0, zn));
  }
  a.divvel[z] = dv;
  const double a13 = fabs(dv) / (a.flatten_coef * wmin) - 1.0;
  double f = a13 <= 0.0 ? 0.0 : fmin(1.0, a13);
  if (a.mask[z] != 1) f = 0.0;
  a.flatten[z] = f;
}

// flatten (stage a) -> work (stage b)
__global__ void __launch_bounds__(256) k_flat_b(const P1 P, const Box b) {
  int i, j, k;
  if (!b.decode(tid(), i, j, k)) return;
  const cs_p1_patch& a = P.a;
  const int64_t z = P.zi(i, j, k);
  double f = a.flatten[z];
  if (in_flat_range(P, i, j, k)) {
    int64_t z6[6];
    six(P, i, j, k, z6);
    const double p0 = a.prs_flatten_coef * P.V(4, 0, z);
#pragma unroll
    for (int q = 0; q < 6; ++q)
      if (P.V(4, 0, z6[q]) > p0) f = fmax(f, a.flatten[z6[q]]);
  }
  a.work[z] = f;
}

// work (stage b) -> flatten (stage c)
__global__ void __launch_bounds__(256) k_flat_c(const P1 P, const Box b) {
  int i, j, k;
  if (!b.decode(tid(), i, j, k)) return;
  const cs_p1_patch& a = P.a;
  const int64_t z = P.zi(i, j, k);
  double f = a.work[z];
  if (in_flat_range(P, i, j, k)) {
    int64_t z6[6];
    six(P, i, j, k, z6);
#pragma unroll
    for (int q = 0; q < 6; ++q) f = fmax(f, a.work[z6[q]]);
  }
  a.flatten[z] = f;
}

// ---------------------------------------------------------------------------
// WENO (410...f:2421-3761, 5437-7100): stencil s uses the x-neighbour
// (R for s in {0,1,4,5}, else L), the y-neighbour (U for s < 4, else D) and the
// z-neighbour (top for even s, else bottom), each stencil's 3 x 3 offset
// matrix inverted by its adjugate (inv3)
__device__ __forceinline__ bool in_weno_range(const P1& P, int i, int j, int k) {
  return i >= -2 && i <= P.N + 3 && j >= -2 && j <= P.N + 3 && k >= -2 && k <= P.NR + 3;
}

// ---------------------------------------------------------------------------
// step 7.a: WENO of the 8 primitives and the entropy, one thread per three
// fields of a zone of the range (or of a zone list).  Inactive columns keep
// the zero modes k_prim left.
__device__ __forceinline__ void zone_of(const P1& P, int64_t z, int& i, int& j, int& k) {
  i = (int)(z % P.nz) + 1 - P.g;
  j = (int)((z / P.nz) % P.nz) + 1 - P.g;
  k = (int)(z / ((int64_t)P.nz * P.nz)) + 1 - P.g;
}

// the fields of one WENO launch: the mean of field f at src[f][z], its three
// gradient modes at dst[f][z + m * stride[f]], m = 0, 1, 2
struct WenoFields {
  const double* src[9];
  double* dst[9];
  int64_t stride[9];
  int n;
  uint32_t noflat;  // bit f: field f's gradients are not multiplied by (1 - flattener)
};

// The WENO of up to three fields of one zone in one pass over the 8
// stencils: per stencil its 3 x 3 inverse (formed once for the three
// fields), each field's gradient X_s, its weight
// w_s = 1 / (|X_s|^2 + smallnum)^4, and the running sums of w_s X_s, w_s and
// X_s; the central candidate (the mean of the 8 gradients, weight 100) is
// added at the end and the sum normalised.  The stencil's neighbours are
// chosen by selects: indexing the small arrays by the loop counter would put
// them in scratch.
__device__ __forceinline__ void weno_group(const P1& P, int i, int j, int k, int64_t z, int c0, const WenoFields W9) {
  if (!P.active(i, j, 1)) return;
  const cs_p1_patch& a = P.a;
  int64_t z6[6];
  six(P, i, j, k, z6);
  const double obl = P.obl(z);
  double off[6][3];
#pragma unroll
  for (int q = 0; q < 6; ++q)
#pragma unroll
    for (int c = 0; c < 3; ++c) off[q][c] = (P.cen(z6[q], c) - P.cen(z, c)) * obl;
  const int nf = 3;  // both launches hold 9 or 3 fields: every group has three
  const double smallnum = a.smallnum, omf = 1.0 - a.flatten[z];
  // the group's field pointers by selects among the table's static entries
  // (c0 is 0, 3 or 6; indexing the argument table at run time would copy it
  // to scratch)
  const double* srcs[3];
  double* dsts[3];
  int64_t strides[3];
#pragma unroll
  for (int f = 0; f < 3; ++f) {
    srcs[f] = c0 == 0 ? W9.src[f] : (c0 == 3 ? W9.src[3 + f] : W9.src[6 + f]);
    dsts[f] = c0 == 0 ? W9.dst[f] : (c0 == 3 ? W9.dst[3 + f] : W9.dst[6 + f]);
    strides[f] = c0 == 0 ? W9.stride[f] : (c0 == 3 ? W9.stride[3 + f] : W9.stride[6 + f]);
  }
  // differences to the six neighbours, one array per neighbour (a select
  // between two entries of one array would be turned into an indexed load)
  double dR[3], dL[3], dU[3], dD[3], dT[3], dB[3], num[3][3], den[3], sx[3][3];
#pragma unroll
  for (int f = 0; f < 3; ++f) {
    const double* src = srcs[f];
    const double f0 = src[z];
    dR[f] = src[z6[0]] - f0;
    dL[f] = src[z6[1]] - f0;
    dU[f] = src[z6[2]] - f0;
    dD[f] = src[z6[3]] - f0;
    dT[f] = src[z6[4]] - f0;
    dB[f] = src[z6[5]] - f0;
    den[f] = 0.0;
#pragma unroll
    for (int m = 0; m < 3; ++m) num[f][m] = sx[f][m] = 0.0;
  }
#pragma unroll 1
  for (int s = 0; s < 8; ++s) {
    const bool bx = (s >> 1) & 1, by = (s >> 2) & 1, bz = s & 1;
    double m3[3][3], A[3][3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      m3[0][c] = bx ? off[1][c] : off[0][c];
      m3[1][c] = by ? off[3][c] : off[2][c];
      m3[2][c] = bz ? off[5][c] : off[4][c];
    }
    inv3(m3, A);
#pragma unroll
    for (int f = 0; f < 3; ++f) {
      const double r0 = bx ? dL[f] : dR[f], r1 = by ? dD[f] : dU[f], r2 = bz ? dB[f] : dT[f];
      double X[3];
#pragma unroll
      for (int m = 0; m < 3; ++m) X[m] = A[m][0] * r0 + A[m][1] * r1 + A[m][2] * r2;
      double tt = X[0] * X[0] + X[1] * X[1] + X[2] * X[2] + smallnum;
      tt = tt * tt;
      const double w = 1.0 / (tt * tt);
      den[f] = s == 0 ? w : den[f] + w;
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        num[f][m] += w * X[m];
        sx[f][m] += X[m];
      }
    }
  }
#pragma unroll
  for (int f = 0; f < 3; ++f) {
    if (f >= nf) break;
    double X8[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) X8[m] = 0.125 * sx[f][m];
    double tt = X8[0] * X8[0] + X8[1] * X8[1] + X8[2] * X8[2] + smallnum;
    tt = tt * tt;
    const double w8 = 100.0 / (tt * tt);
    const double os = 1.0 / (den[f] + w8);
    double* dst = dsts[f];
    const int64_t stride = strides[f];
    const double of = ((W9.noflat >> (c0 + f)) & 1u) ? 1.0 : omf;
#pragma unroll
    for (int m = 0; m < 3; ++m) dst[z + stride * m] = (num[f][m] + w8 * X8[m]) * os * of;
  }
}

// thread t: fields 3 (t / n) .. 3 (t / n) + 2 of zone t % n of the box
__global__ void __launch_bounds__(128) k_weno9(const P1 P, const Box b, const WenoFields W9) {
  const int64_t t = tid(), n = b.count();
  if (t >= (int64_t)(W9.n / 3) * n) return;  // 3 or 9 fields
  int i, j, k;
  b.decode(t % n, i, j, k);
  weno_group(P, i, j, k, P.zi(i, j, k), 3 * (int)(t / n), W9);
}

// ---------------------------------------------------------------------------
// step 7.b: ENFORCE_PRESSURE_POSITIVITY_PRIM (440...f:6-830).
// the 27 zones around (i, j, k): the column and its 8 stencil neighbours
// (R, L, U, D, RU, LU, LD, RD), each at k-1, k, k+1, as the zone index of
// layer 0 of each column
__device__ __forceinline__ void columns9(const P1& P, int i, int j, int64_t* col) {
  col[0] = P.zi(i, j, 0);
  const int dirs[8] = {0, 1, 2, 3, 8, 9, 10, 11};
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    int ai, bj;
    P.nbr(i, j, dirs[q], ai, bj);
    col[q + 1] = P.zi(ai, bj, 0);
  }
}

// NM = 4: LIMIT_ALL_SLOPES_P1; NM = 10: LIMIT_ALL_SLOPES_P12 (step 7.c), the
// node values carrying the quadratic modes about the zone's own moments mom
// (440...f:594-600) and every mode above the mean reduced.  Two waves per
// SIMD: at NM = 10 the registers are held to 256 with a small spill, which
// the second wave more than pays for (the NM = 4 form fits without one)
template <int NM>
__device__ __forceinline__ void pos_zone(const P1& P, int i, int j, int k, int64_t z, int sweep, const Flags& F,
                                         const double* __restrict__ mom) {
  const cs_p1_patch& a = P.a;
  int64_t col[9];
  columns9(P, i, j, col);
  const int64_t ks = (int64_t)P.nz * P.nz;
  // ranges of rho, p and the entropy over the 27 zones, widened by 20 % where
  // the flattener is below 0.1 (440...f:169-280)
  double rmin = 1e300, rmax = -1e300, pmin = 1e300, pmax = -1e300, emin = 1e300, emax = -1e300;
#pragma unroll 1
  for (int q = 0; q < 9; ++q)
#pragma unroll
    for (int dk = -1; dk <= 1; ++dk) {
      const int64_t zz = col[q] + ks * (k + dk);
      const double r = P.V(0, 0, zz), p = P.V(4, 0, zz);
      double e = a.ent[zz];
      if (sweep >= 0 && zz < z && F.fl[sweep & 1][zz]) e = 0.0;
      rmin = fmin(rmin, r);
      rmax = fmax(rmax, r);
      pmin = fmin(pmin, p);
      pmax = fmax(pmax, p);
      emin = fmin(emin, e);
      emax = fmax(emax, e);
    }
  const double expandfac = 0.2;
  const double ff = fmax(fmin((a.flatten[z] - 0.1) / 0.4, 1.0), 0.0), omff = 1.0 - ff;
  rmin = fmax(rmin * (1.0 - expandfac * omff), a.rhofloor);
  rmax = fmax(rmax * (1.0 + expandfac * omff), a.rhofloor);
  pmin = fmax(pmin * (1.0 - expandfac * omff), a.prsfloor);
  pmax = fmax(pmax * (1.0 + expandfac * omff), a.prsfloor);
  emin = emin * (1.0 - expandfac * omff);
  emax = emax * (1.0 + expandfac * omff);
  // the modes checked at the 27 nodes: rho, p and the entropy
  const double r0 = P.V(0, 0, z), p0 = P.V(4, 0, z), e0 = a.ent[z];
  double rm[NM - 1], pm[NM - 1], em[3], q0[6];
#pragma unroll
  for (int m = 0; m < NM - 1; ++m) {
    rm[m] = P.V(0, m + 1, z);
    pm[m] = P.V(4, m + 1, z);
  }
#pragma unroll
  for (int m = 0; m < 3; ++m) em[m] = a.ent[z + P.NZ * (m + 1)];
#pragma unroll
  for (int m = 0; m < 6; ++m) q0[m] = NM == 10 ? mom[z + P.NZ * (4 + m)] : 0.0;
  const double obl = P.obl(z);
  double c0[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) c0[c] = P.cen(z, c);
  // the zone's 8 vertices and 6 face centroids, loaded once; the 27 nodes
  // (vertices, face centroids, edge midpoints, centroid) are formed from them
  double vx[8][3], fcx[6][3];
#pragma unroll
  for (int n = 0; n < 8; ++n) {
    const int vi = (n & 1) ? i : i - 1, vj = (n & 2) ? j : j - 1, vk = (n & 4) ? k : k - 1;
#pragma unroll
    for (int c = 0; c < 3; ++c) vx[n][c] = a.vert[P.fci(vi, vj, vk) + P.NFC * c];
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    fcx[0][c] = a.xf_centroid[P.xfi(i, j, k) + P.NXF * c];
    fcx[1][c] = a.xf_centroid[P.xfi(i - 1, j, k) + P.NXF * c];
    fcx[2][c] = a.yf_centroid[P.yfi(i, j, k) + P.NXF * c];
    fcx[3][c] = a.yf_centroid[P.yfi(i, j - 1, k) + P.NXF * c];
    fcx[4][c] = a.zf_centroid[P.zfi(i, j, k) + P.NZF * c];
    fcx[5][c] = a.zf_centroid[P.zfi(i, j, k - 1) + P.NZF * c];
  }
  const double ratio = 0.85769589859089412;  // 0.1^(1/15)
  // does every node pass with the slopes reduced n times?  The reduced slopes
  // are formed by n multiplications, as the reference's loop forms them
  auto passes = [&](int n) -> bool {
    double r[NM - 1], p[NM - 1], e[3];
#pragma unroll
    for (int m = 0; m < NM - 1; ++m) {
      r[m] = rm[m];
      p[m] = pm[m];
    }
#pragma unroll
    for (int m = 0; m < 3; ++m) e[m] = em[m];
    for (int q = 0; q < n; ++q) {
#pragma unroll
      for (int m = 0; m < NM - 1; ++m) {
        r[m] = ratio * r[m];
        p[m] = ratio * p[m];
      }
#pragma unroll
      for (int m = 0; m < 3; ++m) e[m] = ratio * e[m];
    }
    bool pass = true;
    // the scale opaque to the optimiser at third order: the nodes' offsets and
    // quadratic basis values are formed in each check instead of being
    // hoisted out of the bisection and held for all 27 nodes at once
    double ob = obl;
    if constexpr (NM == 10) asm volatile("" : "+v"(ob));
    // one node: scaled offset from the centroid, then the three checks
    auto node = [&](const double* x0) {
      double x[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) x[c] = (x0[c] - c0[c]) * ob;
      double rn = r0 + r[0] * x[0] + r[1] * x[1] + r[2] * x[2];
      double pn = p0 + p[0] * x[0] + p[1] * x[1] + p[2] * x[2];
      if constexpr (NM == 10) {
        const double b[6] = {x[0] * x[0] - q0[0], x[1] * x[1] - q0[1], x[2] * x[2] - q0[2],
                             x[0] * x[1] - q0[3], x[1] * x[2] - q0[4], x[0] * x[2] - q0[5]};
#pragma unroll
        for (int m = 0; m < 6; ++m) {
          rn = rn + r[3 + m] * b[m];
          pn = pn + p[3 + m] * b[m];
        }
      }
      const double en = e0 + e[0] * x[0] + e[1] * x[1] + e[2] * x[2];
      if (rn < rmin || rn > rmax || pn < pmin || pn > pmax || en < emin || en > emax) pass = false;
    };
#pragma unroll
    for (int v = 0; v < 8; ++v) node(vx[v]);
#pragma unroll
    for (int f = 0; f < 6; ++f) node(fcx[f]);
    // edge midpoints: vertex pairs along x, then y, then z
#pragma unroll
    for (int q = 0; q < 12; ++q) {
      const int va = q < 4 ? 2 * q : (q < 8 ? ((q - 4) & 1) + 4 * ((q - 4) >> 1) : q - 8);
      const int vb = q < 4 ? va + 1 : (q < 8 ? va + 2 : va + 4);
      double m[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) m[c] = (vx[va][c] + vx[vb][c]) * 0.5;
      node(m);
    }
    node(c0);
    return pass;
  };
  // the reference (440...f:553-600) checks 0, 1, ..., 14 reductions in turn and
  // takes the first that passes, removing the slopes when none does.  With
  // the zone's mean inside the bounds, passing is monotone in the number of
  // reductions (in exact arithmetic), so the first passing count is found by
  // bisection: 2 to 6 checks instead of up to 15.  The count found passes and
  // the one below it fails (both are checked); only a node value that rounds
  // across a bound at a smaller count, although the counts' node values
  // differ by 14 % of the slope part, could make the reference's scan stop
  // earlier
  // one call site (the check is large): probe 0, then 14, then bisect; lo is
  // the largest count known to fail, hi the smallest known to pass (15: none)
  int lo = -1, hi = 15, n = 0;
#pragma unroll 1
  while (hi - lo > 1) {
    const bool ok = passes(n);
    if (ok) hi = n;
    else lo = n;
    n = lo < 0 ? 0 : (lo == 0 && hi == 15 ? 14 : (lo + hi) >> 1);
  }
  const bool removed = hi == 15;
  const int nred = removed ? 0 : hi;
  if (!removed)
    for (int q = 0; q < nred; ++q)
#pragma unroll
      for (int m = 0; m < 3; ++m) em[m] = ratio * em[m];
  // the same reductions on every component (repeated, as the reference
  // multiplies once per iteration); B_zc copies the B modes
  if (nred > 0 || removed) {
    for (int c = 0; c < 8; ++c)
#pragma unroll
      for (int m = 0; m < NM - 1; ++m) {
        double v = P.V(c, m + 1, z);
        if (removed) {
          v = 0.0;
        } else {
          for (int r = 0; r < nred; ++r) v = ratio * v;
        }
        P.Vr(c, m + 1, z) = v;
      }
#pragma unroll
    for (int m = 0; m < 3; ++m) a.ent[z + P.NZ * (m + 1)] = removed ? 0.0 : em[m];
  }
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    a.B1_zc[z + P.NZ * m] = P.V(5, m, z);
    a.B2_zc[z + P.NZ * m] = P.V(6, m, z);
    a.B3_zc[z + P.NZ * m] = P.V(7, m, z);
  }
  const uint8_t flag = removed ? 1 : 0;
  if (sweep < 0) {
    F.fl[0][z] = flag;
    F.fl[1][z] = flag;
    F.ever[z] = flag;
    if (removed) atomicAdd(&F.ctr[0], 1u);
  } else {
    F.fl[(sweep + 1) & 1][z] = flag;
    if (flag) F.ever[z] = 1;
    if (flag != F.fl[sweep & 1][z]) atomicAdd(&F.ctr[4 + sweep], 1u);
  }
}
template <int NM>
__global__ void __attribute__((amdgpu_waves_per_eu(2))) __launch_bounds__(256)
    k_pos(const P1 P, const Box b, const Flags F, const double* __restrict__ mom) {
  int i, j, k;
  if (!b.decode(tid(), i, j, k)) return;
  pos_zone<NM>(P, i, j, k, P.zi(i, j, k), -1, F, mom);
}

// the zones of the range with a zone ever flagged earlier in the loop order
// among their 27 and not yet on the list: appended to it (order immaterial;
// the list only grows, so a zone whose result depends on a flag is
// recomputed in every later sweep; a zone that joins has its first pass's
// flag in both arrays)
constexpr int kListBlocks = 512;   // grids of the list's kernels at 256 threads (grid-stride)
constexpr int kCandBlocks = 2048;  // largest grid of k_cands (grid-stride)
__global__ void __launch_bounds__(256) k_cands(const P1 P, const Box b, const Flags F, int sweep) {
  if (F.done(sweep)) return;
  const int64_t n = b.count(), ks = (int64_t)P.nz * P.nz;
  for (int64_t t = tid(); t < n; t += (int64_t)gridDim.x * blockDim.x) {
    int i, j, k;
    b.decode(t, i, j, k);
    const int64_t z = P.zi(i, j, k);
    if (F.inlist[z]) continue;
    int64_t col[9];
    columns9(P, i, j, col);
    bool cand = false;
    for (int q = 0; q < 9; ++q)
#pragma unroll
      for (int dk = -1; dk <= 1; ++dk) {
        const int64_t zz = col[q] + ks * (k + dk);
        cand = cand || (zz < z && F.ever[zz]);
      }
    if (cand) {
      F.inlist[z] = 1;
      F.list[atomicAdd(&F.ctr[1], 1u)] = z;
    }
  }
}
// one sweep over the list: WENO again, then positivity.  A list that gives
// every workgroup one group of 64 zones at most is latency: three waves take
// the zones' fields, three each, then the first wave their positivity.  A
// longer one is throughput: a lane does both for its zone, so that all four
// waves work on positivity (192^2 x 64 with noise of 1.0 on the density 27.6 ->
// 14.8 ms a call, 128^2 x 48 with 1.5 7.8 -> 4.5).  The counts and the flags stay on the device, so
// the host looks once per kSweepBatch sweeps instead of twice per sweep (the
// call on a noisy 16^2 x 6 patch 423 -> 370 us, 128^2 x 48 2.42 -> 2.29 ms)
constexpr int kReplayZones = 64, kReplayThreads = 256;
__global__ void __attribute__((amdgpu_waves_per_eu(2))) __launch_bounds__(kReplayThreads)
    k_replay(const P1 P, const Flags F, const WenoFields W9, int sweep) {
  if (F.done(sweep)) return;
  const int64_t n = F.ctr[1];
  const int nzb = n <= (int64_t)gridDim.x * kReplayZones ? kReplayZones : kReplayThreads;
  const int q = threadIdx.x % nzb, grp = threadIdx.x / nzb;
  for (int64_t t0 = (int64_t)blockIdx.x * nzb; t0 < n; t0 += (int64_t)gridDim.x * nzb) {
    const bool on = t0 + q < n;
    int i = 0, j = 0, k = 0;
    int64_t z = 0;
    if (on) {
      z = F.list[t0 + q];
      zone_of(P, z, i, j, k);
#pragma unroll 1
      for (int c = grp; c < 3; c += kReplayThreads / nzb) weno_group(P, i, j, k, z, 3 * c, W9);
    }
    __syncthreads();  // the zone's slopes are written before its positivity reads them
    if (on && grp == 0) pos_zone<4>(P, i, j, k, z, sweep, F, nullptr);
  }
}
// the same at third order in three launches, the WENO-AO (k_weno_ao_list) between
__global__ void __launch_bounds__(128) k_weno9_list(const P1 P, const Flags F, const WenoFields W9, int sweep) {
  if (F.done(sweep)) return;
  const int64_t n = F.ctr[1];
  for (int64_t t = tid(); t < 3 * n; t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t z = F.list[t % n];
    int i, j, k;
    zone_of(P, z, i, j, k);
    weno_group(P, i, j, k, z, 3 * (int)(t / n), W9);
  }
}
__global__ void __attribute__((amdgpu_waves_per_eu(2))) __launch_bounds__(256)
    k_pos10_list(const P1 P, const Flags F, const double* __restrict__ mom, int sweep) {
  if (F.done(sweep)) return;
  const int64_t n = F.ctr[1];
  for (int64_t t = tid(); t < n; t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t z = F.list[t];
    int i, j, k;
    zone_of(P, z, i, j, k);
    pos_zone<10>(P, i, j, k, z, sweep, F, mom);
  }
}

// the entropy means of the zones that lost all their slopes
__global__ void __launch_bounds__(256) k_clear_ent(const P1 P, const Box b, const uint8_t* flags) {
  int i, j, k;
  if (!b.decode(tid(), i, j, k)) return;
  const int64_t z = P.zi(i, j, k);
  if (flags[z]) P.a.ent[z] = 0.0;
}

// ---------------------------------------------------------------------------
// step 8.a-c: blockIdx.y = family
// NM = 10: the third-order form (421...f:4817-4879), each side's field with
// its quadratic modes about that zone's own moments mom
template <int NM>
__global__ void __launch_bounds__(256) k_face_pts(const P1 P, const Box bx, const Box by, const Box bz,
                                                  const double* __restrict__ mom) {
  const int fam = blockIdx.y;
  const Box& b = fam == 0 ? bx : (fam == 1 ? by : bz);
  int i, j, k;
  if (!b.decode(tid(), i, j, k)) return;
  const cs_p1_patch& a = P.a;
  double* Bq = fam == 0 ? a.Bxf_q : (fam == 1 ? a.Byf_q : a.Bzf_q);
  const double* Bf = fam == 0 ? a.Bxf : (fam == 1 ? a.Byf : a.Bzf);
  const double* pts = fam == 0 ? a.xb_pts : (fam == 1 ? a.yb_pts : a.zb_pts);
  const double* wts = fam == 0 ? a.xb_wts : (fam == 1 ? a.yb_wts : a.zb_wts);
  const double* nrm = fam == 0 ? a.xb_normal : (fam == 1 ? a.yb_normal : a.zb_normal);
  const int64_t NF = fam == 2 ? P.NZF : P.NXF;
  const int64_t fb = P.fci(i, j, k), fg = fam == 0 ? P.xfi(i, j, k) : (fam == 1 ? P.yfi(i, j, k) : P.zfi(i, j, k));
  int li = i, lj = j, ri = i + (fam == 0), rj = j + (fam == 1);
  bool skip = false;
  if (fam < 2) {
    const bool al = P.active(li, lj, k), ar = P.active(ri, rj, k);
    if (!al && ar) {
      P.nbr(ri, rj, fam == 0 ? 1 : 3, li, lj);
    } else if (al && !ar) {
      P.nbr(li, lj, fam == 0 ? 0 : 2, ri, rj);
    } else if (!al && !ar) {
      skip = true;
    }
  } else {
    skip = !P.active(i, j, k);
  }
  double q5[5];
  if (skip) {
#pragma unroll
    for (int q = 0; q < 5; ++q) q5[q] = 0.0;
  } else {
    const int64_t zl = P.zi(li, lj, k), zr = P.zi(ri, rj, fam == 2 ? k + 1 : k);
    const double oll = P.obl(zl), olr = P.obl(zr);
    double vl[3][NM], vr[3][NM], ql[6], qr[6];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        vl[c][m] = P.V(5 + c, m, zl);
        vr[c][m] = P.V(5 + c, m, zr);
      }
#pragma unroll
    for (int m = 0; m < 6; ++m) {
      ql[m] = NM == 10 ? mom[zl + P.NZ * (4 + m)] : 0.0;
      qr[m] = NM == 10 ? mom[zr + P.NZ * (4 + m)] : 0.0;
    }
    double n[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) n[c] = nrm[fg + NF * c];
#pragma unroll
    for (int q = 0; q < 5; ++q) {
      if (fam == 2) {
#pragma unroll
        for (int c = 0; c < 3; ++c) n[c] = nrm[fg + NF * (c + 3 * q)];
      }
      double rl[3], rr[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double x = pts[fg + NF * (c + 3 * q)];
        rl[c] = (x - P.cen(zl, c)) * oll;
        rr[c] = (x - P.cen(zr, c)) * olr;
      }
      double s[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        double bl = vl[c][0] + vl[c][1] * rl[0] + vl[c][2] * rl[1] + vl[c][3] * rl[2];
        double br = vr[c][0] + vr[c][1] * rr[0] + vr[c][2] * rr[1] + vr[c][3] * rr[2];
        if constexpr (NM == 10) {
          const double pl[6] = {rl[0] * rl[0] - ql[0], rl[1] * rl[1] - ql[1], rl[2] * rl[2] - ql[2],
                                rl[0] * rl[1] - ql[3], rl[1] * rl[2] - ql[4], rl[0] * rl[2] - ql[5]};
          const double pr[6] = {rr[0] * rr[0] - qr[0], rr[1] * rr[1] - qr[1], rr[2] * rr[2] - qr[2],
                                rr[0] * rr[1] - qr[3], rr[1] * rr[2] - qr[4], rr[0] * rr[2] - qr[5]};
#pragma unroll
          for (int m = 0; m < 6; ++m) {
            bl = bl + vl[c][4 + m] * pl[m];
            br = br + vr[c][4 + m] * pr[m];
          }
        }
        s[c] = bl + br;
      }
      q5[q] = 0.5 * (n[0] * s[0] + n[1] * s[1] + n[2] * s[2]);
    }
  }
  double bd = Bf[fb];
#pragma unroll
  for (int q = 0; q < 5; ++q) bd = bd - wts[fg + NF * q] * q5[q];
#pragma unroll
  for (int q = 0; q < 5; ++q) Bq[fb + P.NFC * q] = q5[q] + bd;
}

// ---------------------------------------------------------------------------

// face f of zone (i, j, k): 0 right x, 1 left x, 2 up y, 3 down y, 4 top z, 5 bottom z
struct FaceRef {
  const double *nrm, *cen, *pts, *Bf, *Bq;
  int64_t fg, fb, NF;
};
__device__ __forceinline__ FaceRef face_of(const P1& P, int f, int i, int j, int k) {
  const cs_p1_patch& a = P.a;
  const int fam = f >> 1;
  const bool hi = (f & 1) == 0;
  const int fi = i - (fam == 0 && !hi), fj = j - (fam == 1 && !hi), fk = k - (fam == 2 && !hi);
  FaceRef r;
  r.fg = fam == 0 ? P.xfi(fi, fj, fk) : (fam == 1 ? P.yfi(fi, fj, fk) : P.zfi(fi, fj, fk));
  r.fb = P.fci(fi, fj, fk);
  r.NF = fam == 2 ? P.NZF : P.NXF;
  r.nrm = fam == 0 ? a.xb_normal : (fam == 1 ? a.yb_normal : a.zb_normal);
  r.cen = fam == 0 ? a.xf_centroid : (fam == 1 ? a.yf_centroid : a.zf_centroid);
  r.pts = fam == 0 ? a.xb_pts : (fam == 1 ? a.yb_pts : a.zb_pts);
  r.Bf = fam == 0 ? a.Bxf : (fam == 1 ? a.Byf : a.Bzf);
  r.Bq = fam == 0 ? a.Bxf_q : (fam == 1 ? a.Byf_q : a.Bzf_q);
  return r;
}

// Two waves per SIMD (216 registers, no LDS) where the 12 x 12 Cholesky and
// Schur form this replaces ran one (402 registers, 36 KB): 128^2 x 48 382 ->
// 220 us.  Against the KKT system in 80-bit arithmetic on this geometry's
// zones its largest relative error is 1.1e-15, the other form's 9.6e-15.
__global__ void __launch_bounds__(64) k_clsq_e(const P1 P, const Box b) {
  int i, j, k;
  if (!b.decode(tid(), i, j, k)) return;
  const cs_p1_patch& a = P.a;
  const int64_t z = P.zi(i, j, k);
  if (in_weno_range(P, i, j, k) && a.mask[z] != 0) {
    const double obl = P.obl(z);
    const double c0[3] = {P.cen(z, 0), P.cen(z, 1), P.cen(z, 2)};
    auto con = [&](int f, double* n, double* r) -> double {
      const FaceRef F = face_of(P, f, i, j, k);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        n[c] = F.nrm[F.fg + F.NF * c];
        r[c] = (F.cen[F.fg + F.NF * c] - c0[c]) * obl;
      }
      return F.Bf[F.fb];
    };
    auto pnt = [&](int f, int t, double* n, double* r) -> double {
      const FaceRef F = face_of(P, f, i, j, k);
      const int pt = 1 + 2 * t;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        n[c] = (f >> 1) == 2 ? F.nrm[F.fg + F.NF * (c + 3 * pt)] : F.nrm[F.fg + F.NF * c];
        r[c] = (F.pts[F.fg + F.NF * (c + 3 * pt)] - c0[c]) * obl;
      }
      return F.Bq[F.fb + P.NFC * pt];
    };
    double u[12];
    adp_clsq(con, pnt, [&](int c, int m) { return P.V(5 + c, m, z); }, u);
    const double aa = (P.Ur(5, 0, z) * P.Ur(5, 0, z) + P.Ur(6, 0, z) * P.Ur(6, 0, z) + P.Ur(7, 0, z) * P.Ur(7, 0, z)) *
                      C<double>::ob8pi;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      a.B1_zc[z + P.NZ * m] = u[m];
      a.B2_zc[z + P.NZ * m] = u[4 + m];
      a.B3_zc[z + P.NZ * m] = u[8 + m];
#pragma unroll
      for (int c = 0; c < 3; ++c) P.Vr(5 + c, m, z) = u[4 * c + m];
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) P.Ur(5 + c, 0, z) = u[4 * c];
    const double bb = (u[0] * u[0] + u[4] * u[4] + u[8] * u[8]) * C<double>::ob8pi;
    P.Ur(4, 0, z) = P.Ur(4, 0, z) - aa + bb;
  }
  // step 9.a: E = -v x B from the zone means
  const double vx = P.V(1, 0, z), vy = P.V(2, 0, z), vz = P.V(3, 0, z);
  const double Bx = P.V(5, 0, z), By = P.V(6, 0, z), Bz = P.V(7, 0, z);
  a.Ex_zc[z] = -(vy * Bz - vz * By);
  a.Ey_zc[z] = -(vz * Bx - vx * Bz);
  a.Ez_zc[z] = -(vx * By - vy * Bx);
}

// ---------------------------------------------------------------------------
// step 10: per-block minima and maxima of the 8 primitives and the
// normalised divergence over the owned active zones (18 values per block)
constexpr int DIAG_THREADS = 256;
__global__ void __launch_bounds__(DIAG_THREADS) k_diag(const P1 P, const Box b, double* part) {
  __shared__ double sh[18][DIAG_THREADS];
  double mn[9], mx[9];
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    mn[q] = 1.0e30;
    mx[q] = -1.0e30;
  }
  int i, j, k;
  if (b.decode(tid(), i, j, k)) {
    const cs_p1_patch& a = P.a;
    const int64_t z = P.zi(i, j, k);
    a.work[z] = 0.0;
    const bool own = i >= 1 && i <= P.N && j >= 1 && j <= P.N && k >= 1 && k <= P.NR && a.mask[z] == 1;
    if (own) {
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        mn[c] = fmin(mn[c], P.V(c, 0, z));
        mx[c] = fmax(mx[c], P.V(c, 0, z));
      }
      const double bxp = a.Bxf[P.fci(i, j, k)], bxm = a.Bxf[P.fci(i - 1, j, k)];
      const double byp = a.Byf[P.fci(i, j, k)], bym = a.Byf[P.fci(i, j - 1, k)];
      const double bzp = a.Bzf[P.fci(i, j, k)], bzm = a.Bzf[P.fci(i, j, k - 1)];
      double a21 = a.xf_area[P.xfi(i, j, k)] * bxp + a.yf_area[P.yfi(i, j, k)] * byp +
                   a.zf_area[P.zfi(i, j, k)] * bzp - a.xf_area[P.xfi(i - 1, j, k)] * bxm -
                   a.yf_area[P.yfi(i, j - 1, k)] * bym - a.zf_area[P.zfi(i, j, k - 1)] * bzm;
      a.work[z] = a21;
      const double v6 = P.V(5, 0, z), v7 = P.V(6, 0, z), v8 = P.V(7, 0, z), rho = P.V(0, 0, z);
      const double a11 = v6 * v6 + v7 * v7 + v8 * v8;
      const double ms = sqrt((a.gamma_sound[z] * P.V(4, 0, z) + C<double>::ob4pi * a11) / rho);
      a.msonic[z] = ms;
      const double den = fmax(fmax(sqrt(bxp * bxp + byp * byp + bzp * bzp), sqrt(bxm * bxm + bym * bym + bzm * bzm)),
                              ms * sqrt(4.0 * 3.14 * rho));
      a21 = a21 / den;
      mn[8] = a21;
      mx[8] = a21;
    }
  }
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    sh[q][threadIdx.x] = mn[q];
    sh[9 + q][threadIdx.x] = mx[q];
  }
  __syncthreads();
  for (int w = DIAG_THREADS / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
#pragma unroll
      for (int q = 0; q < 9; ++q) {
        sh[q][threadIdx.x] = fmin(sh[q][threadIdx.x], sh[q][threadIdx.x + w]);
        sh[9 + q][threadIdx.x] = fmax(sh[9 + q][threadIdx.x], sh[9 + q][threadIdx.x + w]);
      }
    __syncthreads();
  }
  if (threadIdx.x < 18) part[(int64_t)blockIdx.x * 18 + threadIdx.x] = sh[threadIdx.x][0];
}

// one block per quantity (9 minima, then 9 maxima)
__global__ void __launch_bounds__(256) k_diag_final(const double* part, int nblocks, double* out) {
  __shared__ double sh[256];
  const int q = blockIdx.x;
  double v = q < 9 ? 1.0e30 : -1.0e30;
  for (int b = threadIdx.x; b < nblocks; b += 256)
    v = q < 9 ? fmin(v, part[(int64_t)b * 18 + q]) : fmax(v, part[(int64_t)b * 18 + q]);
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
      sh[threadIdx.x] = q < 9 ? fmin(sh[threadIdx.x], sh[threadIdx.x + w]) : fmax(sh[threadIdx.x], sh[threadIdx.x + w]);
    __syncthreads();
  }
  if (threadIdx.x == 0) out[q] = sh[0];
}

// ---------------------------------------------------------------------------
// per-device work memory, one owner at a time: a call holds g_mu while it
// puts its kernels on its stream, and `done`, recorded behind them, makes the
// next call's stream wait for them
struct Scratch {
  void* mem = nullptr;
  size_t bytes = 0;
  hipEvent_t done = nullptr;
  bool used = false;
};
static std::mutex g_mu;
static std::vector<Scratch> g_scratch;

}  // namespace csp1

using namespace csp1;

static int p1_check(const cs_p1_patch* p) {
  if (!p) {
    cs::set_error("cs_limit_all_slopes_p1: null patch");
    return CS_E_INVALID;
  }
  if (p->ntp < 1 || p->nr < 1 || p->nghost < 4) {
    cs::set_error("cs_limit_all_slopes_p1: need ntp >= 1, nr >= 1, nghost >= 4 (got %d, %d, %d)", p->ntp, p->nr,
                  p->nghost);
    return CS_E_INVALID;
  }
  if (p->nghost >= p->ntp) {
    cs::set_error("cs_limit_all_slopes_p1: nghost (%d) must be below ntp (%d)", p->nghost, p->ntp);
    return CS_E_BAD_DECOMP;
  }
  if (!(p->gamma > 1.0) || !(p->smallnum > 0.0) || !(p->rhofloor > 0.0) || !(p->prsfloor > 0.0)) {
    cs::set_error("cs_limit_all_slopes_p1: gamma > 1 and positive floors and smallnum required");
    return CS_E_INVALID;
  }
  const void* ptrs[] = {p->vert, p->mask, p->stencil, p->xf_normal, p->xf_area, p->xf_centroid, p->yf_normal,
                        p->yf_area, p->yf_centroid, p->zf_area, p->zf_centroid, p->xb_pts, p->xb_wts,
                        p->xb_normal, p->yb_pts, p->yb_wts, p->yb_normal, p->zb_pts, p->zb_wts, p->zb_normal,
                        p->scale, p->v_centroid, p->U, p->ent, p->Bxf, p->Byf, p->Bzf, p->V, p->B1_zc, p->B2_zc,
                        p->B3_zc, p->Ex_zc, p->Ey_zc, p->Ez_zc, p->gamma_eos, p->gamma_sound, p->mean_mol_wt,
                        p->divvel, p->msonic, p->flatten, p->work, p->Bxf_q, p->Byf_q, p->Bzf_q};
  for (const void* q : ptrs)
    if (!q) {
      cs::set_error("cs_limit_all_slopes_p1: null array in the patch");
      return CS_E_INVALID;
    }
  return 0;
}

#define P1_HIP(call)                                                                  \
  do {                                                                                \
    hipError_t e_ = (call);                                                           \
    if (e_ != hipSuccess) {                                                           \
      cs::set_error("cs_limit_all_slopes_p1: %s: %s", #call, hipGetErrorString(e_)); \
      return CS_E_HIP;                                                                \
    }                                                                                 \
  } while (0)

// the scratch of at least `need` bytes for work put on st from here on
static int scratch_open(Scratch& S, size_t need, hipStream_t st, const char* who) {
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  P1_HIP(hipStreamIsCapturing(st, &cap));
  if (cap != hipStreamCaptureStatusNone) {
    cs::set_error("%s: work memory shared with other calls cannot be used by a captured graph", who);
    return CS_E_HIP;
  }
  if (!S.done) P1_HIP(hipEventCreateWithFlags(&S.done, hipEventDisableTiming));
  if (S.used) P1_HIP(hipStreamWaitEvent(st, S.done, 0));
  if (S.bytes < need) {
    if (S.mem) P1_HIP(hipFree(S.mem));  // waits for the device
    S.mem = nullptr;
    S.bytes = 0;
    if (hipMalloc(&S.mem, need) != hipSuccess) {
      (void)hipGetLastError();
      cs::set_error("%s: cannot allocate %zu bytes of work memory", who, need);
      return CS_E_NOMEM;
    }
    S.bytes = need;
  }
  return 0;
}
// closes the scratch on every way out of the call
struct ScratchUse {
  Scratch* S;
  hipStream_t st;
  ~ScratchUse() {
    if (S) S->used = hipEventRecord(S->done, st) == hipSuccess || S->used;
  }
};

static inline unsigned grid_of(int64_t n, int threads) { return (unsigned)((n + threads - 1) / threads); }

// kernel_ms (optional): per-stage times from HIP events on the stream
// ext (optional): caller-provided device work memory of ext_bytes, used
// instead of the library's per-device allocation (no allocation then)
namespace csp1 {
__global__ void __launch_bounds__(256) k_zero_hi(const P1 P, const Box b);
__global__ void __attribute__((amdgpu_waves_per_eu(2))) __launch_bounds__(64)
    k_clsq12(const P1 P, const Box b, const double* __restrict__ mom);
constexpr int kSqZones = 4;  // zones per wave of k_clsq12
__global__ void __launch_bounds__(256) k_e12(const P1 P, const Box b, const double* __restrict__ mom);
__global__ void __launch_bounds__(256) k_ao_order(const P1 P, const Box b, unsigned int* bad);
constexpr int kAoRec = 208;     // doubles per zone record of k_ao_e_pre
constexpr int kAoLanes = 16;    // lanes per zone of k_ao_e_sweep
constexpr int kAoGroups = 28;   // zones of one plane in flight at most (448 threads, and a wave that publishes)
// the in-plane level of box zone (ir, jr) is ir + s jr: s >= 3 keeps the order,
// s kAoGroups >= ni leaves at most one row per group of lanes
__host__ __device__ static inline int ao_stride(int ni) {
  const int s = (ni + kAoGroups - 1) / kAoGroups;
  return s < 3 ? 3 : s;
}
__global__ void __launch_bounds__(128) k_ao_e_pre(const P1 P, const Box b, const double* __restrict__ mom,
                                                  double* __restrict__ rec, double* __restrict__ xnew);
__global__ void __launch_bounds__(kAoLanes * kAoGroups + 64)
    k_ao_e_sweep(const P1 P, const Box b, double* rec, double* xnew, unsigned int* ticket, int s);
__global__ void __launch_bounds__(256) k_ao_e_put(const P1 P, const Box b, const double* __restrict__ rec);
__global__ void __attribute__((amdgpu_waves_per_eu(2))) __launch_bounds__(128)
    k_weno_ao(const P1 P, const Box b, const double* __restrict__ mom);
__global__ void __attribute__((amdgpu_waves_per_eu(2))) __launch_bounds__(128)
    k_weno_ao_list(const P1 P, const Box b, const double* __restrict__ mom, const Flags F, int sweep);
}  // namespace csp1

// mom (optional, DEVICE zone x 10): the third-order form, LIMIT_ALL_SLOPES_P12:
// U, V, B_zc and E_zc of ten modes, the WENO gradients left unflattened and
// followed by the WENO-AO hybridisation of step 7.b, the positivity limiter
// and the face-point B with the quadratic modes, the 30-unknown constrained
// least squares, the zone E at the centroid with its own WENO-AO (step 9)
static int run_p1(const cs_p1_patch* p, void* stream_, float* kernel_ms, uint8_t* ext = nullptr,
                  size_t ext_bytes = 0, const double* mom = nullptr) {
  int rc = p1_check(p);
  if (rc) return rc;
  hipStream_t st = (hipStream_t)stream_;
  P1 P;
  P.a = *p;
  P.N = p->ntp;
  P.NR = p->nr;
  P.g = p->nghost;
  P.nz = P.N + 2 * P.g;
  P.nzr = P.NR + 2 * P.g;
  P.nf = P.nz + 1;
  P.nfr = P.nzr + 1;
  P.NZ = (int64_t)P.nz * P.nz * P.nzr;
  P.NXF = (int64_t)P.nf * P.nz * P.nzr;
  P.NZF = (int64_t)P.nz * P.nz * P.nfr;
  P.NFC = (int64_t)P.nf * P.nf * P.nfr;
  const int N = P.N, NR = P.NR, g = P.g;
  const Box all = make_box(1 - g, N + g, 1 - g, N + g, 1 - g, NR + g);
  const Box wr = make_box(-2, N + 3, -2, N + 3, -2, NR + 3);
  const Box own = make_box(1, N, 1, N, 1, NR);
  const Box fx = make_box(-3, N + 3, -2, N + 3, -2, NR + 3), fy = make_box(-2, N + 3, -3, N + 3, -2, NR + 3),
            fz = make_box(-2, N + 3, -2, N + 3, -3, NR + 3);
  const int nblk_diag = (int)grid_of(all.count(), DIAG_THREADS);

  int dev = 0;
  P1_HIP(hipGetDevice(&dev));
  const size_t flag_bytes = ((size_t)P.NZ + 255) / 256 * 256;
  const size_t list_bytes = (size_t)wr.count() * sizeof(int64_t);
  const Box ao = make_box(-1, N + 2, -1, N + 2, -1, NR + 2);
  const size_t ctr_bytes = (kCtrWords * sizeof(unsigned int) + 255) / 256 * 256;
  const size_t base_bytes = (4 * flag_bytes + ctr_bytes + (size_t)nblk_diag * 18 * sizeof(double) + 18 * sizeof(double) +
                             list_bytes + 255) / 256 * 256;
  const size_t need = base_bytes + (mom ? (size_t)ao.count() * (kAoRec + 4) * sizeof(double) : 0);
  if (mom && P.NZ >= ((int64_t)1 << 31)) {
    cs::set_error("cs_limit_all_slopes_p12: the patch has %lld zones, more than int32 indices reach",
                  (long long)P.NZ);
    return CS_E_INVALID;
  }
  std::unique_lock<std::mutex> lock(g_mu, std::defer_lock);
  ScratchUse use{nullptr, st};
  uint8_t* base = nullptr;
  if (ext) {
    if (need > ext_bytes) {
      cs::set_error("cs_limit_all_slopes_p1_noalloc: the patch (%d^2 x %d, nghost %d) needs %zu bytes of work "
                    "memory, the entry point holds %zu", N, NR, g, need, ext_bytes);
      return CS_E_INVALID;
    }
    base = ext;
  } else {
    lock.lock();
    if ((int)g_scratch.size() <= dev) g_scratch.resize(dev + 1);
    Scratch& S = g_scratch[dev];
    if ((rc = scratch_open(S, need, st, "cs_limit_all_slopes_p1"))) return rc;
    use.S = &S;
    base = (uint8_t*)S.mem;
  }
  Flags F;
  F.fl[0] = base;
  F.fl[1] = base + flag_bytes;
  F.ever = base + 2 * flag_bytes;
  F.inlist = base + 3 * flag_bytes;
  F.ctr = (unsigned int*)(base + 4 * flag_bytes);
  double* part = (double*)(base + 4 * flag_bytes + ctr_bytes);
  double* red = part + (size_t)nblk_diag * 18;
  F.list = (int64_t*)(red + 18);
  double* aorec = (double*)(base + base_bytes);  // third order: the records of k_ao_e_pre

  constexpr int NEV = CS_P1_STAGES + 1;
  hipEvent_t ev[NEV];
  int nev = 0;
  if (kernel_ms) {
    for (int q = 0; q < NEV; ++q) P1_HIP(hipEventCreate(&ev[q]));
  }
  auto mark = [&]() -> int {
    if (kernel_ms) P1_HIP(hipEventRecord(ev[nev++], st));
    return 0;
  };
  if ((rc = mark())) return rc;
  if (mom) k_zero_hi<<<grid_of(all.count(), 256), 256, 0, st>>>(P, all);
  k_prim<<<grid_of(all.count(), 256), 256, 0, st>>>(P, all, F);
  if ((rc = mark())) return rc;
  k_face_zero<<<dim3(grid_of(P.NFC, 256), 3), 256, 0, st>>>(P);
  k_tricorner<<<grid_of(4 * (int64_t)g * P.nzr, 256), 256, 0, st>>>(P);
  if ((rc = mark())) return rc;
  k_flat_a<<<grid_of(all.count(), 256), 256, 0, st>>>(P, all);
  k_flat_b<<<grid_of(all.count(), 256), 256, 0, st>>>(P, all);
  k_flat_c<<<grid_of(all.count(), 256), 256, 0, st>>>(P, all);
  if ((rc = mark())) return rc;
  WenoFields wv, we;
  wv.n = 9;
  wv.noflat = mom ? 0xffu : 0u;  // third order: V flattened after the hybridisation
  we.noflat = mom ? 0x7u : 0u;  // third order: E flattened after its hybridisation
  for (int c = 0; c < 8; ++c) {
    wv.src[c] = p->V + P.NZ * c;
    wv.dst[c] = p->V + P.NZ * (c + 8);
    wv.stride[c] = 8 * P.NZ;
  }
  wv.src[8] = p->ent;
  wv.dst[8] = p->ent + P.NZ;
  wv.stride[8] = P.NZ;
  we.n = 3;
  double* E3[3] = {p->Ex_zc, p->Ey_zc, p->Ez_zc};
  for (int c = 0; c < 3; ++c) {
    we.src[c] = E3[c];
    we.dst[c] = E3[c] + P.NZ;
    we.stride[c] = P.NZ;
  }
  k_weno9<<<grid_of(3 * wr.count(), 128), 128, 0, st>>>(P, wr, wv);
  if (mom) {
    k_weno_ao<<<grid_of(ao.count(), 128), 128, 0, st>>>(P, ao, mom);
    k_pos<10><<<grid_of(wr.count(), 256), 256, 0, st>>>(P, wr, F, mom);
  } else {
    k_pos<4><<<grid_of(wr.count(), 256), 256, 0, st>>>(P, wr, F, nullptr);
  }
  P1_HIP(hipGetLastError());
  unsigned int nfail = 0;
  P1_HIP(hipMemcpyAsync(&nfail, F.ctr, sizeof(unsigned int), hipMemcpyDeviceToHost, st));
  P1_HIP(hipStreamSynchronize(st));
  if (nfail > 0) {
    // replay the loop-order dependence on the zones it can reach until the
    // flags settle: every sweep recomputes the list with the previous sweep's
    // flags; a zone newly flagged in a sweep brings its later neighbours
    // onto the list before the next one
    unsigned int nchg = 1;
    // no more workgroups than a list of the whole range has groups of 64
    const unsigned nlist = std::min<unsigned>(kListBlocks, grid_of(wr.count(), kReplayZones));
    for (int sw = 0; sw < kMaxSweeps && nchg > 0;) {
      for (int q = 0; q < kSweepBatch; ++q, ++sw) {
        k_cands<<<std::min<unsigned>(kCandBlocks, grid_of(wr.count(), 256)), 256, 0, st>>>(P, wr, F, sw);
        if (mom) {
          k_weno9_list<<<2 * kListBlocks, 128, 0, st>>>(P, F, wv, sw);
          k_weno_ao_list<<<2 * kListBlocks, 128, 0, st>>>(P, ao, mom, F, sw);
          k_pos10_list<<<kListBlocks, 256, 0, st>>>(P, F, mom, sw);
        } else {
          k_replay<<<nlist, kReplayThreads, 0, st>>>(P, F, wv, sw);
        }
      }
      P1_HIP(hipGetLastError());
      P1_HIP(hipMemcpyAsync(&nchg, F.ctr + 4 + sw - 1, sizeof(unsigned int), hipMemcpyDeviceToHost, st));
      P1_HIP(hipStreamSynchronize(st));
    }
    if (nchg > 0) {
      cs::set_error("cs_limit_all_slopes_p1: positivity replay did not settle");
      return CS_E_INVALID;
    }
    k_clear_ent<<<grid_of(wr.count(), 256), 256, 0, st>>>(P, wr, F.fl[0]);
  }
  if ((rc = mark())) return rc;
  if (mom)
    k_face_pts<10><<<dim3(grid_of(std::max(fx.count(), std::max(fy.count(), fz.count())), 256), 3), 256, 0, st>>>(
        P, fx, fy, fz, mom);
  else
    k_face_pts<4><<<dim3(grid_of(std::max(fx.count(), std::max(fy.count(), fz.count())), 256), 3), 256, 0, st>>>(
        P, fx, fy, fz, nullptr);
  if ((rc = mark())) return rc;
  if (mom) {
    k_clsq12<<<grid_of(wr.count(), kSqZones), 64, 0, st>>>(P, wr, mom);
    k_e12<<<grid_of(all.count(), 256), 256, 0, st>>>(P, all, mom);
  } else {
    k_clsq_e<<<grid_of(all.count(), 64), 64, 0, st>>>(P, all);
  }
  if ((rc = mark())) return rc;
  k_weno9<<<grid_of(wr.count(), 128), 128, 0, st>>>(P, wr, we);
  if (mom) {
    // 9.c in the loop order of the reference's serial build (k_ao_e_sweep);
    // k_ao_order flags a stencil table for which a zone's earlier neighbours
    // are not all on lower levels and its later ones all on higher levels
    // (F.ctr[2] and the sweep's ticket F.ctr[3] are clear since k_prim)
    double* xnew = aorec + (size_t)ao.count() * kAoRec;
    const int sj = ao_stride(ao.ni), threads = ((ao.ni + sj - 1) / sj * kAoLanes + 63) / 64 * 64 + 64;
    k_ao_order<<<grid_of((int64_t)ao.ni * ao.nj, 256), 256, 0, st>>>(P, ao, F.ctr + 2);
    k_ao_e_pre<<<grid_of(ao.count(), 128), 128, 0, st>>>(P, ao, mom, aorec, xnew);
    k_ao_e_sweep<<<ao.nk, threads, 0, st>>>(P, ao, aorec, xnew, F.ctr + 3, sj);
    k_ao_e_put<<<grid_of(ao.count(), 256), 256, 0, st>>>(P, ao, aorec);
  }
  if ((rc = mark())) return rc;
  k_diag<<<nblk_diag, DIAG_THREADS, 0, st>>>(P, all, part);
  if (p->V_min_local || p->V_max_local) k_diag_final<<<18, 256, 0, st>>>(part, nblk_diag, red);
  if ((rc = mark())) return rc;
  P1_HIP(hipGetLastError());
  if (kernel_ms) {
    P1_HIP(hipEventSynchronize(ev[nev - 1]));
    for (int q = 0; q + 1 < nev; ++q) P1_HIP(hipEventElapsedTime(&kernel_ms[q], ev[q], ev[q + 1]));
    for (int q = 0; q < NEV; ++q) (void)hipEventDestroy(ev[q]);
  }
  if (mom) {
    unsigned int bad = 0;
    P1_HIP(hipMemcpyAsync(&bad, F.ctr + 2, sizeof(unsigned int), hipMemcpyDeviceToHost, st));
    P1_HIP(hipStreamSynchronize(st));
    if (bad) {
      cs::set_error("cs_limit_all_slopes_p12: the stencil table breaks the level order of step 9.c (an entry "
                    "beyond two zones in i or j), so it cannot follow the serial loop order level by level");
      return CS_E_INVALID;
    }
  }
  if (p->V_min_local || p->V_max_local) {
    double h[18];
    P1_HIP(hipMemcpyAsync(h, red, sizeof(h), hipMemcpyDeviceToHost, st));
    P1_HIP(hipStreamSynchronize(st));
    for (int q = 0; q < 9; ++q) {
      if (p->V_min_local) p->V_min_local[q] = h[q];
      if (p->V_max_local) p->V_max_local[q] = h[9 + q];
    }
  }
  (void)own;
  return 0;
}

extern "C" int cs_limit_all_slopes_p1(const cs_p1_patch* p, void* stream) { return run_p1(p, stream, nullptr); }

extern "C" int cs_limit_all_slopes_p1_timed(const cs_p1_patch* p, void* stream, float* kernel_ms) {
  if (!kernel_ms) {
    cs::set_error("cs_limit_all_slopes_p1_timed: kernel_ms is null");
    return CS_E_INVALID;
  }
  return run_p1(p, stream, kernel_ms);
}

// Work memory of cs_limit_all_slopes_p1_noalloc: the positivity flags, the
// replay list and counters and the min/max partials live in this fixed
// array instead of a hipMalloc'd buffer.  Each device holds its own copy
// (from the module load until the process ends) at its own address, which
// the host must look up: the array's name is no device address in host code.
constexpr size_t kNoAllocBytes = (size_t)48 << 20;
__device__ __align__(256) uint8_t scratch[kNoAllocBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_na_mu;
uint8_t* g_na_ptr[kMaxDevices] = {};  // device address of scratch, per device
}  // namespace

extern "C" int cs_limit_all_slopes_p1_noalloc(const cs_p1_patch* p, void* stream) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    cs::set_error("cs_limit_all_slopes_p1_noalloc: no usable current device");
    return CS_E_HIP;
  }
  uint8_t* ptr = nullptr;
  {
    std::lock_guard<std::mutex> lk(g_na_mu);
    if (!g_na_ptr[dev]) {
      void* q = nullptr;
      const hipError_t e = hipGetSymbolAddress(&q, HIP_SYMBOL(scratch));
      if (e != hipSuccess || !q) {
        cs::set_error("cs_limit_all_slopes_p1_noalloc: hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
        return CS_E_HIP;
      }
      g_na_ptr[dev] = (uint8_t*)q;
    }
    ptr = g_na_ptr[dev];
  }
  return run_p1(p, stream, nullptr, ptr, kNoAllocBytes);
}

// ===========================================================================
// MAKE_FACIAL_FLUXES (400riemann_integrate/450make_facial_fluxes.f:5) for one
// patch at second order, behind cs_make_facial_fluxes_p1.
//
//   k_ff_face   one face of one family (blockIdx.y): the two zones' linear
//               fields at the face centroid, the face frame, the point Riemann
//               solver OneD_RS_MHD_Ptwise; S, fluctuations and entropy flux
//               written, and the two zones' shares of the update kept
//   k_ff_gather one zone: dU_dt from the shares of its six faces, in the
//               reference's order (x-faces, then y, then z; lower face first)
//   k_ff_remap  the few zones that also take the share of a face whose own
//               zone on that side is a tri-corner zone (the face then points
//               at the stencil neighbour): dU_dt rebuilt with those shares in
//               the order of the reference's loops
namespace csp1 {

struct P1F {
  cs_p1_flux a;
  int N, NR, g, nz, nzr, nf, nfr;
  int64_t NZ, NXF, NZF, NFC;
  __device__ __forceinline__ int64_t zi(int i, int j, int k) const {
    return (int64_t)(i - 1 + g) + (int64_t)nz * ((j - 1 + g) + (int64_t)nz * (k - 1 + g));
  }
  __device__ __forceinline__ int64_t fci(int i, int j, int k) const {
    return (int64_t)(i + g) + (int64_t)nf * ((j + g) + (int64_t)nf * (k + g));
  }
  __device__ __forceinline__ int64_t xfi(int i, int j, int k) const {
    return (int64_t)(i + g) + (int64_t)nf * ((j - 1 + g) + (int64_t)nz * (k - 1 + g));
  }
  __device__ __forceinline__ int64_t yfi(int i, int j, int k) const {
    return (int64_t)(i - 1 + g) + (int64_t)nz * ((j + g) + (int64_t)nf * (k - 1 + g));
  }
  __device__ __forceinline__ int64_t zfi(int i, int j, int k) const {
    return (int64_t)(i - 1 + g) + (int64_t)nz * ((j - 1 + g) + (int64_t)nz * (k + g));
  }
  __device__ __forceinline__ void nbr(int i, int j, int n, int& ni, int& nj) const {
    const int64_t s = (int64_t)(i - 1 + g) + (int64_t)nz * (j - 1 + g), plane = (int64_t)nz * nz;
    ni = min(max(a.stencil[s + plane * (2 * n)], 1 - g), N + g);
    nj = min(max(a.stencil[s + plane * (2 * n + 1)], 1 - g), N + g);
  }
  __device__ __forceinline__ bool active(int i, int j, int k) const { return a.mask[zi(i, j, k)] == 1; }
  __device__ __forceinline__ double obl(int64_t z) const { return 1.0 / fmax(a.scale[z], a.smallnum); }
  // face range of family fam (the reference's loops with iexpand = 1)
  __device__ __forceinline__ bool in_range(int fam, int i, int j, int k) const {
    return i >= (fam == 0 ? -1 : 0) && i <= N + 1 && j >= (fam == 1 ? -1 : 0) && j <= N + 1 &&
           k >= (fam == 2 ? -1 : 0) && k <= NR + 1;
  }
};

// OneD_RS_MHD_Ptwise with every output (610...f:96-220, 644-704), face frame
__device__ __forceinline__ void rs_ptwise(const Gas<double>& gs, double* VL, double* VR, double entL, double entR,
                                          double& SL, double& SR, double& entF, double* FlL, double* FlR,
                                          double* FL, double* FR) {
  const double bx = 0.5 * (VL[5] + VR[5]);
  VL[5] = bx;
  VR[5] = bx;
  double UL[8], UR[8], Vm[8];
  prim_to_cons(gs, entL, VL, UL);
  prim_to_cons(gs, entR, VR, UR);
  flux_x(VL, UL, FL);
  flux_x(VR, UR, FR);
  double smin, smax;
  SR = -1e30;
  SL = 1e30;
  wavspd_x(gs, VL, smin, smax);
  SL = fmin(SL, smin);
  SR = fmax(SR, smax);
  wavspd_x(gs, VR, smin, smax);
  SL = fmin(SL, smin);
  SR = fmax(SR, smax);
#pragma unroll
  for (int c = 0; c < 8; ++c) Vm[c] = 0.5 * (VL[c] + VR[c]);
  wavspd_x(gs, Vm, smin, smax);
  SL = fmin(SL, smin);
  SR = fmax(SR, smax);
  if (SL >= 0.0) {
    // U* = U_L before the one-sided fluctuation is formed (610...f:653-658)
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      FlR[c] = SR * (UR[c] - UL[c]);
      FlL[c] = 0.0;
    }
    entF = entL * VL[1];
    return;
  }
  if (SR <= 0.0) {
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      FlL[c] = SL * (UR[c] - UL[c]);
      FlR[c] = 0.0;
    }
    entF = entR * VR[1];
    return;
  }
  const double t3 = 1.0 / (SR - SL), t1 = SR * t3, t2 = SL * t3;
  double Us[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) Us[c] = t1 * UR[c] - t2 * UL[c] - t3 * (FR[c] - FL[c]);
  const double entUs = t1 * entR - t2 * entL - t3 * (entR * VR[1] - entL * VL[1]);
  const double pent = entUs * rpow_gm1(gs, Us[0]);
  const double peng = gs.gm1 * (Us[4] - 0.5 * (Us[1] * Us[1] + Us[2] * Us[2] + Us[3] * Us[3]) / Us[0] -
                                C<double>::ob8pi * (Us[5] * Us[5] + Us[6] * Us[6] + Us[7] * Us[7]));
  if (peng <= gs.prsfloor) Us[4] = Us[4] + (pent - peng) * gs.igm1;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    FlL[c] = SL * (Us[c] - UL[c]);
    FlR[c] = SR * (UR[c] - Us[c]);
  }
  const double o = 1.0 / (SR - SL);
  entF = (SR * entL * VL[1] - SL * entR * VR[1]) * o + (entR - entL) * (SR * SL * o);
}

// one face; the shares cl (to the left zone) and cr (to the right) are kept
// in share[fam][c][face] (c < 8 left, c >= 8 right); faces whose side zone was
// re-pointed through the stencil join that zone's list: entry e holds
// (face, family, side) and the entry before it in the zone's list
struct FfList {
  int64_t *zone, *code;  // [entry], cap of them
  int32_t* next;         // [entry]
  int32_t* head;         // [zone] the zone's latest entry, -1: none
  unsigned int* count;
  __host__ __device__ FfList(int64_t* list, int64_t cap, unsigned int* n)
      : zone(list), code(list + cap), next((int32_t*)(list + 2 * cap)), head(next + cap), count(n) {}
};
__global__ void __launch_bounds__(128) k_ff_face(const P1F P, double* share, int64_t* rlist, int64_t cap,
                                                 unsigned int* rcount) {
  const int fam = blockIdx.y;
  const int64_t t = tid();
  if (t >= P.NFC) return;
  const int n = P.nf;
  const int i = (int)(t % n) - P.g, j = (int)((t / n) % n) - P.g, k = (int)(t / ((int64_t)n * n)) - P.g;
  const cs_p1_flux& a = P.a;
  const int64_t fb = t;
  double* FPl = fam == 0 ? a.Fluct_x_Pl : (fam == 1 ? a.Fluct_y_Pl : a.Fluct_z_Pl);
  double* FMi = fam == 0 ? a.Fluct_x_Mi : (fam == 1 ? a.Fluct_y_Mi : a.Fluct_z_Mi);
  // faces outside the range or between two tri-corner zones keep zero
  // fluctuations (450...f:370-380)
  auto zero = [&]() {
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      FPl[fb + P.NFC * c] = 0.0;
      FMi[fb + P.NFC * c] = 0.0;
    }
  };
  if (!P.in_range(fam, i, j, k)) {
    zero();
    return;
  }
  int li = i, lj = j, ri = i + (fam == 0), rj = j + (fam == 1);
  const int rk = k + (fam == 2);
  int remapped = 0;  // 1: left side re-pointed, 2: right side
  if (fam < 2) {
    const bool al = P.active(li, lj, k), ar = P.active(ri, rj, k);
    if (!al && ar) {
      P.nbr(ri, rj, fam == 0 ? 1 : 3, li, lj);
      remapped = 1;
    } else if (al && !ar) {
      P.nbr(li, lj, fam == 0 ? 0 : 2, ri, rj);
      remapped = 2;
    } else if (!al && !ar) {
      zero();
      return;
    }
  } else if (!P.active(i, j, k)) {
    zero();
    return;
  }
  const int64_t zl = P.zi(li, lj, k), zr = P.zi(ri, rj, fam == 2 ? rk : k);
  const int64_t fg = fam == 0 ? P.xfi(i, j, k) : (fam == 1 ? P.yfi(i, j, k) : P.zfi(i, j, k));
  const int64_t NF = fam == 2 ? P.NZF : P.NXF;
  const double* nrm = fam == 0 ? a.xf_normal : (fam == 1 ? a.yf_normal : a.zf_normal);
  const double* fcen = fam == 0 ? a.xf_centroid : (fam == 1 ? a.yf_centroid : a.zf_centroid);
  const double* pts = fam == 0 ? a.xf_pts : (fam == 1 ? a.yf_pts : a.zf_pts);
  const double sm = a.smallnum;
  double A[3], B[3], Cv[3];
  if (fam == 0) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      A[c] = nrm[fg + NF * c];
      Cv[c] = fcen[fg + NF * c];
    }
    const double s = 1.0 / fmax(sqrt(Cv[0] * Cv[0] + Cv[1] * Cv[1] + Cv[2] * Cv[2]), sm);
#pragma unroll
    for (int c = 0; c < 3; ++c) Cv[c] = Cv[c] * s;
    B[0] = Cv[1] * A[2] - Cv[2] * A[1];
    B[1] = Cv[2] * A[0] - Cv[0] * A[2];
    B[2] = Cv[0] * A[1] - Cv[1] * A[0];
  } else if (fam == 1) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      A[c] = nrm[fg + NF * c];
      B[c] = fcen[fg + NF * c];
    }
    const double s = 1.0 / fmax(sqrt(B[0] * B[0] + B[1] * B[1] + B[2] * B[2]), sm);
#pragma unroll
    for (int c = 0; c < 3; ++c) B[c] = B[c] * s;
    Cv[0] = A[1] * B[2] - A[2] * B[1];
    Cv[1] = A[2] * B[0] - A[0] * B[2];
    Cv[2] = A[0] * B[1] - A[1] * B[0];
  } else {
#pragma unroll
    for (int c = 0; c < 3; ++c) A[c] = nrm[fg + NF * c];
    double s = 1.0 / fmax(sqrt(A[0] * A[0] + A[1] * A[1] + A[2] * A[2]), sm);
#pragma unroll
    for (int c = 0; c < 3; ++c) A[c] = A[c] * s;
#pragma unroll
    for (int c = 0; c < 3; ++c)
      B[c] = a.vert[P.fci(i, j, k) + P.NFC * c] + a.vert[P.fci(i, j - 1, k) + P.NFC * c] -
             a.vert[P.fci(i - 1, j, k) + P.NFC * c] - a.vert[P.fci(i - 1, j - 1, k) + P.NFC * c];
    s = B[0] * A[0] + B[1] * A[1] + B[2] * A[2];
#pragma unroll
    for (int c = 0; c < 3; ++c) B[c] = B[c] - s * A[c];
    s = 1.0 / fmax(sqrt(B[0] * B[0] + B[1] * B[1] + B[2] * B[2]), sm);
#pragma unroll
    for (int c = 0; c < 3; ++c) B[c] = B[c] * s;
    Cv[0] = A[1] * B[2] - A[2] * B[1];
    Cv[1] = A[2] * B[0] - A[0] * B[2];
    Cv[2] = A[0] * B[1] - A[1] * B[0];
    s = 1.0 / fmax(sqrt(Cv[0] * Cv[0] + Cv[1] * Cv[1] + Cv[2] * Cv[2]), sm);
#pragma unroll
    for (int c = 0; c < 3; ++c) Cv[c] = Cv[c] * s;
    B[0] = Cv[1] * A[2] - Cv[2] * A[1];
    B[1] = Cv[2] * A[0] - Cv[0] * A[2];
    B[2] = Cv[0] * A[1] - Cv[1] * A[0];
  }
  // both zones' linear fields at the face centroid, into the face frame
  double VL[8], VR[8], eL, eR;
  {
    const double ol = P.obl(zl), orr = P.obl(zr);
    double rl[3], rr[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double x = pts[fg + NF * c];
      rl[c] = (x - a.v_centroid[zl + P.NZ * c]) * ol;
      rr[c] = (x - a.v_centroid[zr + P.NZ * c]) * orr;
    }
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const double* v = a.V + P.NZ * c;
      VL[c] = v[zl] + v[zl + 8 * P.NZ] * rl[0] + v[zl + 16 * P.NZ] * rl[1] + v[zl + 24 * P.NZ] * rl[2];
      VR[c] = v[zr] + v[zr + 8 * P.NZ] * rr[0] + v[zr + 16 * P.NZ] * rr[1] + v[zr + 24 * P.NZ] * rr[2];
    }
    eL = a.ent[zl] + a.ent[zl + P.NZ] * rl[0] + a.ent[zl + 2 * P.NZ] * rl[1] + a.ent[zl + 3 * P.NZ] * rl[2];
    eR = a.ent[zr] + a.ent[zr + P.NZ] * rr[0] + a.ent[zr + 2 * P.NZ] * rr[1] + a.ent[zr + 3 * P.NZ] * rr[2];
#pragma unroll
    for (int o = 1; o <= 5; o += 4) {
      const double la = A[0] * VL[o] + A[1] * VL[o + 1] + A[2] * VL[o + 2];
      const double lb = B[0] * VL[o] + B[1] * VL[o + 1] + B[2] * VL[o + 2];
      const double lc = Cv[0] * VL[o] + Cv[1] * VL[o + 1] + Cv[2] * VL[o + 2];
      VL[o] = la;
      VL[o + 1] = lb;
      VL[o + 2] = lc;
      const double ra = A[0] * VR[o] + A[1] * VR[o + 1] + A[2] * VR[o + 2];
      const double rb = B[0] * VR[o] + B[1] * VR[o + 1] + B[2] * VR[o + 2];
      const double rc = Cv[0] * VR[o] + Cv[1] * VR[o + 1] + Cv[2] * VR[o + 2];
      VR[o] = ra;
      VR[o + 1] = rb;
      VR[o + 2] = rc;
    }
  }
  const Gas<double> gs{a.gamma, a.gamma - 1.0, a.rhofloor, a.prsfloor, 1.0 / (a.gamma - 1.0)};
  double SL, SR, eF, FlL[8], FlR[8], FL[8], FR[8];
  rs_ptwise(gs, VL, VR, eL, eR, SL, SR, eF, FlL, FlR, FL, FR);
  (fam == 0 ? a.S_L : fam == 1 ? a.S_D : a.S_B)[fb] = SL;
  (fam == 0 ? a.S_R : fam == 1 ? a.S_U : a.S_T)[fb] = SR;
  (fam == 0 ? a.EntFlux_x : fam == 1 ? a.EntFlux_y : a.EntFlux_z)[fb] = eF;
  const double ar = (fam == 0 ? a.xf_area : fam == 1 ? a.yf_area : a.zf_area)[fg];
  const double vl = a.v_volume[zl], vr = a.v_volume[zr];
  double* sh = share + (int64_t)fam * 16 * P.NFC;
  // back to the global frame: scalars as they are, vectors through (A, B, C)
  auto back = [&](const double* f, int c) -> double {
    if (c == 0 || c == 4) return f[c];
    const int o = c < 4 ? 1 : 5, q = c - o;
    return A[q] * f[o] + B[q] * f[o + 1] + Cv[q] * f[o + 2];
  };
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const double pl = back(FlR, c), mi = back(FlL, c), fll = back(FL, c), frr = back(FR, c);
    FPl[fb + P.NFC * c] = pl;
    FMi[fb + P.NFC * c] = mi;
    sh[fb + P.NFC * c] = (mi + fll) * ar / vl;
    sh[fb + P.NFC * (8 + c)] = (pl - frr) * ar / vr;
  }
  if (remapped) {
    const FfList R(rlist, cap, rcount);
    const unsigned int e = atomicAdd(R.count, 1u);
    const int64_t T = remapped == 1 ? zl : zr;
    R.zone[e] = T;
    R.code[e] = (((int64_t)fam * P.NFC + fb) << 1) | (remapped == 1 ? 0 : 1);
    R.next[e] = atomicExch(&R.head[T], (int32_t)e);
  }
}

// dU_dt of one zone from its own faces: x lower (as right zone), x upper (as
// left zone), then y, then z
__global__ void __launch_bounds__(256) k_ff_gather(const P1F P, const double* share) {
  const int64_t z = tid();
  if (z >= P.NZ) return;
  const int i = (int)(z % P.nz) + 1 - P.g, j = (int)((z / P.nz) % P.nz) + 1 - P.g,
            k = (int)(z / ((int64_t)P.nz * P.nz)) + 1 - P.g;
  double d[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) d[c] = 0.0;
  // a tri-corner zone takes no share of any face
  const bool act = P.active(i, j, k);
#pragma unroll
  for (int fam = 0; fam < 3; ++fam) {
    if (!act) break;
    const double* sh = share + (int64_t)fam * 16 * P.NFC;
    const int di = fam == 0, dj = fam == 1, dk = fam == 2;
    if (P.in_range(fam, i - di, j - dj, k - dk)) {
      const int64_t f = P.fci(i - di, j - dj, k - dk);
#pragma unroll
      for (int c = 0; c < 8; ++c) d[c] = d[c] - sh[f + P.NFC * (8 + c)];
    }
    if (P.in_range(fam, i, j, k)) {
      const int64_t f = P.fci(i, j, k);
#pragma unroll
      for (int c = 0; c < 8; ++c) d[c] = d[c] - sh[f + P.NFC * c];
    }
  }
#pragma unroll
  for (int c = 0; c < 8; ++c) P.a.dU_dt[z + P.NZ * c] = d[c];
}

// dU_dt of zone T, whose list starts at entry e0
__device__ __forceinline__ void ff_rebuild(const P1F& P, const double* share, const FfList& R, int64_t T, int32_t e0) {
  const int i = (int)(T % P.nz) + 1 - P.g, j = (int)((T / P.nz) % P.nz) + 1 - P.g,
            k = (int)(T / ((int64_t)P.nz * P.nz)) + 1 - P.g;
  double d[8];
  for (int c = 0; c < 8; ++c) d[c] = 0.0;
  for (int fam = 0; fam < 3; ++fam) {
    // the shares reaching T in this family: (face, side), sorted by face
    int64_t fc[8];
    int sd[8], m = 0;
    const int di = fam == 0, dj = fam == 1, dk = fam == 2;
    if (P.active(i, j, k)) {
      if (P.in_range(fam, i - di, j - dj, k - dk)) {
        fc[m] = P.fci(i - di, j - dj, k - dk);
        sd[m++] = 1;
      }
      if (P.in_range(fam, i, j, k)) {
        fc[m] = P.fci(i, j, k);
        sd[m++] = 0;
      }
    }
    for (int32_t q = e0; q >= 0 && m < 8; q = R.next[q]) {
      const int64_t code = R.code[q], ff = code >> 1;
      if (ff / P.NFC != fam) continue;
      fc[m] = ff % P.NFC;
      sd[m++] = (int)(code & 1);
    }
    for (int a1 = 1; a1 < m; ++a1)  // insertion sort by face index
      for (int b1 = a1; b1 > 0 && fc[b1] < fc[b1 - 1]; --b1) {
        const int64_t tf = fc[b1];
        fc[b1] = fc[b1 - 1];
        fc[b1 - 1] = tf;
        const int ts = sd[b1];
        sd[b1] = sd[b1 - 1];
        sd[b1 - 1] = ts;
      }
    const double* sh = share + (int64_t)fam * 16 * P.NFC;
    for (int q = 0; q < m; ++q)
      for (int c = 0; c < 8; ++c) d[c] = d[c] - sh[fc[q] + P.NFC * (8 * sd[q] + c)];
  }
  for (int c = 0; c < 8; ++c) P.a.dU_dt[T + P.NZ * c] = d[c];
}

// zones that also take re-pointed shares: dU_dt rebuilt in loop order, one
// thread per such zone, the thread of its list's head.  Grid-stride over the
// entries, whose number stays on the device: the host neither waits for it
// nor groups them (fluxes, edge fields and sources of a 95^2 x 33 patch with
// the host's grouping 398 us, without 324; the driver's step on six 24^2 x 8
// patches 5.3 -> 4.3 ms).
__global__ void __launch_bounds__(64) k_ff_remap(const P1F P, const double* share, const FfList R) {
  const int64_t n = *R.count;
  for (int64_t t = tid(); t < n; t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t T = R.zone[t];
    if (R.head[T] == (int32_t)t) ff_rebuild(P, share, R, T, (int32_t)t);
  }
}

// the electric fields of the zone range, the zones' lists and their count
__global__ void __launch_bounds__(256) k_ff_zero_e(const P1F P, const FfList R) {
  const int64_t z = tid();
  if (z >= P.NZ) return;
  R.head[z] = -1;
  if (z == 0) *R.count = 0;
  const int i = (int)(z % P.nz) + 1 - P.g, j = (int)((z / P.nz) % P.nz) + 1 - P.g,
            k = (int)(z / ((int64_t)P.nz * P.nz)) + 1 - P.g;
  const int64_t f = P.fci(i, j, k);
  P.a.Efx[f] = 0.0;
  P.a.Efy[f] = 0.0;
  P.a.Efz[f] = 0.0;
}

static std::vector<Scratch> g_ff_scratch;

}  // namespace csp1

extern "C" int cs_make_facial_fluxes_p1(const cs_p1_flux* p, void* stream_) {
  if (!p) {
    cs::set_error("cs_make_facial_fluxes_p1: null argument");
    return CS_E_INVALID;
  }
  if (p->ntp < 1 || p->nr < 1 || p->nghost < 4) {
    cs::set_error("cs_make_facial_fluxes_p1: need ntp >= 1, nr >= 1, nghost >= 4 (got %d, %d, %d)", p->ntp, p->nr,
                  p->nghost);
    return CS_E_INVALID;
  }
  if (p->nghost >= p->ntp) {
    cs::set_error("cs_make_facial_fluxes_p1: nghost (%d) must be below ntp (%d)", p->nghost, p->ntp);
    return CS_E_BAD_DECOMP;
  }
  if (!(p->gamma > 1.0) || !(p->smallnum > 0.0) || !(p->rhofloor > 0.0) || !(p->prsfloor > 0.0)) {
    cs::set_error("cs_make_facial_fluxes_p1: gamma > 1 and positive floors and smallnum required");
    return CS_E_INVALID;
  }
  const void* ptrs[] = {p->vert, p->mask, p->stencil, p->xf_pts, p->xf_normal, p->xf_area, p->xf_centroid,
                        p->yf_pts, p->yf_normal, p->yf_area, p->yf_centroid, p->zf_pts, p->zf_normal, p->zf_area,
                        p->zf_centroid, p->scale, p->v_volume, p->v_centroid, p->V, p->ent, p->flatten, p->S_L,
                        p->S_R, p->S_D, p->S_U, p->S_B, p->S_T, p->Fluct_x_Pl, p->Fluct_y_Pl, p->Fluct_z_Pl,
                        p->Fluct_x_Mi, p->Fluct_y_Mi, p->Fluct_z_Mi, p->dU_dt, p->EntFlux_x, p->EntFlux_y,
                        p->EntFlux_z, p->Efx, p->Efy, p->Efz};
  for (const void* q : ptrs)
    if (!q) {
      cs::set_error("cs_make_facial_fluxes_p1: null array");
      return CS_E_INVALID;
    }
  hipStream_t st = (hipStream_t)stream_;
  P1F P;
  P.a = *p;
  P.N = p->ntp;
  P.NR = p->nr;
  P.g = p->nghost;
  P.nz = P.N + 2 * P.g;
  P.nzr = P.NR + 2 * P.g;
  P.nf = P.nz + 1;
  P.nfr = P.nzr + 1;
  P.NZ = (int64_t)P.nz * P.nz * P.nzr;
  P.NXF = (int64_t)P.nf * P.nz * P.nzr;
  P.NZF = (int64_t)P.nz * P.nz * P.nfr;
  P.NFC = (int64_t)P.nf * P.nf * P.nfr;
  int dev = 0, rc;
  P1_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(g_mu);
  if ((int)g_ff_scratch.size() <= dev) g_ff_scratch.resize(dev + 1);
  Scratch& S = g_ff_scratch[dev];
  const size_t share_bytes = (size_t)48 * P.NFC * sizeof(double);
  const size_t list_cap = (size_t)2 * P.NFC;  // faces of two families at most
  const size_t need = share_bytes + 256 + list_cap * (2 * sizeof(int64_t) + sizeof(int32_t)) + P.NZ * sizeof(int32_t);
  if ((rc = scratch_open(S, need, st, "cs_make_facial_fluxes_p1"))) return rc;
  const ScratchUse use{&S, st};
  double* share = (double*)S.mem;
  unsigned int* rcount = (unsigned int*)((uint8_t*)S.mem + share_bytes);
  int64_t* rlist = (int64_t*)((uint8_t*)S.mem + share_bytes + 256);
  const FfList R(rlist, (int64_t)list_cap, rcount);
  // the face kernel writes every fluctuation (zero where no Riemann problem
  // is solved) and the gather every zone's update; the electric fields of
  // the zone range are zeroed (450...f:400-420)
  k_ff_zero_e<<<grid_of(P.NZ, 256), 256, 0, st>>>(P, R);
  k_ff_face<<<dim3(grid_of(P.NFC, 128), 3), 128, 0, st>>>(P, share, rlist, (int64_t)list_cap, rcount);
  k_ff_gather<<<grid_of(P.NZ, 256), 256, 0, st>>>(P, share);
  k_ff_remap<<<64, 64, 0, st>>>(P, share, R);
  P1_HIP(hipGetLastError());
  return 0;
}

// ===========================================================================
// UPDATE_IMEX_RK_STEP_P1 (400riemann_integrate/484update_imex_rk_step_p1.f:7),
// MHD, behind cs_update_imex_rk_step_p1:
//   k_upd_zone  every zone: U += dt dU_dt (:483-489); owned zones: entropy from
//               the face entropy fluxes, CONS_TO_PRIM, its flag (:540-628)
//   k_upd_face  owned faces of one family (blockIdx.y): constrained transport
//               with the edges' radial lengths and arc lengths (:630-906)
namespace csp1 {

struct P1U {
  cs_p1_update a;
  int N, NR, g, nz, nf;
  int64_t NZ, NXF, NZF, NFC;
  __device__ __forceinline__ int64_t fci(int i, int j, int k) const {
    return (int64_t)(i + g) + (int64_t)nf * ((j + g) + (int64_t)nf * (k + g));
  }
  __device__ __forceinline__ int64_t xfi(int i, int j, int k) const {
    return (int64_t)(i + g) + (int64_t)nf * ((j - 1 + g) + (int64_t)nz * (k - 1 + g));
  }
  __device__ __forceinline__ int64_t yfi(int i, int j, int k) const {
    return (int64_t)(i - 1 + g) + (int64_t)nz * ((j + g) + (int64_t)nf * (k - 1 + g));
  }
  __device__ __forceinline__ int64_t zfi(int i, int j, int k) const {
    return (int64_t)(i - 1 + g) + (int64_t)nz * ((j - 1 + g) + (int64_t)nz * (k + g));
  }
  __device__ __forceinline__ double vx(int i, int j, int k, int c) const { return a.vert[fci(i, j, k) + NFC * c]; }
  __device__ __forceinline__ double rad(int i, int j, int k) const {
    const double x = vx(i, j, k, 0), y = vx(i, j, k, 1), z = vx(i, j, k, 2);
    return sqrt(x * x + y * y + z * z);
  }
  // arc between vertices (i1, j1) and (i2, j2) of level k: both directions
  // scaled by t = 1 / (radius of the face's own vertex), as the reference does
  __device__ __forceinline__ double angle(int i1, int j1, int i2, int j2, int k, double t) const {
    const double d = (vx(i1, j1, k, 0) * t) * (vx(i2, j2, k, 0) * t) + (vx(i1, j1, k, 1) * t) * (vx(i2, j2, k, 1) * t) +
                     (vx(i1, j1, k, 2) * t) * (vx(i2, j2, k, 2) * t);
    return acos(d);
  }
};

__global__ void __launch_bounds__(256) k_upd_zone(const P1U P) {
  const int64_t z = tid();
  if (z >= P.NZ) return;
  const cs_p1_update& a = P.a;
  const int i = (int)(z % P.nz) + 1 - P.g, j = (int)((z / P.nz) % P.nz) + 1 - P.g,
            k = (int)(z / ((int64_t)P.nz * P.nz)) + 1 - P.g;
  const double dt = a.dtmove;
  double U[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) U[c] = a.U[z + P.NZ * c] + dt * a.dU_dt[z + P.NZ * c];
  double flag = 0.0;
  if (i >= 1 && i <= P.N && j >= 1 && j <= P.N && k >= 1 && k <= P.NR) {
    const double s = a.xf_area[P.xfi(i, j, k)] * a.EntFlux_x[P.fci(i, j, k)] -
                     a.xf_area[P.xfi(i - 1, j, k)] * a.EntFlux_x[P.fci(i - 1, j, k)] +
                     a.yf_area[P.yfi(i, j, k)] * a.EntFlux_y[P.fci(i, j, k)] -
                     a.yf_area[P.yfi(i, j - 1, k)] * a.EntFlux_y[P.fci(i, j - 1, k)] +
                     a.zf_area[P.zfi(i, j, k)] * a.EntFlux_z[P.fci(i, j, k)] -
                     a.zf_area[P.zfi(i, j, k - 1)] * a.EntFlux_z[P.fci(i, j, k - 1)];
    double e = a.ent[z] - dt * s / a.v_volume[z];
    const Gas<double> gs{a.gamma, a.gamma - 1.0, a.rhofloor, a.prsfloor, 1.0 / (a.gamma - 1.0)};
    double V[8];
    flag = (double)cons_to_prim(gs, U, V, e);
    a.ent[z] = e;
  }
#pragma unroll
  for (int c = 0; c < 8; ++c) a.U[z + P.NZ * c] = U[c];
  a.flag_entprs[z] = flag;
}

__global__ void __launch_bounds__(256) k_upd_face(const P1U P) {
  const int fam = blockIdx.y;
  const int64_t t = tid();
  const int N = P.N, NR = P.NR;
  // owned faces: x (0..N, 1..N, 1..NR), y (1..N, 0..N, 1..NR), z (1..N, 1..N, 0..NR)
  const int ni = fam == 0 ? N + 1 : N, nj = fam == 1 ? N + 1 : N, nk = fam == 2 ? NR + 1 : NR;
  if (t >= (int64_t)ni * nj * nk) return;
  const int i = (int)(t % ni) + (fam == 0 ? 0 : 1), j = (int)((t / ni) % nj) + (fam == 1 ? 0 : 1),
            k = (int)(t / ((int64_t)ni * nj)) + (fam == 2 ? 0 : 1);
  const cs_p1_update& a = P.a;
  const double dt = a.dtmove;
  const int64_t f = P.fci(i, j, k);
  const double rout = P.rad(i, j, k), tt = 1.0 / rout;
  if (fam == 0) {
    const double rin = P.rad(i, j, k - 1), dr = rout - rin, th = P.angle(i, j, i, j - 1, k, tt);
    const double lin = rin * th, lout = rout * th;
    a.Bxf[f] = a.Bxf[f] - dt * (dr * a.Efz[f] - dr * a.Efz[P.fci(i, j - 1, k)] - lout * a.Efy[f] +
                                lin * a.Efy[P.fci(i, j, k - 1)]) / a.xf_area[P.xfi(i, j, k)];
  } else if (fam == 1) {
    const double rin = P.rad(i, j, k - 1), dr = rout - rin, th = P.angle(i, j, i - 1, j, k, tt);
    const double lin = rin * th, lout = rout * th;
    a.Byf[f] = a.Byf[f] - dt * (-(dr * a.Efz[f]) + dr * a.Efz[P.fci(i - 1, j, k)] + lout * a.Efx[f] -
                                lin * a.Efx[P.fci(i, j, k - 1)]) / a.yf_area[P.yfi(i, j, k)];
  } else {
    const double lxp = rout * P.angle(i, j, i - 1, j, k, tt), lxm = rout * P.angle(i, j - 1, i - 1, j - 1, k, tt);
    const double lyp = rout * P.angle(i, j, i, j - 1, k, tt), lym = rout * P.angle(i - 1, j, i - 1, j - 1, k, tt);
    a.Bzf[f] = a.Bzf[f] - dt * (lyp * a.Efy[f] - lym * a.Efy[P.fci(i - 1, j, k)] - lxp * a.Efx[f] +
                                lxm * a.Efx[P.fci(i, j - 1, k)]) / a.zf_area[P.zfi(i, j, k)];
  }
}

}  // namespace csp1

extern "C" int cs_update_imex_rk_step_p1(const cs_p1_update* p, void* stream_) {
  if (!p) {
    cs::set_error("cs_update_imex_rk_step_p1: null argument");
    return CS_E_INVALID;
  }
  if (p->ntp < 1 || p->nr < 1 || p->nghost < 1) {
    cs::set_error("cs_update_imex_rk_step_p1: need ntp, nr, nghost >= 1 (got %d, %d, %d)", p->ntp, p->nr,
                  p->nghost);
    return CS_E_INVALID;
  }
  if (!(p->gamma > 1.0) || !(p->rhofloor > 0.0) || !(p->prsfloor > 0.0)) {
    cs::set_error("cs_update_imex_rk_step_p1: gamma > 1 and positive floors required");
    return CS_E_INVALID;
  }
  const void* ptrs[] = {p->vert, p->xf_area, p->yf_area, p->zf_area, p->v_volume, p->U, p->ent, p->Bxf,
                        p->Byf, p->Bzf, p->dU_dt, p->EntFlux_x, p->EntFlux_y, p->EntFlux_z, p->Efx, p->Efy,
                        p->Efz, p->flag_entprs};
  for (const void* q : ptrs)
    if (!q) {
      cs::set_error("cs_update_imex_rk_step_p1: null array");
      return CS_E_INVALID;
    }
  hipStream_t st = (hipStream_t)stream_;
  P1U P;
  P.a = *p;
  P.N = p->ntp;
  P.NR = p->nr;
  P.g = p->nghost;
  P.nz = P.N + 2 * P.g;
  P.nf = P.nz + 1;
  const int nzr = P.NR + 2 * P.g;
  P.NZ = (int64_t)P.nz * P.nz * nzr;
  P.NXF = (int64_t)P.nf * P.nz * nzr;
  P.NZF = (int64_t)P.nz * P.nz * (nzr + 1);
  P.NFC = (int64_t)P.nf * P.nf * (nzr + 1);
  const int64_t nfaces = (int64_t)(P.N + 1) * (P.N + 1) * (P.NR + 1);
  k_upd_zone<<<grid_of(P.NZ, 256), 256, 0, st>>>(P);
  k_upd_face<<<dim3(grid_of(nfaces, 256), 3), 256, 0, st>>>(P);
  P1_HIP(hipGetLastError());
  return 0;
}

// ---------------------------------------------------------------------------
// CLEANUP_AFTER_UPDATE (cubesphere/400riemann_integrate/485cleanup_after_update.f:1)
// and EVALUATE_TIMESTEP (490evaluate_timestep.f:1) of one patch, MHD, on the
// fields of cs_p1_patch:
//   k_face_zero, k_tricorner  steps 2 (faces) and 3 of the cleanup: the
//                             reconstruction's kernels, whose ranges and rules
//                             are the same (485...f:366-686)
//   k_cleanup_zone            step 2 (zones), step 4.a: the zone B as the least-
//                             squares fit of the six face values over the face
//                             normals, the energy rebalanced (:691-865), and
//                             step 5: CONS_TO_PRIM of every zone (:1180-1280)
//   k_dt_init, k_dt           CONS_TO_PRIM of the owned active zones, their
//                             magnetosonic speed, and the minimum of
//                             cfl l / (|v| + c_f) with 1.1 dt (490...f:72-163):
//                             a block minimum, folded into the output by a
//                             compare-and-swap minimum (positive values, so
//                             the result does not depend on the block order)
namespace csp1 {

__global__ void __launch_bounds__(256) k_cleanup_zone(const P1 P) {
  const int64_t z = tid();
  if (z >= P.NZ) return;
  const cs_p1_patch& a = P.a;
  const int i = (int)(z % P.nz) + 1 - P.g, j = (int)((z / P.nz) % P.nz) + 1 - P.g,
            k = (int)(z / ((int64_t)P.nz * P.nz)) + 1 - P.g;
  const double gam = a.gamma;
  a.gamma_eos[z] = gam;
  a.gamma_sound[z] = gam;
  a.mean_mol_wt[z] = a.molewt;
#pragma unroll
  for (int c = 0; c < 8; ++c)
#pragma unroll
    for (int m = 1; m < 4; ++m) {
      P.Ur(c, m, z) = 0.0;
      P.Vr(c, m, z) = 0.0;
    }
#pragma unroll
  for (int m = 1; m < 4; ++m) a.ent[z + P.NZ * m] = 0.0;
  double U[8], was[8], V[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) was[c] = P.Ur(c, 0, z);
  if (a.mask[z] == 0) {
#pragma unroll
    for (int c = 0; c < 8; ++c) U[c] = 0.0;
    U[0] = a.rhofloor;
    U[4] = a.prsfloor / (gam - 1.0);
    a.scale[z] = a.smallnum;
  } else {
#pragma unroll
    for (int c = 0; c < 8; ++c) U[c] = was[c];
  }
  if (P.active(i, j, 1)) {
    // rows: x+ and x- face normals, y+ and y-, and the radial direction of
    // the zone's upper z-face centroid for both z-faces
    double A[6][3], R[6];
    const int64_t fz = P.zfi(i, j, k), xp = P.xfi(i, j, k), xm = P.xfi(i - 1, j, k), yp = P.yfi(i, j, k),
                  ym = P.yfi(i, j - 1, k);
    double nv[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) nv[c] = a.zf_centroid[fz + P.NZF * c];
    const double t = 1.0 / fmax(a.smallnum, sqrt(nv[0] * nv[0] + nv[1] * nv[1] + nv[2] * nv[2]));
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      A[0][c] = a.xf_normal[xp + P.NXF * c];
      A[1][c] = a.xf_normal[xm + P.NXF * c];
      A[2][c] = a.yf_normal[yp + P.NXF * c];
      A[3][c] = a.yf_normal[ym + P.NXF * c];
      A[4][c] = nv[c] * t;
      A[5][c] = A[4][c];
    }
    R[0] = a.Bxf[P.fci(i, j, k)];
    R[1] = a.Bxf[P.fci(i - 1, j, k)];
    R[2] = a.Byf[P.fci(i, j, k)];
    R[3] = a.Byf[P.fci(i, j - 1, k)];
    R[4] = a.Bzf[P.fci(i, j, k)];
    R[5] = a.Bzf[P.fci(i, j, k - 1)];
    double M[3][3], r3[3];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        double s = 0.0;
#pragma unroll
        for (int r = 0; r < 6; ++r) s += A[r][p] * A[r][q];
        M[p][q] = s;
      }
      double s = 0.0;
#pragma unroll
      for (int r = 0; r < 6; ++r) s += A[r][p] * R[r];
      r3[p] = s;
    }
    const double det = M[0][0] * (M[1][1] * M[2][2] - M[2][1] * M[1][2]) -
                       M[0][1] * (M[1][0] * M[2][2] - M[2][0] * M[1][2]) +
                       M[0][2] * (M[1][0] * M[2][1] - M[2][0] * M[1][1]);
    const double od = copysign(1.0, det) / fmax(1.0e-32, fabs(det));
    const double b[3][3] = {{(M[1][1] * M[2][2] - M[1][2] * M[2][1]) * od, (M[0][2] * M[2][1] - M[0][1] * M[2][2]) * od,
                             (M[0][1] * M[1][2] - M[1][1] * M[0][2]) * od},
                            {(M[1][2] * M[2][0] - M[1][0] * M[2][2]) * od, (M[0][0] * M[2][2] - M[0][2] * M[2][0]) * od,
                             (M[0][2] * M[1][0] - M[0][0] * M[1][2]) * od},
                            {(M[1][0] * M[2][1] - M[1][1] * M[2][0]) * od, (M[0][1] * M[2][0] - M[0][0] * M[2][1]) * od,
                             (M[0][0] * M[1][1] - M[0][1] * M[1][0]) * od}};
    const double b2old = U[5] * U[5] + U[6] * U[6] + U[7] * U[7];
#pragma unroll
    for (int p = 0; p < 3; ++p) U[5 + p] = b[p][0] * r3[0] + b[p][1] * r3[1] + b[p][2] * r3[2];
    const double ob8pi = 0.5 * C<double>::ob4pi;
    U[4] = U[4] - b2old * ob8pi + (U[5] * U[5] + U[6] * U[6] + U[7] * U[7]) * ob8pi;
    a.B1_zc[z] = U[5];
    a.B2_zc[z] = U[6];
    a.B3_zc[z] = U[7];
  }
  double e = a.ent[z];
  Gas<double> gs{gam, gam - 1.0, a.rhofloor, a.prsfloor, 1.0 / (gam - 1.0)};
  V[4] = 0.0;
  cons_to_prim(gs, U, V, e);
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    P.Vr(c, 0, z) = V[c];
    put_changed(P.Ur(c, 0, z), U[c], was[c]);
  }
  a.ent[z] = e;
}

constexpr int DT_THREADS = 256, DT_BLOCKS = 1024;

__global__ void k_dt_init(double dt0, double* out) { out[0] = dt0; }

// min of a positive double into *out by compare-and-swap (order-independent)
__device__ __forceinline__ void atomic_min_pos(double* out, double v) {
  unsigned long long* w = (unsigned long long*)out;
  unsigned long long cur = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  while (v < __longlong_as_double((long long)cur)) {
    const unsigned long long seen = atomicCAS(w, cur, (unsigned long long)__double_as_longlong(v));
    if (seen == cur) break;
    cur = seen;
  }
}

__global__ void __launch_bounds__(DT_THREADS) k_dt(const P1 P, const Box own, double cfl, double dt0,
                                                   double* out) {
  __shared__ double red[DT_THREADS];
  const cs_p1_patch& a = P.a;
  const Gas<double> gs{a.gamma, a.gamma - 1.0, a.rhofloor, a.prsfloor, 1.0 / (a.gamma - 1.0)};
  double best = dt0;
  const int64_t n = own.count(), stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t t = tid(); t < n; t += stride) {
    int i, j, k;
    own.decode(t, i, j, k);
    const int64_t z = P.zi(i, j, k);
    if (a.mask[z] == 0) continue;
    double U[8], was[8], V[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) U[c] = was[c] = P.Ur(c, 0, z);
    double e = a.ent[z];  // the routine keeps its entropy array as it is
    V[4] = 0.0;
    cons_to_prim(gs, U, V, e);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      put_changed(P.Ur(c, 0, z), U[c], was[c]);
      P.Vr(c, 0, z) = V[c];
    }
    const double b2 = V[5] * V[5] + V[6] * V[6] + V[7] * V[7];
    const double ms = sqrt((a.gamma_sound[z] * V[4] + C<double>::ob4pi * b2) / V[0]);
    a.msonic[z] = ms;
    const double s = sqrt(V[1] * V[1] + V[2] * V[2] + V[3] * V[3]) + ms;
    best = fmin(best, cfl * a.scale[z] / s);
  }
  red[threadIdx.x] = best;
  __syncthreads();
  for (int h = DT_THREADS / 2; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] = fmin(red[threadIdx.x], red[threadIdx.x + h]);
    __syncthreads();
  }
  if (threadIdx.x == 0) atomic_min_pos(out, red[0]);
}

static int p1_dims_check(const cs_p1_patch* p, const char* who, P1& P) {
  if (!p) {
    cs::set_error("%s: null patch", who);
    return CS_E_INVALID;
  }
  if (p->ntp < 1 || p->nr < 1 || p->nghost < 1) {
    cs::set_error("%s: need ntp, nr, nghost >= 1 (got %d, %d, %d)", who, p->ntp, p->nr, p->nghost);
    return CS_E_INVALID;
  }
  if (p->nghost >= p->ntp) {
    cs::set_error("%s: nghost (%d) must be below ntp (%d)", who, p->nghost, p->ntp);
    return CS_E_BAD_DECOMP;
  }
  if (!(p->gamma > 1.0) || !(p->rhofloor > 0.0) || !(p->prsfloor > 0.0) || !(p->smallnum > 0.0)) {
    cs::set_error("%s: gamma > 1 and positive floors and smallnum required", who);
    return CS_E_INVALID;
  }
  P.a = *p;
  P.N = p->ntp;
  P.NR = p->nr;
  P.g = p->nghost;
  P.nz = P.N + 2 * P.g;
  P.nzr = P.NR + 2 * P.g;
  P.nf = P.nz + 1;
  P.nfr = P.nzr + 1;
  P.NZ = (int64_t)P.nz * P.nz * P.nzr;
  P.NXF = (int64_t)P.nf * P.nz * P.nzr;
  P.NZF = (int64_t)P.nz * P.nz * P.nfr;
  P.NFC = (int64_t)P.nf * P.nf * P.nfr;
  return 0;
}

}  // namespace csp1

extern "C" int cs_cleanup_after_update_p1(const cs_p1_patch* p, void* stream_) {
  P1 P;
  int rc = p1_dims_check(p, "cs_cleanup_after_update_p1", P);
  if (rc) return rc;
  const void* ptrs[] = {p->mask, p->stencil, p->xf_normal, p->yf_normal, p->zf_centroid, p->scale, p->U,
                        p->ent, p->Bxf, p->Byf, p->Bzf, p->V, p->B1_zc, p->B2_zc, p->B3_zc, p->gamma_eos,
                        p->gamma_sound, p->mean_mol_wt};
  for (const void* q : ptrs)
    if (!q) {
      cs::set_error("cs_cleanup_after_update_p1: null array in the patch");
      return CS_E_INVALID;
    }
  hipStream_t st = (hipStream_t)stream_;
  k_face_zero<<<dim3(grid_of(P.NFC, 256), 3), 256, 0, st>>>(P);
  k_tricorner<<<grid_of(4 * (int64_t)P.g * P.nzr, 256), 256, 0, st>>>(P);
  k_cleanup_zone<<<grid_of(P.NZ, 256), 256, 0, st>>>(P);
  P1_HIP(hipGetLastError());
  return 0;
}

extern "C" int cs_evaluate_timestep_p1(const cs_p1_patch* p, double cfl, double dtcur, double* dt_new,
                                       void* stream_) {
  P1 P;
  int rc = p1_dims_check(p, "cs_evaluate_timestep_p1", P);
  if (rc) return rc;
  const void* ptrs[] = {p->mask, p->scale, p->U, p->ent, p->V, p->gamma_sound, p->msonic, dt_new};
  for (const void* q : ptrs)
    if (!q) {
      cs::set_error("cs_evaluate_timestep_p1: null array in the patch or null dt_new");
      return CS_E_INVALID;
    }
  if (!(cfl > 0.0) || !(dtcur > 0.0)) {
    cs::set_error("cs_evaluate_timestep_p1: cfl and dtcur must be positive (got %g, %g)", cfl, dtcur);
    return CS_E_INVALID;
  }
  hipStream_t st = (hipStream_t)stream_;
  const Box own = make_box(1, P.N, 1, P.N, 1, P.NR);
  const int nblk = (int)std::min<int64_t>(grid_of(own.count(), DT_THREADS), DT_BLOCKS);
  k_dt_init<<<1, 1, 0, st>>>(1.1 * dtcur, dt_new);
  k_dt<<<nblk, DT_THREADS, 0, st>>>(P, own, cfl, 1.1 * dtcur, dt_new);
  P1_HIP(hipGetLastError());
  return 0;
}

// ---------------------------------------------------------------------------
// MAKE_EDGE_EFIELDS_P1 (cubesphere/400riemann_integrate/460make_edge_fields_p1.f:5)
// of one patch at second order, FP64.  k_edge: one work item per entry of the
// face-B-shaped edge arrays, the family (x, y, z edges) in blockIdx.y; items
// on an edge of the owned faces compute it, all others write the zero the
// routine leaves there, so the arrays need no separate clearing.  An edge's
// field: the mean mode-1 E of its four zones along the edge's tangent, the
// face-point normal B of the four faces around it (LIMIT_ALL_SLOPES_P1) and
// their wave speeds (MAKE_FACIAL_FLUXES) symmetrised to +-max|S|, and the
// 4-state HLL of 630...f (csp::emf4_hll).  z-edges with an inactive zone keep
// zero; at a flagged tri-corner the edge where the three active zones meet
// adds the 3-state HLL of 631...f (emf3_hll below).
namespace csp1 {

struct P1E {
  cs_p1_edge a;
  int N, NR, g, nz, nf;
  int64_t NZ, NFC;
  __device__ __forceinline__ int64_t zi(int i, int j, int k) const {
    return (int64_t)(i - 1 + g) + (int64_t)nz * ((j - 1 + g) + (int64_t)nz * (k - 1 + g));
  }
  __device__ __forceinline__ int64_t fci(int i, int j, int k) const {
    return (int64_t)(i + g) + (int64_t)nf * ((j + g) + (int64_t)nf * (k + g));
  }
  __device__ __forceinline__ double vx(int i, int j, int k, int c) const { return a.vert[fci(i, j, k) + NFC * c]; }
  __device__ __forceinline__ double emean(int c, const int64_t* z, int n) const {
    const double* E = c == 0 ? a.Ex_zc : c == 1 ? a.Ey_zc : a.Ez_zc;
    return n == 4 ? (E[z[0]] + E[z[1]] + E[z[2]] + E[z[3]]) * 0.25 : (E[z[0]] + E[z[1]] + E[z[2]]) * (1.0 / 3.0);
  }
};

__global__ void __launch_bounds__(256) k_edge(const P1E P) {
  const int fam = blockIdx.y;
  const int64_t t = tid();
  if (t >= P.NFC) return;
  const cs_p1_edge& a = P.a;
  const int n = P.nf, N = P.N, NR = P.NR;
  const int i = (int)(t % n) - P.g, j = (int)((t / n) % n) - P.g, k = (int)(t / ((int64_t)n * n)) - P.g;
  double* out = fam == 0 ? a.Efx : fam == 1 ? a.Efy : a.Efz;
  const bool on = fam == 0   ? (i >= 1 && i <= N && j >= 0 && j <= N && k >= 0 && k <= NR)
                  : fam == 1 ? (i >= 0 && i <= N && j >= 1 && j <= N && k >= 0 && k <= NR)
                             : (i >= 0 && i <= N && j >= 0 && j <= N && k >= 1 && k <= NR);
  double val = 0.0;
  if (on) {
    // zones LD, RD, RU, LU around the edge, and the edge's other vertex
    int zc[4][3];
    int pi = i, pj = j, pk = k;
    if (fam == 0) {
      const int q[4][3] = {{i, j, k}, {i, j + 1, k}, {i, j + 1, k + 1}, {i, j, k + 1}};
      memcpy(zc, q, sizeof(zc));
      pi = i - 1;
    } else if (fam == 1) {
      const int q[4][3] = {{i, j, k}, {i, j, k + 1}, {i + 1, j, k + 1}, {i + 1, j, k}};
      memcpy(zc, q, sizeof(zc));
      pj = j - 1;
    } else {
      const int q[4][3] = {{i, j, k}, {i + 1, j, k}, {i + 1, j + 1, k}, {i, j + 1, k}};
      memcpy(zc, q, sizeof(zc));
      pk = k - 1;
    }
    int64_t z[4], f[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      z[q] = P.zi(zc[q][0], zc[q][1], zc[q][2]);
      f[q] = P.fci(zc[q][0], zc[q][1], zc[q][2]);
    }
    const bool active = fam < 2 || (a.mask[z[0]] && a.mask[z[1]] && a.mask[z[2]] && a.mask[z[3]]);
    double ec[3], tg[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) ec[c] = 0.5 * (P.vx(i, j, k, c) + P.vx(pi, pj, pk, c));
    if (active) {
      double ct = 0.0, st = 1.0;
      if (fam < 2) {
        // tangent: the chord, made normal to the radius at the edge centre
        // (the centre lifted to the vertices' sphere)
        const double rv = sqrt(P.vx(i, j, k, 0) * P.vx(i, j, k, 0) + P.vx(i, j, k, 1) * P.vx(i, j, k, 1) +
                               P.vx(i, j, k, 2) * P.vx(i, j, k, 2));
        const double lift = rv / sqrt(ec[0] * ec[0] + ec[1] * ec[1] + ec[2] * ec[2]);
        double r[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) r[c] = ec[c] * lift;
        const double ir = 1.0 / sqrt(r[0] * r[0] + r[1] * r[1] + r[2] * r[2]);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          r[c] *= ir;
          tg[c] = P.vx(i, j, k, c) - P.vx(pi, pj, pk, c);
        }
        const double d = tg[0] * r[0] + tg[1] * r[1] + tg[2] * r[2];
#pragma unroll
        for (int c = 0; c < 3; ++c) tg[c] -= d * r[c];
        const double it = 1.0 / sqrt(tg[0] * tg[0] + tg[1] * tg[1] + tg[2] * tg[2]);
#pragma unroll
        for (int c = 0; c < 3; ++c) tg[c] *= it;
      } else {
        // tangent: radial; the angle between the x and y lattice directions
        const double ir = 1.0 / sqrt(ec[0] * ec[0] + ec[1] * ec[1] + ec[2] * ec[2]);
        double n1[3], tau[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          tg[c] = ec[c] * ir;
          n1[c] = P.vx(i + 1, j, k, c) - P.vx(i - 1, j, k, c);
          tau[c] = P.vx(i, j + 1, k, c) - P.vx(i, j - 1, k, c);
        }
        const double d1 = n1[0] * tg[0] + n1[1] * tg[1] + n1[2] * tg[2];
        const double d2 = tau[0] * tg[0] + tau[1] * tg[1] + tau[2] * tg[2];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          n1[c] -= d1 * tg[c];
          tau[c] -= d2 * tg[c];
        }
        const double i1 = 1.0 / sqrt(n1[0] * n1[0] + n1[1] * n1[1] + n1[2] * n1[2]);
        const double i2 = 1.0 / sqrt(tau[0] * tau[0] + tau[1] * tau[1] + tau[2] * tau[2]);
        ct = (tau[0] * i2) * (n1[0] * i1) + (tau[1] * i2) * (n1[1] * i1) + (tau[2] * i2) * (n1[2] * i1);
        st = sqrt(1.0 - ct * ct);
      }
      const double Et = P.emean(0, z, 4) * tg[0] + P.emean(1, z, 4) * tg[1] + P.emean(2, z, 4) * tg[2];
      // face-point normal B (points 2..5 of the faces around the edge) and speeds
      const double* byq = fam == 0 ? a.Bzf_q : fam == 1 ? a.Bxf_q : a.Byf_q;
      const double* bnq = fam == 0 ? a.Byf_q : fam == 1 ? a.Bzf_q : a.Bxf_q;
      const double By_R = byq[f[1] + 4 * P.NFC], By_L = byq[f[0] + 3 * P.NFC];
      const double Bn_U = bnq[f[3] + 2 * P.NFC], Bn_D = bnq[f[0] + P.NFC];
      const double *sHi1, *sLo1, *sHi2, *sLo2;
      int a1, b1, a2, b2;  // zones whose speeds make S_R, S_L (a1, b1) and S_U, S_D (a2, b2)
      if (fam == 0) {
        sHi1 = a.S_U; sLo1 = a.S_D; sHi2 = a.S_T; sLo2 = a.S_B; a1 = 3; b1 = 0; a2 = 1; b2 = 0;
      } else if (fam == 1) {
        sHi1 = a.S_T; sLo1 = a.S_B; sHi2 = a.S_R; sLo2 = a.S_L; a1 = 3; b1 = 0; a2 = 0; b2 = 1;
      } else {
        sHi1 = a.S_R; sLo1 = a.S_L; sHi2 = a.S_U; sLo2 = a.S_D; a1 = 3; b1 = 0; a2 = 1; b2 = 0;
      }
      const double sR = fmax(sHi1[f[a1]], sHi1[f[b1]]), sL = fmin(sLo1[f[a1]], sLo1[f[b1]]);
      const double sU = fmax(sHi2[f[a2]], sHi2[f[b2]]), sD = fmin(sLo2[f[a2]], sLo2[f[b2]]);
      const double S = fmax(fmax(fabs(sR), fabs(sL)), fmax(fabs(sU), fabs(sD)));
      val = emf4_hll<double>(S, -S, S, -S, ct, st, Et, Et, Et, Et, Bn_U, Bn_D, By_R, By_L);
    }
    if (fam == 2) {
      const int corner = (i == 0 && j == 0) ? 0 : (i == N && j == 0) ? 1 : (i == N && j == N) ? 2
                                                : (i == 0 && j == N) ? 3 : -1;
      if (corner >= 0 && a.itri[corner]) {
        // the three active zones 1, 2, 3 of the corner (460...f tri-corner blocks)
        int q1[2], q2[2], q3[2];
        if (corner == 0) {
          q1[0] = i + 1; q1[1] = j + 1; q2[0] = i; q2[1] = j + 1; q3[0] = i + 1; q3[1] = j;
        } else if (corner == 1) {
          q1[0] = i + 1; q1[1] = j + 1; q2[0] = i; q2[1] = j + 1; q3[0] = i; q3[1] = j;
        } else if (corner == 2) {
          q1[0] = i; q1[1] = j + 1; q2[0] = i; q2[1] = j; q3[0] = i + 1; q3[1] = j;
        } else {
          q1[0] = i + 1; q1[1] = j + 1; q2[0] = i; q2[1] = j; q3[0] = i + 1; q3[1] = j;
        }
        const int64_t z3[3] = {P.zi(q1[0], q1[1], k), P.zi(q2[0], q2[1], k), P.zi(q3[0], q3[1], k)};
        const double ir = 1.0 / sqrt(ec[0] * ec[0] + ec[1] * ec[1] + ec[2] * ec[2]);
        const double Et = P.emean(0, z3, 3) * (ec[0] * ir) + P.emean(1, z3, 3) * (ec[1] * ir) +
                          P.emean(2, z3, 3) * (ec[2] * ir);
        const int64_t f1 = P.fci(q1[0], q1[1], k), f2 = P.fci(q2[0], q2[1], k), f3 = P.fci(q3[0], q3[1], k),
                      f2d = P.fci(q2[0], q2[1] - 1, k), f1d = P.fci(q1[0], q1[1] - 1, k);
        const int64_t NF = P.NFC;
        double bn[3], sr[3], sl[3];
        if (corner == 0) {
          bn[0] = -a.Byf_q[f3 + 4 * NF]; bn[1] = a.Bxf_q[f2 + 2 * NF]; bn[2] = a.Byf_q[f2d + 3 * NF];
          sr[0] = -a.S_D[f3]; sl[0] = -a.S_U[f3]; sr[1] = a.S_R[f2]; sl[1] = a.S_L[f2];
          sr[2] = a.S_U[f2d]; sl[2] = a.S_D[f2d];
        } else if (corner == 1) {
          bn[0] = -a.Byf_q[f1d + 4 * NF]; bn[1] = a.Bxf_q[f2 + 2 * NF]; bn[2] = a.Byf_q[f3 + 3 * NF];
          sr[0] = -a.S_L[f3]; sl[0] = -a.S_R[f3]; sr[1] = a.S_R[f2]; sl[1] = a.S_L[f2];
          sr[2] = a.S_U[f3]; sl[2] = a.S_D[f3];
        } else if (corner == 2) {
          bn[0] = a.Bxf_q[f1 + 2 * NF]; bn[1] = a.Byf_q[f2 + 3 * NF]; bn[2] = -a.Bxf_q[f2 + NF];
          sr[0] = a.S_R[f1]; sl[0] = a.S_L[f1]; sr[1] = a.S_U[f2]; sl[1] = a.S_D[f2];
          sr[2] = -a.S_L[f2]; sl[2] = -a.S_R[f2];
        } else {
          bn[0] = -a.Byf_q[f3 + 4 * NF]; bn[1] = a.Byf_q[f2 + 3 * NF]; bn[2] = -a.Bxf_q[f2 + NF];
          sr[0] = -a.S_D[f3]; sl[0] = -a.S_U[f3]; sr[1] = a.S_U[f2]; sl[1] = a.S_D[f2];
          sr[2] = -a.S_L[f2]; sl[2] = -a.S_R[f2];
        }
        const double S = fmax(fmax(fmax(fabs(sr[0]), fabs(sl[0])), fmax(fabs(sr[1]), fabs(sl[1]))),
                              fmax(fabs(sr[2]), fabs(sl[2])));
        const double Sr[3] = {S, S, S}, Sl[3] = {-S, -S, -S}, E3[3] = {Et, Et, Et};
        val += emf3_hll(Sr, Sl, E3, bn);
      }
    }
  }
  out[t] = val;
}

}  // namespace csp1

extern "C" int cs_make_edge_efields_p1(const cs_p1_edge* p, void* stream_) {
  if (!p) {
    cs::set_error("cs_make_edge_efields_p1: null argument");
    return CS_E_INVALID;
  }
  if (p->ntp < 1 || p->nr < 1 || p->nghost < 1) {
    cs::set_error("cs_make_edge_efields_p1: need ntp, nr, nghost >= 1 (got %d, %d, %d)", p->ntp, p->nr,
                  p->nghost);
    return CS_E_INVALID;
  }
  if (p->nghost >= p->ntp) {
    cs::set_error("cs_make_edge_efields_p1: nghost (%d) must be below ntp (%d)", p->nghost, p->ntp);
    return CS_E_BAD_DECOMP;
  }
  const void* ptrs[] = {p->vert, p->mask, p->Ex_zc, p->Ey_zc, p->Ez_zc, p->Bxf_q, p->Byf_q, p->Bzf_q, p->S_L,
                        p->S_R, p->S_D, p->S_U, p->S_B, p->S_T, p->Efx, p->Efy, p->Efz};
  for (const void* q : ptrs)
    if (!q) {
      cs::set_error("cs_make_edge_efields_p1: null array");
      return CS_E_INVALID;
    }
  hipStream_t st = (hipStream_t)stream_;
  P1E P;
  P.a = *p;
  P.N = p->ntp;
  P.NR = p->nr;
  P.g = p->nghost;
  P.nz = P.N + 2 * P.g;
  P.nf = P.nz + 1;
  P.NZ = (int64_t)P.nz * P.nz * (P.NR + 2 * P.g);
  P.NFC = (int64_t)P.nf * P.nf * (P.NR + 2 * P.g + 1);
  k_edge<<<dim3(grid_of(P.NFC, 256), 3), 256, 0, st>>>(P);
  P1_HIP(hipGetLastError());
  return 0;
}

// ---------------------------------------------------------------------------
// BUILD_NON_STIFF_SOURCES (cubesphere/400riemann_integrate/470build_non_stiff_sources.f:6)
// of one patch, MHD, adiabatic, no external source.  k_src: one work item per
// zone; every zone's Source is written (zero outside the routine's range), and
// on the active zones of (0..N+1)^2 x (0..nr+1) the point-mass gravity at the
// zone centroid, the centrifugal and the Coriolis terms of omega_passive and
// the energy source v . S go into Source and are added to dU_dt (:150-250).
namespace csp1 {

__global__ void __launch_bounds__(256) k_src(const cs_p1_source a, int N, int NR, int g, int64_t NZ) {
  const int64_t z = tid();
  if (z >= NZ) return;
  const int nz = N + 2 * g;
  const int i = (int)(z % nz) + 1 - g, j = (int)((z / nz) % nz) + 1 - g, k = (int)(z / ((int64_t)nz * nz)) + 1 - g;
  const bool on = i >= 0 && i <= N + 1 && j >= 0 && j <= N + 1 && k >= 0 && k <= NR + 1 && a.mask[z] == 1;
  double S[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  const double ox = a.omega[0], oy = a.omega[1], oz = a.omega[2];
  if (on && (a.mstar > a.smallnum || sqrt(ox * ox + oy * oy + oz * oz) > a.smallnum)) {
    const double x = a.v_centroid[z], y = a.v_centroid[z + NZ], w = a.v_centroid[z + 2 * NZ];
    const double rho = a.V[z], vx = a.V[z + NZ], vy = a.V[z + 2 * NZ], vz = a.V[z + 3 * NZ];
    const double rad = sqrt(x * x + y * y + w * w);
    const double gmr3 = a.newtonsc * a.mstar / (rad * rad * rad);
    const double cx = oy * w - oz * y, cy = oz * x - ox * w, cz = ox * y - oy * x;  // omega x r
    S[1] = -gmr3 * x * rho - rho * (oy * cz - oz * cy) - 2.0 * rho * (oy * vz - oz * vy);
    S[2] = -gmr3 * y * rho - rho * (oz * cx - ox * cz) - 2.0 * rho * (oz * vx - ox * vz);
    S[3] = -gmr3 * w * rho - rho * (ox * cy - oy * cx) - 2.0 * rho * (ox * vy - oy * vx);
    S[4] = vx * S[1] + vy * S[2] + vz * S[3];
  }
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    a.Source[z + NZ * c] = S[c];
    if (on) a.dU_dt[z + NZ * c] += S[c];
  }
}

}  // namespace csp1

extern "C" int cs_build_non_stiff_sources_p1(const cs_p1_source* p, void* stream_) {
  if (!p) {
    cs::set_error("cs_build_non_stiff_sources_p1: null argument");
    return CS_E_INVALID;
  }
  if (p->ntp < 1 || p->nr < 1 || p->nghost < 1) {
    cs::set_error("cs_build_non_stiff_sources_p1: need ntp, nr, nghost >= 1 (got %d, %d, %d)", p->ntp, p->nr,
                  p->nghost);
    return CS_E_INVALID;
  }
  if (!p->mask || !p->v_centroid || !p->V || !p->Source || !p->dU_dt) {
    cs::set_error("cs_build_non_stiff_sources_p1: null array");
    return CS_E_INVALID;
  }
  const int64_t nz = p->ntp + 2 * p->nghost;
  const int64_t NZ = nz * nz * (p->nr + 2 * p->nghost);
  k_src<<<grid_of(NZ, 256), 256, 0, (hipStream_t)stream_>>>(*p, p->ntp, p->nr, p->nghost, NZ);
  P1_HIP(hipGetLastError());
  return 0;
}

// ---------------------------------------------------------------------------
// The defect correction of the driver over the P1 patches of one shell
// (FILL_FLUX_SND_PATCH 599..., FETCH_BUFFERS_FILL_IN_FLUX_X/Y/Z 334-336...,
// SYNCHRONIZE_EFZ_QUAD_CORNER 340..., UNPACK_DEFECT_FLUXES 341...,
// UPDATE_DEFECT_IMEX_RK 485update_defect_imex_rk.f): the fluctuations and
// entropy fluxes of every face that two patches share take the mean of the
// two patches' values (334...f:100-116), the electric field of every shared
// edge the mean of its two or three patches' values (334...f:128-160, the
// tri-corner edges a third of three), and each patch's boundary zones get the
// difference of their fluctuations, -(mean - own) A / V, in dU_dt.  Done
// before the update instead of re-applied after it; the update is linear in
// these, so the result is the same.  The face and edge pairings, with their
// orientations, come from the host (matched geometrically once).
namespace csp1 {

struct P1Sync {
  double* Fl_Pl[6][3];  // [patch][family]
  double* Fl_Mi[6][3];
  double* EntF[6][3];
  double* Ef[6][3];
  double* dU_dt[6];
  const double* area[6][3];
  const double* vol[6];
  int N, g, nz, nf;
  int64_t NZ, NFC, NXF, NZF;
};

using FacePair = cs_p1_face_pair;
using EdgeGroup = cs_p1_edge_group;

__global__ void __launch_bounds__(256) k_sync_faces(const P1Sync S, const FacePair* fp, int64_t n) {
  const int64_t t = tid();
  if (t >= n) return;
  const FacePair q = fp[t];
  const int64_t NFC = S.NFC;
  double ePl[2][8], eMi[2][8];
  double ent[2];
  const int pp[2] = {q.pa, q.pb}, ff[2] = {q.fa, q.fb};
  const int64_t ii[2] = {q.ia, q.ib};
#pragma unroll
  for (int s = 0; s < 2; ++s) {
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      ePl[s][c] = S.Fl_Pl[pp[s]][ff[s]][ii[s] + NFC * c];
      eMi[s][c] = S.Fl_Mi[pp[s]][ff[s]][ii[s] + NFC * c];
    }
    ent[s] = S.EntF[pp[s]][ff[s]][ii[s]];
  }
  // the mean in a's orientation: with opposite normals b's plus side is a's
  // minus side and its entropy flux has the other sign
  double mPl[8], mMi[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    mPl[c] = 0.5 * (ePl[0][c] + (q.flip ? eMi[1][c] : ePl[1][c]));
    mMi[c] = 0.5 * (eMi[0][c] + (q.flip ? ePl[1][c] : eMi[1][c]));
  }
  const double mEnt = 0.5 * (ent[0] + (q.flip ? -ent[1] : ent[1]));
  const int64_t zz[2] = {q.za, q.zb}, ar[2] = {q.aa, q.ab};
  const int sd[2] = {q.sa, q.sb};
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const bool swap = s == 1 && q.flip;
    const double* nPl = swap ? mMi : mPl;
    const double* nMi = swap ? mPl : mMi;
    const double w = S.area[pp[s]][ff[s]][ar[s]] / S.vol[pp[s]][zz[s]];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const double own = sd[s] ? ePl[s][c] : eMi[s][c], mean = sd[s] ? nPl[c] : nMi[c];
      atomicAdd(&S.dU_dt[pp[s]][zz[s] + S.NZ * c], -(mean - own) * w);
      S.Fl_Pl[pp[s]][ff[s]][ii[s] + NFC * c] = nPl[c];
      S.Fl_Mi[pp[s]][ff[s]][ii[s] + NFC * c] = nMi[c];
    }
    S.EntF[pp[s]][ff[s]][ii[s]] = (s == 1 && q.flip) ? -mEnt : mEnt;
  }
}

__global__ void __launch_bounds__(256) k_sync_edges(const P1Sync S, const EdgeGroup* eg, int64_t n) {
  const int64_t t = tid();
  if (t >= n) return;
  const EdgeGroup q = eg[t];
  double sum = 0.0;
  for (int m = 0; m < q.n; ++m) sum += q.sign[m] * S.Ef[q.p[m]][q.f[m]][q.idx[m]];
  const double mean = q.n == 3 ? sum * (1.0 / 3.0) : 0.5 * sum;
  for (int m = 0; m < q.n; ++m) S.Ef[q.p[m]][q.f[m]][q.idx[m]] = q.sign[m] * mean;
}

}  // namespace csp1

extern "C" int cs_sync_shared_p1(const cs_p1_shell_sync* p, void* stream_) {
  if (!p || !p->faces || !p->edges) {
    cs::set_error("cs_sync_shared_p1: null argument");
    return CS_E_INVALID;
  }
  if (p->ntp < 1 || p->nr < 1 || p->nghost < 1 || p->nface < 0 || p->nedge < 0) {
    cs::set_error("cs_sync_shared_p1: bad sizes");
    return CS_E_INVALID;
  }
  P1Sync S;
  for (int s = 0; s < 6; ++s) {
    const cs_p1_patch_fluxes& q = p->patch[s];
    const void* ptrs[] = {q.Fluct_x_Pl, q.Fluct_y_Pl, q.Fluct_z_Pl, q.Fluct_x_Mi, q.Fluct_y_Mi, q.Fluct_z_Mi,
                          q.EntFlux_x, q.EntFlux_y, q.EntFlux_z, q.Efx, q.Efy, q.Efz, q.dU_dt,
                          q.xf_area, q.yf_area, q.zf_area, q.v_volume};
    for (const void* r : ptrs)
      if (!r) {
        cs::set_error("cs_sync_shared_p1: null array of patch %d", s);
        return CS_E_INVALID;
      }
    S.Fl_Pl[s][0] = q.Fluct_x_Pl; S.Fl_Pl[s][1] = q.Fluct_y_Pl; S.Fl_Pl[s][2] = q.Fluct_z_Pl;
    S.Fl_Mi[s][0] = q.Fluct_x_Mi; S.Fl_Mi[s][1] = q.Fluct_y_Mi; S.Fl_Mi[s][2] = q.Fluct_z_Mi;
    S.EntF[s][0] = q.EntFlux_x; S.EntF[s][1] = q.EntFlux_y; S.EntF[s][2] = q.EntFlux_z;
    S.Ef[s][0] = q.Efx; S.Ef[s][1] = q.Efy; S.Ef[s][2] = q.Efz;
    S.dU_dt[s] = q.dU_dt;
    S.area[s][0] = q.xf_area; S.area[s][1] = q.yf_area; S.area[s][2] = q.zf_area;
    S.vol[s] = q.v_volume;
  }
  S.N = p->ntp;
  S.g = p->nghost;
  S.nz = p->ntp + 2 * p->nghost;
  S.nf = S.nz + 1;
  S.NZ = (int64_t)S.nz * S.nz * (p->nr + 2 * p->nghost);
  S.NFC = (int64_t)S.nf * S.nf * (p->nr + 2 * p->nghost + 1);
  hipStream_t st = (hipStream_t)stream_;
  if (p->nface > 0)
    k_sync_faces<<<grid_of(p->nface, 256), 256, 0, st>>>(S, (const FacePair*)p->faces, p->nface);
  if (p->nedge > 0)
    k_sync_edges<<<grid_of(p->nedge, 256), 256, 0, st>>>(S, (const EdgeGroup*)p->edges, p->nedge);
  P1_HIP(hipGetLastError());
  return 0;
}

// ---------------------------------------------------------------------------
// PAD_BOUNDARY_R (800applications_cs/826pad_boundary_r.f:1) of one patch,
// outflow pads.  One work item per (column, ghost layer izz); every write
// reads only layer 1 / face 0 (inner) or layer nr / face nr (outer), and the
// faces two columns share get the same value from both, so the items are
// independent.
namespace csp1 {

__global__ void __launch_bounds__(256) k_pad_r(const cs_p1_pad P, int N, int NR, int g, int64_t NZ) {
  const int64_t nz = N + 2 * g, nf = nz + 1;
  const int64_t t = tid();
  if (t >= nz * nz * g) return;
  const int ix = (int)(t % nz) + 1 - g, iy = (int)((t / nz) % nz) + 1 - g, izz = (int)(t / (nz * nz)) + 1;
  auto zi = [&](int i, int j, int k) { return (int64_t)(i - 1 + g) + nz * ((j - 1 + g) + nz * (k - 1 + g)); };
  auto fc = [&](int i, int j, int k) { return (int64_t)(i + g) + nf * ((j + g) + nf * (k + g)); };
  auto xa = [&](int i, int j, int k) { return (int64_t)(i + g) + nf * ((j - 1 + g) + nz * (k - 1 + g)); };
  auto ya = [&](int i, int j, int k) { return (int64_t)(i - 1 + g) + nz * ((j + g) + nf * (k - 1 + g)); };
  auto za = [&](int i, int j, int k) { return (int64_t)(i - 1 + g) + nz * ((j - 1 + g) + nz * (k + g)); };
  if (P.mask[zi(ix, iy, izz)] != 1) return;
  const int64_t col = (int64_t)(ix - 1 + g) + nz * (iy - 1 + g);
  if (P.bcarr_r[col] == 2) {
    const int l = 1 - izz, r = 1;
#pragma unroll
    for (int c = 0; c < 8; ++c) P.U[zi(ix, iy, l) + NZ * c] = P.U[zi(ix, iy, r) + NZ * c];
    P.Bxf[fc(ix, iy, l)] = P.Bxf[fc(ix, iy, r)];
    P.Bxf[fc(ix - 1, iy, l)] = P.Bxf[fc(ix - 1, iy, r)];
    P.Byf[fc(ix, iy, l)] = P.Byf[fc(ix, iy, r)];
    P.Byf[fc(ix, iy - 1, l)] = P.Byf[fc(ix, iy - 1, r)];
    P.Bzf[fc(ix, iy, l - 1)] = P.Bzf[fc(ix, iy, r - 1)];
  }
  if (P.bcarr_r[col + nz * nz] == 2) {
    const int l = NR + izz, r = NR;
    const double vr = P.v_volume[zi(ix, iy, r)], vl = P.v_volume[zi(ix, iy, l)];
#pragma unroll
    for (int c = 0; c < 8; ++c) P.U[zi(ix, iy, l) + NZ * c] = P.U[zi(ix, iy, r) + NZ * c] * vr / vl;
    P.Bzf[fc(ix, iy, l)] = P.Bzf[fc(ix, iy, r)] * P.zf_area[za(ix, iy, r)] / P.zf_area[za(ix, iy, l)];
    P.Bxf[fc(ix, iy, l)] = P.Bxf[fc(ix, iy, r)] * P.xf_area[xa(ix, iy, r)] / P.xf_area[xa(ix, iy, l)];
    P.Byf[fc(ix, iy, l)] = P.Byf[fc(ix, iy, r)] * P.yf_area[ya(ix, iy, r)] / P.yf_area[ya(ix, iy, l)];
    P.Bxf[fc(ix - 1, iy, l)] =
        P.Bxf[fc(ix - 1, iy, r)] * P.xf_area[xa(ix - 1, iy, r)] / P.xf_area[xa(ix - 1, iy, l)];
    P.Byf[fc(ix, iy - 1, l)] =
        P.Byf[fc(ix, iy - 1, r)] * P.yf_area[ya(ix, iy - 1, r)] / P.yf_area[ya(ix, iy - 1, l)];
  }
}

}  // namespace csp1

extern "C" int cs_pad_boundary_r_p1(const cs_p1_pad* p, void* stream_) {
  if (!p) {
    cs::set_error("cs_pad_boundary_r_p1: null argument");
    return CS_E_INVALID;
  }
  if (p->ntp < 1 || p->nr < 1 || p->nghost < 1) {
    cs::set_error("cs_pad_boundary_r_p1: need ntp, nr, nghost >= 1 (got %d, %d, %d)", p->ntp, p->nr, p->nghost);
    return CS_E_INVALID;
  }
  if (!p->mask || !p->bcarr_r || !p->xf_area || !p->yf_area || !p->zf_area || !p->v_volume || !p->U || !p->Bxf ||
      !p->Byf || !p->Bzf) {
    cs::set_error("cs_pad_boundary_r_p1: null array");
    return CS_E_INVALID;
  }
  const int64_t nz = p->ntp + 2 * p->nghost;
  const int64_t NZ = nz * nz * (p->nr + 2 * p->nghost);
  csp1::k_pad_r<<<grid_of(nz * nz * p->nghost, 256), 256, 0, (hipStream_t)stream_>>>(*p, p->ntp, p->nr,
                                                                                       p->nghost, NZ);
  P1_HIP(hipGetLastError());
  return 0;
}

// ---------------------------------------------------------------------------
// Third order: LIMIT_ALL_SLOPES_P12 (421limit_all_slopes_p12.f:9) on one patch
// whose U and V hold ten modes.  Steps 2-7.a are the P1 kernels above (they
// address modes 1-4, which a ten-mode array lays out exactly as a four-mode
// one); k_zero_hi clears modes 5-10, k_weno_ao is step 7.b, k_pos<10> 7.c,
// k_face_pts<10> 8.a-c, k_clsq12 8.d, k_e12 9.a, k_weno9 on E 9.b,
// k_ao_order / k_ao_e_pre / k_ao_e_sweep / k_ao_e_put 9.c, and the P1
// diagnostics step 10.
namespace csp1 {

__global__ void __launch_bounds__(256) k_zero_hi(const P1 P, const Box b) {
  int i, j, k;
  if (!b.decode(tid(), i, j, k)) return;
  const int64_t z = P.zi(i, j, k);
#pragma unroll
  for (int m = 4; m < 10; ++m)
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      P.Ur(c, m, z) = 0.0;
      P.Vr(c, m, z) = 0.0;
    }
}

// the 18 zones of the central quadratic stencil (421...f:3888-4350, in that
// order): stencil direction (R L U D, then RU LU LD RD as 4-7) and k offset
__constant__ int c_ao_dir[18] = {0, 1, 2, 3, -1, -1, 4, 5, 6, 7, 0, 1, 0, 1, 2, 3, 2, 3};
__constant__ int c_ao_dk[18] = {0, 0, 0, 0, 1, -1, 0, 0, 0, 0, 1, 1, -1, -1, 1, 1, -1, -1};

// packed lower triangle of a symmetric 9 x 9 matrix
__device__ __forceinline__ constexpr int lt(int r, int c) { return r * (r + 1) / 2 + c; }

// Step 7.b (421...f:3811-4557), one thread per zone: the 18 x 9 rows of
// RECONSTRUCTION_COEFS (251reconstruction_coefs.f:3) — the average over the
// stencil zone of this zone's quadratic basis, from the centroid offset, the
// two scale lengths and the ten basis moments — give the normal equations
// (A^T A) X = A^T R; A^T A is factored once (Cholesky, in registers) and
// solved for the eight primitives, four at a time with the rows formed
// again for the second four.  The fit is hybridised with the P1 gradients
// (MR-WENO linear weights 0.95 / 0.05 for smooth flow, 0.6 / 0.4 where the
// flattener is 1; smoothness indicators of the two polynomials; weights
// (1 + tau / IS)), and every mode above the mean is multiplied by
// (1 - flattener).  The reference inverts A^T A by LU (MATINV); the two
// agree to rounding.  Two waves per SIMD, the registers held to 256 with a
// small spill.
__device__ __forceinline__ void weno_ao_zone(const P1& P, int i, int j, int k, const double* __restrict__ mom) {
  if (!P.active(i, j, 1)) return;
  const cs_p1_patch& a = P.a;
  const int64_t z = P.zi(i, j, k), NZ = P.NZ;
  const double sm = a.smallnum, ell0 = fmax(a.scale[z], sm), obl0 = 1.0 / ell0;
  double c0[6], cz[3];
#pragma unroll
  for (int m = 0; m < 6; ++m) c0[m] = mom[z + NZ * (4 + m)];
#pragma unroll
  for (int c = 0; c < 3; ++c) cz[c] = a.v_centroid[z + NZ * c];
  int ni[8], nj[8];
  {
    const int dirs[8] = {0, 1, 2, 3, 8, 9, 10, 11};
#pragma unroll
    for (int q = 0; q < 8; ++q) P.nbr(i, j, dirs[q], ni[q], nj[q]);
  }
  const double f = a.flatten[z];
  const double betalo = f + (1.0 - f) * 2.0;
  const double gammahi = f * 0.6 + (1.0 - f) * 0.95, gammalo = 1.0 - gammahi;
  const double obgammahi = 1.0 / gammahi, gammaratio = gammalo / gammahi;
  const double ob12 = 1.0 / 12.0, ob180 = 1.0 / 180.0, ob144 = 1.0 / 144.0;
  const double m5 = c0[0] - ob12, m6 = c0[1] - ob12, m7 = c0[2] - ob12;
  const double q4 = m5 * m5 + ob180, q5 = m6 * m6 + ob180, q6 = m7 * m7 + ob180;
  const double q7 = c0[3] * c0[3] + ob144, q8 = c0[4] * c0[4] + ob144, q9 = c0[5] * c0[5] + ob144;
  double L[45];
#pragma unroll
  for (int e = 0; e < 45; ++e) L[e] = 0.0;
#pragma unroll 1
  for (int grp = 0; grp < 2; ++grp) {
    double Y[4][9];
    double v0[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      v0[c] = P.V(4 * grp + c, 0, z);
#pragma unroll
      for (int m = 0; m < 9; ++m) Y[c][m] = 0.0;
    }
#pragma unroll 1
    for (int r = 0; r < 18; ++r) {
      const int dir = c_ao_dir[r];
      int ii = i, jj = j;
      if (dir >= 0) {
        // selects, not an indexed read of ni / nj (which would go to scratch)
#pragma unroll
        for (int q = 0; q < 8; ++q)
          if (q == dir) {
            ii = ni[q];
            jj = nj[q];
          }
      }
      const int64_t zr = P.zi(ii, jj, k + c_ao_dk[r]);
      double x[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) x[c] = (a.v_centroid[zr + NZ * c] - cz[c]) * obl0;
      const double rho = fmax(a.scale[zr], sm) / ell0, r2 = rho * rho;
      double row[9];
      row[0] = x[0];
      row[1] = x[1];
      row[2] = x[2];
      row[3] = x[0] * x[0] - c0[0] + mom[zr + NZ * 4] * r2;
      row[4] = x[1] * x[1] - c0[1] + mom[zr + NZ * 5] * r2;
      row[5] = x[2] * x[2] - c0[2] + mom[zr + NZ * 6] * r2;
      row[6] = x[0] * x[1] - c0[3] + mom[zr + NZ * 7] * r2;
      row[7] = x[1] * x[2] - c0[4] + mom[zr + NZ * 8] * r2;
      row[8] = x[0] * x[2] - c0[5] + mom[zr + NZ * 9] * r2;
      if (grp == 0) {
#pragma unroll
        for (int p = 0; p < 9; ++p)
#pragma unroll
          for (int q = 0; q <= p; ++q) L[lt(p, q)] += row[p] * row[q];
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const double R = P.V(4 * grp + c, 0, zr) - v0[c];
#pragma unroll
        for (int m = 0; m < 9; ++m) Y[c][m] += row[m] * R;
      }
    }
    if (grp == 0) {  // Cholesky factor of A^T A in place
#pragma unroll
      for (int p = 0; p < 9; ++p) {
        double d = L[lt(p, p)];
#pragma unroll
        for (int q = 0; q < p; ++q) d -= L[lt(p, q)] * L[lt(p, q)];
        d = sqrt(fmax(d, 1.0e-300));
        L[lt(p, p)] = d;
        const double od = 1.0 / d;
#pragma unroll
        for (int r = p + 1; r < 9; ++r) {
          double t = L[lt(r, p)];
#pragma unroll
          for (int q = 0; q < p; ++q) t -= L[lt(r, q)] * L[lt(p, q)];
          L[lt(r, p)] = t * od;
        }
      }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      double X[9];
#pragma unroll
      for (int p = 0; p < 9; ++p) {  // L y = Y
        double t = Y[c][p];
#pragma unroll
        for (int q = 0; q < p; ++q) t -= L[lt(p, q)] * X[q];
        X[p] = t / L[lt(p, p)];
      }
#pragma unroll
      for (int p = 8; p >= 0; --p) {  // L^T x = y
        double t = X[p];
#pragma unroll
        for (int q = p + 1; q < 9; ++q) t -= L[lt(q, p)] * X[q];
        X[p] = t / L[lt(p, p)];
      }
      const int comp = 4 * grp + c;
      const double g1 = P.V(comp, 1, z), g2 = P.V(comp, 2, z), g3 = P.V(comp, 3, z);
      const double ISlo = betalo * (g1 * g1 + g2 * g2 + g3 * g3) * ob12;
      double Phi[9];
      Phi[0] = X[0] * obgammahi - g1 * gammaratio;
      Phi[1] = X[1] * obgammahi - g2 * gammaratio;
      Phi[2] = X[2] * obgammahi - g3 * gammaratio;
#pragma unroll
      for (int m = 3; m < 9; ++m) Phi[m] = X[m] * obgammahi;
      const double IShi = (Phi[0] * Phi[0] + Phi[1] * Phi[1] + Phi[2] * Phi[2]) * ob12 + Phi[3] * Phi[3] * q4 +
                          Phi[4] * Phi[4] * q5 + Phi[5] * Phi[5] * q6 + Phi[6] * Phi[6] * q7 +
                          Phi[7] * Phi[7] * q8 + Phi[8] * Phi[8] * q9;
      const double tau = fabs(IShi - ISlo);
      double wlo = gammalo * (1.0 + tau / (ISlo + sm)), whi = gammahi * (1.0 + tau / (IShi + sm));
      const double aa = 1.0 / (wlo + whi);
      wlo *= aa;
      whi *= aa;
      const double x1 = 1.0 - f;
      P.Vr(comp, 1, z) = (whi * Phi[0] + wlo * g1) * x1;
      P.Vr(comp, 2, z) = (whi * Phi[1] + wlo * g2) * x1;
      P.Vr(comp, 3, z) = (whi * Phi[2] + wlo * g3) * x1;
#pragma unroll
      for (int m = 3; m < 9; ++m) P.Vr(comp, m + 1, z) = whi * Phi[m] * x1;
    }
  }
}

__global__ void __attribute__((amdgpu_waves_per_eu(2))) __launch_bounds__(128)
    k_weno_ao(const P1 P, const Box b, const double* __restrict__ mom) {
  int i, j, k;
  if (b.decode(tid(), i, j, k)) weno_ao_zone(P, i, j, k, mom);
}
// the positivity replay's zones inside the range
__global__ void __attribute__((amdgpu_waves_per_eu(2))) __launch_bounds__(128)
    k_weno_ao_list(const P1 P, const Box b, const double* __restrict__ mom, const Flags F, int sweep) {
  if (F.done(sweep)) return;
  const int64_t n = F.ctr[1];
  for (int64_t t = tid(); t < n; t += (int64_t)gridDim.x * blockDim.x) {
    int i, j, k;
    zone_of(P, F.list[t], i, j, k);
    if (i < b.i0 || i >= b.i0 + b.ni || j < b.j0 || j >= b.j0 + b.nj || k < b.k0 || k >= b.k0 + b.nk) continue;
    weno_ao_zone(P, i, j, k, mom);
  }
}

// LDS words written before by a wave's lanes, read after by its others
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Step 8.d at third order (421...f:5574-6680), four zones per wave, 16 lanes
// each: the 36 x 36 system of the normal equations of the 64 least-squares
// rows (n . B at the 30 face points against their face-point B, the 30 WENO-AO
// modes, the divergence and its gradient) and the 6 face-mean constraints.
// The face points' words (normal, the ten basis values about the zone's
// moments, B-field weight, face-point B) go through LDS; lane r holds the rows
// r, r + 16 and r + 32 of the lower triangle (K = P^T P + I + D^T D above the
// constraint rows C) in registers, 84 doubles.  L D L^T in natural order: the
// leading 30 x 30 block has every eigenvalue at least 1, so its pivots are too,
// and the trailing block then holds -C K^-1 C^T, negative definite for the six
// independent rows C, so no pivot search is needed.  A column entry reaches
// the zone's lanes by a row broadcast (DPP), a row of L the back substitution
// through LDS, where its words have taken the face points' place.  The
// reference solves the same system by Numerical Recipes' LU with partial
// pivoting (MATSOLVE): the two agree to rounding.
//
// One zone per wave with the whole rows in 36 lanes and v_readlane broadcasts
// (the Gram by FP64 MFMA) spent two broadcast instructions on each multiply-add
// and eliminated both triangles: 64^2 x 25 1.34 -> 0.60 ms, 192^2 x 64 22.5 ->
// 10.5 ms with k_e12, 49,644 operations a zone at 13.0 TFLOP/s.  What bounds
// it now is FP64 issue at two waves per SIMD (per lane 1,380 multiply-adds of
// the Gram and 1,250 of the elimination, and 1,400 broadcast moves); the point loop unrolled five-fold spills
// (0.69 ms at 64^2 x 25).  Against the system in 80-bit arithmetic its largest
// relative error is 4.0e-15, the earlier form's 4.2e-15.
constexpr int kSqStride = 484;    // LDS words per zone: 30 points of 16, and 4 against bank conflicts

// lane N of each row of 16 lanes, in all of them
template <int N>
__device__ __forceinline__ double row_lane(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x150 + N, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x150 + N, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
// f(integral_constant) for I = A .. B - 1
template <int A, int B, class F>
__device__ __forceinline__ void static_for(const F& f) {
  if constexpr (A < B) {
    f(std::integral_constant<int, A>{});
    static_for<A + 1, B>(f);
  }
}

__global__ void __attribute__((amdgpu_waves_per_eu(2))) __launch_bounds__(64)
    k_clsq12(const P1 P, const Box b, const double* __restrict__ mom) {
  __shared__ double2 sh[kSqZones * kSqStride / 2];
  const int r = threadIdx.x % 16, g = threadIdx.x / 16;
  int i, j, k;
  if (!b.decode((int64_t)blockIdx.x * kSqZones + g, i, j, k)) return;  // all 16 lanes of a zone
  const cs_p1_patch& a = P.a;
  const int64_t z = P.zi(i, j, k), NZ = P.NZ;
  if (a.mask[z] == 0) return;
  double* const pt = (double*)sh + g * kSqStride;  // [30][16]: n (3), basis (10), weight, face-point B
  {
    const double obl = P.obl(z);
    double c0[6];
#pragma unroll
    for (int m = 0; m < 6; ++m) c0[m] = mom[z + NZ * (4 + m)];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int pq = r + 16 * h;
      if (pq < 30) {
        const int f = pq / 5, q = pq % 5, fam = f >> 1;
        const bool hi = (f & 1) == 0;
        const int fi = i - (fam == 0 && !hi), fj = j - (fam == 1 && !hi), fk = k - (fam == 2 && !hi);
        const int64_t fg = fam == 0 ? P.xfi(fi, fj, fk) : (fam == 1 ? P.yfi(fi, fj, fk) : P.zfi(fi, fj, fk));
        const int64_t NF = fam == 2 ? P.NZF : P.NXF, fb = P.fci(fi, fj, fk);
        const double* nrm = fam == 0 ? a.xb_normal : (fam == 1 ? a.yb_normal : a.zb_normal);
        const double* pts = fam == 0 ? a.xb_pts : (fam == 1 ? a.yb_pts : a.zb_pts);
        const double* wts = fam == 0 ? a.xb_wts : (fam == 1 ? a.yb_wts : a.zb_wts);
        const double* Bq = fam == 0 ? a.Bxf_q : (fam == 1 ? a.Byf_q : a.Bzf_q);
        double x[3];
        double* w = pt + 16 * pq;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          w[c] = fam == 2 ? nrm[fg + NF * (c + 3 * q)] : nrm[fg + NF * c];
          x[c] = (pts[fg + NF * (c + 3 * q)] - P.cen(z, c)) * obl;
        }
        w[3] = 1.0;
        w[4] = x[0];
        w[5] = x[1];
        w[6] = x[2];
        w[7] = x[0] * x[0] - c0[0];
        w[8] = x[1] * x[1] - c0[1];
        w[9] = x[2] * x[2] - c0[2];
        w[10] = x[0] * x[1] - c0[3];
        w[11] = x[1] * x[2] - c0[4];
        w[12] = x[0] * x[2] - c0[5];
        w[13] = wts[fg + NF * q];
        w[14] = Bq[fb + P.NFC * q];
      }
    }
  }
  wave_sync();
  // rows r and r + 16 (r < 14) of K: their component and mode
  const int ca = r / 10, ma = r % 10, cb = r < 14 ? (r + 16) / 10 : 0, mb = r < 14 ? (r + 16) % 10 : 0;
  double K0[16], K1[32], K2[36], y0, y1, y2 = 0.0;
#pragma unroll
  for (int e = 0; e < 16; ++e) K0[e] = e == r ? 1.0 : 0.0;
#pragma unroll
  for (int e = 0; e < 32; ++e) K1[e] = e == r + 16 && r < 14 ? 1.0 : 0.0;
  y0 = P.V(5 + ca, ma, z);
  y1 = r < 14 ? P.V(5 + cb, mb, z) : 0.0;
  // the Gram of the point rows, their right-hand side; a finished face's
  // points make room for its constraint row
#pragma unroll 1
  for (int f = 0; f < 6; ++f) {
    double Ca = 0.0, Cb = 0.0, d = 0.0;
#pragma unroll 1
    for (int q = 0; q < 5; ++q) {
      const double* w = pt + 16 * (5 * f + q);
      const double pa = w[ca] * w[3 + ma], pb = r < 14 ? w[cb] * w[3 + mb] : 0.0;
      double v[16];
#pragma unroll
      for (int h = 0; h < 8; ++h) {
        const double2 t = ((const double2*)w)[h];
        v[2 * h] = t.x;
        v[2 * h + 1] = t.y;
      }
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double na = pa * v[c], nb = pb * v[c];
#pragma unroll
        for (int m = 0; m < 10; ++m) {
          if (10 * c + m < 16) K0[10 * c + m] += na * v[3 + m];
          K1[10 * c + m] += nb * v[3 + m];
        }
      }
      y0 += pa * v[14];
      y1 += pb * v[14];
      Ca += v[13] * pa;
      Cb += v[13] * pb;
      d += v[13] * v[14];
    }
    wave_sync();
    pt[80 * f + r] = Ca;
    pt[80 * f + 16 + r] = Cb;
    wave_sync();
    if (r == 14 + f) y1 = d;  // f = 0, 1
    if (r == f - 2) y2 = d;   // f = 2 .. 5
  }
  // the constraint rows: 30 and 31 in the second set, 32 to 35 in the third
#pragma unroll
  for (int e = 0; e < 30; ++e) {
    const double t1 = pt[80 * (r >= 14 ? r - 14 : 0) + e], t2 = pt[80 * (r < 4 ? r + 2 : 2) + e];
    K1[e] = r >= 14 ? t1 : K1[e];
    K2[e] = r < 4 ? t2 : 0.0;
  }
#pragma unroll
  for (int e = 30; e < 36; ++e) K2[e] = 0.0;
  // D^T D of the four divergence rows (421...f:6000-6200): row d has 1 at three
  // modes, 2 at the own quadratic one
  {
    auto dv = [](int row, int e1, int e2, int e3, int two) {
      return (row == e1 || row == e2 || row == e3) ? (row == two ? 2.0 : 1.0) : 0.0;
    };
    auto add = [&](int row, auto& K, auto limit) {
      constexpr int n = decltype(limit)::value;
      const double d0 = dv(row, 1, 12, 23, -1), d1 = dv(row, 4, 17, 29, 4), d2 = dv(row, 7, 15, 28, 15),
                   d3 = dv(row, 9, 18, 26, 26);
      K[1] += d0;
      K[4] += 2.0 * d1;
      K[7] += d2;
      K[9] += d3;
      K[12] += d0;
      K[15] += 2.0 * d2;
      if constexpr (n > 16) {
        K[17] += d1;
        K[18] += d3;
        K[23] += d0;
        K[26] += 2.0 * d3;
        K[28] += d2;
        K[29] += d1;
      }
    };
    add(r, K0, std::integral_constant<int, 16>{});
    add(r < 14 ? r + 16 : -1, K1, std::integral_constant<int, 32>{});
  }
  // elimination: step jj takes row jj out of the rows below it.  The entries
  // of column jj are the multipliers times the pivot; a lane whose row is jj
  // or above takes none
  static_for<0, 36>([&](auto J) {
    constexpr int jj = J, ps = jj / 16, pl = jj % 16;
    double col[3] = {ps == 0 ? K0[ps == 0 ? jj : 0] : 0.0, ps <= 1 ? K1[ps <= 1 ? jj : 0] : 0.0, K2[jj]};
    const double piv = row_lane<pl>(col[ps]), od = 1.0 / piv;
    double mul[3];
#pragma unroll
    for (int s = 0; s < 3; ++s) mul[s] = s < ps ? 0.0 : col[s] * od;
    if (r <= pl) mul[ps] = 0.0;
    const double yj = row_lane<pl>(ps == 0 ? y0 : (ps == 1 ? y1 : y2));
    if constexpr (ps == 0) y0 = r == pl ? y0 * od : y0 - mul[0] * yj;
    if constexpr (ps == 1) y1 = r == pl ? y1 * od : y1 - mul[1] * yj;
    if constexpr (ps == 2) y2 = r == pl ? y2 * od : y2 - mul[2] * yj;
    if constexpr (ps < 1) y1 -= mul[1] * yj;
    if constexpr (ps < 2) y2 -= mul[2] * yj;
    static_for<jj + 1, 36>([&](auto E) {
      constexpr int e = E;
      const double v = row_lane<e % 16>(col[e / 16]);
      if constexpr (e < 16) K0[e] -= mul[0] * v;
      if constexpr (e < 32 && ps <= 1) K1[e] -= mul[1] * v;
      K2[e] -= mul[2] * v;
    });
    if constexpr (ps == 0) K0[jj] = mul[0];
    if constexpr (ps <= 1) K1[jj] = mul[1];
    K2[jj] = mul[2];
  });
  // back substitution with the rows of L from LDS: the third set, then the
  // second's own block, its part in the first's unknowns, the first
  double* const lt = pt;
  wave_sync();
  if (r < 4) {
#pragma unroll
    for (int e = 0; e < 36; ++e) lt[37 * r + e] = K2[e];
  }
  wave_sync();
  static_for<0, 4>([&](auto J) {
    constexpr int q = 3 - J;
    const double x = row_lane<q>(y2);
    y0 -= lt[37 * q + r] * x;
    y1 -= lt[37 * q + 16 + r] * x;
    const double t = lt[37 * q + 32 + (r < 4 ? r : 0)];
    if (r < q) y2 -= t * x;
  });
  wave_sync();
#pragma unroll
  for (int e = 0; e < 16; ++e) lt[17 * r + e] = K1[16 + e];
  wave_sync();
  static_for<0, 16>([&](auto J) {
    constexpr int q = 15 - J;
    const double x = row_lane<q>(y1), t = lt[17 * q + r];
    if (r < q) y1 -= t * x;
  });
  wave_sync();
#pragma unroll
  for (int e = 0; e < 16; ++e) lt[17 * r + e] = K1[e];
  wave_sync();
  static_for<0, 16>([&](auto J) {
    constexpr int q = J;
    y0 -= lt[17 * q + r] * row_lane<q>(y1);
  });
  wave_sync();
#pragma unroll
  for (int e = 0; e < 16; ++e) lt[17 * r + e] = K0[e];
  wave_sync();
  static_for<0, 16>([&](auto J) {
    constexpr int q = 15 - J;
    const double x = row_lane<q>(y0), t = lt[17 * q + r];
    if (r < q) y0 -= t * x;
  });
  auto out = [&](int c, int m, double v) {
    double* Bz = c == 0 ? a.B1_zc : (c == 1 ? a.B2_zc : a.B3_zc);
    Bz[z + NZ * m] = v;
    P.Vr(5 + c, m, z) = v;
  };
  out(ca, ma, y0);
  if (r < 14) out(cb, mb, y1);
  const double b0 = row_lane<0>(y0), b1 = row_lane<10>(y0), b2 = row_lane<4>(y1);
  if (r == 0) {
    const double ob8pi = 1.0 / (8.0 * M_PI);
    const double aa = (P.Ur(5, 0, z) * P.Ur(5, 0, z) + P.Ur(6, 0, z) * P.Ur(6, 0, z) + P.Ur(7, 0, z) * P.Ur(7, 0, z)) * ob8pi;
    P.Ur(5, 0, z) = b0;
    P.Ur(6, 0, z) = b1;
    P.Ur(7, 0, z) = b2;
    const double bb = (b0 * b0 + b1 * b1 + b2 * b2) * ob8pi;
    P.Ur(4, 0, z) = P.Ur(4, 0, z) - aa + bb;
  }
}

// Step 9.a at third order (421...f:6684-6795): E = -v x B at the zone's
// centroid, v and B the quadratic fields there (the mean minus the quadratic
// modes times the moments), every zone.
__global__ void __launch_bounds__(256) k_e12(const P1 P, const Box b, const double* __restrict__ mom) {
  int i, j, k;
  if (!b.decode(tid(), i, j, k)) return;
  const int64_t z = P.zi(i, j, k), NZ = P.NZ;
  double q[6];
#pragma unroll
  for (int m = 0; m < 6; ++m) q[m] = mom[z + NZ * (4 + m)];
  auto at = [&](int c) {
    double v = P.V(c, 0, z);
#pragma unroll
    for (int m = 0; m < 6; ++m) v = v - P.V(c, 4 + m, z) * q[m];
    return v;
  };
  const double Bx = at(5), By = at(6), Bz = at(7), vx = at(1), vy = at(2), vz = at(3);
  const cs_p1_patch& a = P.a;
  a.Ex_zc[z] = -(vy * Bz - vz * By);
  a.Ey_zc[z] = -(vz * Bx - vx * Bz);
  a.Ez_zc[z] = -(vx * By - vy * Bx);
}

// The reference's step 9.c overwrites each zone's point value of E
// (421...f:9030) while later zones of the same loop read it as a stencil
// value (:8899-8935): its serial build gives a zone the new point values of
// the active box zones before it in (k, j, i) order and the old ones of those
// after it.  Level (i+1) + 3 (j+1) + 9 (k+1) reproduces that order when every
// stencil entry lies within two zones in i and j: a neighbour in the plane
// differs by at most 2 in i, so a row step of 3 outweighs it, and a neighbour
// above or below by at most 2 + 3 * 2 = 8 within the plane, which a plane step
// of 9 outweighs.  One thread per (i, j) of the box sets *bad when a pair of
// zones of the box breaks the order: the entry point's contract, and more than
// the sweep needs, which is that an earlier neighbour of the same plane
// (dj <= 0) has di + 3 dj < 0 and so di + s dj < 0 for every s >= 3.
__global__ void __launch_bounds__(256) k_ao_order(const P1 P, const Box b, unsigned int* bad) {
  const int64_t t = tid();
  if (t >= (int64_t)b.ni * b.nj) return;
  const int i = b.i0 + (int)(t % b.ni), j = b.j0 + (int)(t / b.ni);
  if (!P.active(i, j, 1)) return;
  int ni[8], nj[8];
  {
    const int dirs[8] = {0, 1, 2, 3, 8, 9, 10, 11};
#pragma unroll
    for (int q = 0; q < 8; ++q) P.nbr(i, j, dirs[q], ni[q], nj[q]);
  }
  bool ok = true;
#pragma unroll
  for (int r = 0; r < 18; ++r) {
    const int dir = c_ao_dir[r], dk = c_ao_dk[r];
    int ii = i, jj = j;
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (q == dir) {
        ii = ni[q];
        jj = nj[q];
      }
    if (ii < b.i0 || ii >= b.i0 + b.ni || jj < b.j0 || jj >= b.j0 + b.nj || !P.active(ii, jj, 1)) continue;
    const int di = ii - i, dj = jj - j;
    const bool earlier = dk < 0 || (dk == 0 && (dj < 0 || (dj == 0 && di < 0)));
    const int dl = di + 3 * dj + 9 * dk;
    if (dk == 0 && dj == 0 && di == 0) continue;
    if (earlier ? dl >= 0 : dl <= 0) ok = false;
  }
  if (!ok) atomicOr(bad, 1u);
}

// Step 9.c's fit (421...f:8406-8936) depends on the stencil's point values
// of E only through its right-hand side: the ten modes are X = G R, R the 19
// point values, G = (A^T A)^-1 A^T, A the 19 x 10 matrix of
// INTERPOLATION_COEFS (252interpolation_coefs.f:5: this zone's basis at each
// stencil zone's centroid, row 0 the zone itself).  k_ao_e_pre, one thread
// per zone of the box, forms G with a Cholesky factor of A^T A, adds up the
// part of X that the loop order leaves at old point values (the zone itself,
// the zones after it and the inactive ones), and keeps, as one record of
// kAoRec doubles, what the ordered sweep needs: G's rows for the zones of the
// plane below and for the earlier zones of the same plane, that partial sum,
// and the zone's own terms of the hybridisation.  Doubles of a record:
constexpr int kAoG = 0;      // [10 modes][10]: G for the five zones below, then for the first four earlier zones of
                             // the plane
constexpr int kAoOut = 0;    // [10][4] in their place, after the sweep: the zone's new modes of E
constexpr int kAoPo = 100;   // [10][4]: the old values' part of X for the three components, the smoothness
                             // indicator's weight of the mode
constexpr int kAoEe = 140;   // [4][4]: the point value and the WENO gradient of the three components of E
constexpr int kAoMi = 156;   // [4]: the three low indicators, the flattener
constexpr int kAoIx = 160;   // 16 int32: [0..4] box index of each zone below (-1: none), [5] how many earlier zones of
                             // the plane (-1: an inactive zone), [8..15] these (ring slot, or -2 - box index)
constexpr int kAoGf = 168;   // [4][10]: G for further earlier zones (tri-corner strips)
// the newest values of each row of a plane in LDS: rows modulo kRingRows, the
// last kRing zones of a row (64 KB; a workgroup of eight waves at two per SIMD
// fills its CU whatever it holds).  With s levels a row the neighbours at
// (-1, -1) lie s + 1 levels back and the farthest entry of a panel's own table,
// at a tri-corner strip, 2 s + 2: kRing covers every entry of patches up to 388
// zones across (s = 14) and the ordinary ones up to 836 (s = 30).  Those
// further back come from memory, a round trip in the level's chain: with 16
// zones a row that began at 389 across for a fourth of the entries, and 392^2 x 1
// took 23.0 ms for step 9 (17.8 now), 512^2 x 1 47.0 (29.2).  A slot is written again no
// sooner than s kRingRows - 28 s levels after its row's last zone, more than kRing.
constexpr int kRing = 32, kRingRows = 64;
// no result of arithmetic: a signalling NaN marks a point value not yet formed
constexpr unsigned long long kAoEmpty = 0x7ff0dead0badf00dull;

__global__ void __launch_bounds__(128) k_ao_e_pre(const P1 P, const Box b, const double* __restrict__ mom,
                                                  double* __restrict__ rec, double* __restrict__ xnew) {
  const int64_t t = tid();
  int i, j, k;
  if (!b.decode(t, i, j, k)) return;
  const cs_p1_patch& a = P.a;
  const int64_t z = P.zi(i, j, k), NZ = P.NZ;
#pragma unroll
  for (int c = 0; c < 3; ++c) ((unsigned long long*)xnew)[4 * t + c] = kAoEmpty;
  if (!P.active(i, j, 1)) {  // the sweep skips it
    ((int*)(rec + t * kAoRec + kAoIx))[5] = -1;
    return;
  }
  const double sm = a.smallnum;
  const double obl0 = 1.0 / fmax(a.scale[z], sm);
  double c0[6], cz[3];
#pragma unroll
  for (int m = 0; m < 6; ++m) c0[m] = mom[z + NZ * (4 + m)];
#pragma unroll
  for (int c = 0; c < 3; ++c) cz[c] = a.v_centroid[z + NZ * c];
  int ni[8], nj[8];
  {
    const int dirs[8] = {0, 1, 2, 3, 8, 9, 10, 11};
#pragma unroll
    for (int q = 0; q < 8; ++q) P.nbr(i, j, dirs[q], ni[q], nj[q]);
  }
  double* G = rec + t * kAoRec;
  int* ix = (int*)(G + kAoIx);
  // row r of A: r = 0 the zone itself, r = 1..18 the stencil zones
  auto where = [&](int r, int& ii, int& jj) {
    const int dir = c_ao_dir[r - 1];
    ii = i;
    jj = j;
    if (dir >= 0) {
#pragma unroll
      for (int q = 0; q < 8; ++q)
        if (q == dir) {
          ii = ni[q];
          jj = nj[q];
        }
    }
  };
  auto arow = [&](int r, int64_t zr, double* row) {
    if (r == 0) {
      row[0] = 1.0;
      row[1] = row[2] = row[3] = 0.0;
#pragma unroll
      for (int m = 0; m < 6; ++m) row[4 + m] = -c0[m];
      return;
    }
    double x[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) x[c] = (a.v_centroid[zr + NZ * c] - cz[c]) * obl0;
    row[0] = 1.0;
    row[1] = x[0];
    row[2] = x[1];
    row[3] = x[2];
    row[4] = x[0] * x[0] - c0[0];
    row[5] = x[1] * x[1] - c0[1];
    row[6] = x[2] * x[2] - c0[2];
    row[7] = x[0] * x[1] - c0[3];
    row[8] = x[1] * x[2] - c0[4];
    row[9] = x[0] * x[2] - c0[5];
  };
  double L[55];
#pragma unroll
  for (int e = 0; e < 55; ++e) L[e] = 0.0;
#pragma unroll 1
  for (int r = 0; r < 19; ++r) {
    double row[10];
    int ii = i, jj = j, dk = 0;
    if (r > 0) {
      where(r, ii, jj);
      dk = c_ao_dk[r - 1];
    }
    arow(r, P.zi(ii, jj, k + dk), row);
#pragma unroll
    for (int p = 0; p < 10; ++p)
#pragma unroll
      for (int q = 0; q <= p; ++q) L[p * (p + 1) / 2 + q] += row[p] * row[q];
  }
  double od[10];
#pragma unroll
  for (int p = 0; p < 10; ++p) {  // Cholesky factor in place, reciprocal diagonal in od
    double d = L[p * (p + 1) / 2 + p];
#pragma unroll
    for (int q = 0; q < p; ++q) d -= L[p * (p + 1) / 2 + q] * L[p * (p + 1) / 2 + q];
    d = sqrt(fmax(d, 1.0e-300));
    L[p * (p + 1) / 2 + p] = d;
    od[p] = 1.0 / d;
#pragma unroll
    for (int r = p + 1; r < 10; ++r) {
      double t2 = L[r * (r + 1) / 2 + p];
#pragma unroll
      for (int q = 0; q < p; ++q) t2 -= L[r * (r + 1) / 2 + q] * L[p * (p + 1) / 2 + q];
      L[r * (r + 1) / 2 + p] = t2 * od[p];
    }
  }
  double po[3][10];
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int m = 0; m < 10; ++m) po[c][m] = 0.0;
  const int s = ao_stride(b.ni);
  int nb = 0, nn = 0;
#pragma unroll 1
  for (int r = 0; r < 19; ++r) {  // column r of G: (A^T A)^-1 times row r
    int ii = i, jj = j, dk = 0;
    if (r > 0) {
      where(r, ii, jj);
      dk = c_ao_dk[r - 1];
    }
    const int64_t zr = P.zi(ii, jj, k + dk);
    double X[10];
    arow(r, zr, X);
#pragma unroll
    for (int p = 0; p < 10; ++p) {
      double t2 = X[p];
#pragma unroll
      for (int q = 0; q < p; ++q) t2 -= L[p * (p + 1) / 2 + q] * X[q];
      X[p] = t2 * od[p];
    }
#pragma unroll
    for (int p = 9; p >= 0; --p) {
      double t2 = X[p];
#pragma unroll
      for (int q = p + 1; q < 10; ++q) t2 -= L[q * (q + 1) / 2 + p] * X[q];
      X[p] = t2 * od[p];
    }
    // the zone's new value is read if the serial loop has passed it: an
    // active zone of the box in the plane below, or earlier in this one
    const int di = ii - i, dj = jj - j, back = -(di + s * dj);
    const bool in = ii >= b.i0 && ii < b.i0 + b.ni && jj >= b.j0 && jj < b.j0 + b.nj && k + dk >= b.k0 &&
                    k + dk < b.k0 + b.nk && P.active(ii, jj, 1);
    const int bi = (ii - b.i0) + b.ni * ((jj - b.j0) + b.nj * (k + dk - b.k0));
    int col = -1;
    double* far = nullptr;
    if (in && dk < 0) {
      ix[nb] = bi;
      col = nb++;
    } else if (in && dk == 0 && (dj < 0 || (dj == 0 && di < 0)) && back > 0) {
      ix[8 + nn] = back < kRing ? ((jj - b.j0) % kRingRows) * kRing + (ii - b.i0) % kRing : -2 - bi;
      if (nn < 4) col = 5 + nn;
      else far = G + kAoGf + 10 * (nn - 4);
      ++nn;
    }
    if (col >= 0) {
#pragma unroll
      for (int m = 0; m < 10; ++m) G[kAoG + 10 * m + col] = X[m];
    } else if (far) {
#pragma unroll
      for (int m = 0; m < 10; ++m) far[m] = X[m];
    } else {
      const double E[3] = {a.Ex_zc[zr], a.Ey_zc[zr], a.Ez_zc[zr]};
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int m = 0; m < 10; ++m) po[c][m] += X[m] * E[c];
    }
  }
  for (int q = nb; q < 5; ++q) {
    ix[q] = -1;
#pragma unroll
    for (int m = 0; m < 10; ++m) G[kAoG + 10 * m + q] = 0.0;
  }
  ix[5] = nn;
  // the zone's own terms (421...f:8937-9030)
  const double ob12 = 1.0 / 12.0, ob180 = 1.0 / 180.0, ob144 = 1.0 / 144.0, f = a.flatten[z];
  const double m5 = c0[0] - ob12, m6 = c0[1] - ob12, m7 = c0[2] - ob12;
  const double wt[10] = {0.0, ob12, ob12, ob12, m5 * m5 + ob180, m6 * m6 + ob180, m7 * m7 + ob180,
                         c0[3] * c0[3] + ob144, c0[4] * c0[4] + ob144, c0[5] * c0[5] + ob144};
#pragma unroll
  for (int m = 0; m < 10; ++m) {
#pragma unroll
    for (int c = 0; c < 3; ++c) G[kAoPo + 4 * m + c] = po[c][m];
    G[kAoPo + 4 * m + 3] = wt[m];
  }
  const double betalo = f + (1.0 - f) * 2.0;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const double* E = c == 0 ? a.Ex_zc : (c == 1 ? a.Ey_zc : a.Ez_zc);
    double e[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      e[m] = E[z + NZ * m];
      G[kAoEe + 4 * m + c] = e[m];
    }
    G[kAoMi + c] = betalo * (e[1] * e[1] + e[2] * e[2] + e[3] * e[3]) * ob12;
  }
  G[kAoMi + 3] = f;
}

// the sum over a row of 16 lanes, in every lane: neighbours, pairs, then the
// mirror images within eight and sixteen lanes
template <int CTRL>
__device__ __forceinline__ double dpp_add(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
  return v + __hiloint2double(hi, lo);
}
__device__ __forceinline__ double row_sum(double v) {
  v = dpp_add<0xb1>(v);       // quad_perm 1 0 3 2
  v = dpp_add<0x4e>(v);       // quad_perm 2 3 0 1
  v = dpp_add<0x141>(v);      // row_half_mirror
  return dpp_add<0x140>(v);   // row_mirror
}
// The workgroup's waves meet with their LDS words written and read.  Only the
// ring passes between the waves of a plane, so nothing waits for the stores to
// memory (a full barrier would, and a store's acknowledgement takes longer
// than a level's arithmetic).
__device__ __forceinline__ void ring_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
__device__ __forceinline__ double ao_load(const double* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool ao_empty(double v) { return (unsigned long long)__double_as_longlong(v) == kAoEmpty; }

// Step 9.c at third order (421...f:8406-9353) in the serial loop order: the
// ten modes of the quadratic interpolant X = G R, their hybridisation with
// the WENO gradients of 9.b as in 7.b, then the point value
// E_pt f + E (1 - f) and the modes times (1 - f).
//
// One workgroup per plane k of the box walks the in-plane levels
// l = ir + s jr; a group of 16 lanes takes the zone of its row (rows
// jr = group, group + Z, ...; Z s >= ni, so a group has one row at a time),
// lane m < 10 the mode m of the three components, so that no lane loads what
// another has (a quad of lanes per component loaded G three times and was
// bound by the address unit).  A zone's record and the values of the plane
// below are read two levels ahead, its indices three; the values of the same
// plane, written in the last levels, come from a ring of the newest values of
// each row in LDS (an entry kRing or more levels back from memory), so
// the chain of a level is: ring, four rows of G, the sum of the indicator
// over the group, the weights, ring.
//
// The planes run side by side.  A point value leaves its plane through xnew
// (device-scope relaxed stores and loads of 8 bytes; old values stay in E
// until k_ao_e_put), and the value itself says that it is there (kAoEmpty
// until then), so nothing needs fences, and a plane follows the one below a
// few levels behind.  Planes are handed out by a ticket in the order that
// workgroups start: a workgroup waits only for the plane of the previous
// ticket, which a running or finished workgroup has, and within its own plane
// only for levels it has passed, so every wait ends, whatever the table.
//
// What bounds it: the chain of (ni - 1) + s (nj - 1) levels and a lag of some
// ten levels a plane, 2 to 3 us a level (the latency of the zone's own loads
// and of the values below, the arithmetic of one wave).  Step 9 with the
// pre-pass, against one launch per level of all planes (9 to 13 us each):
// 64^2 x 25 5.0 -> 1.5 ms (521 launches), 192^2 x 64 20.6 -> 11.9 ms (1,384).
__global__ void __launch_bounds__(kAoLanes * kAoGroups + 64)
    k_ao_e_sweep(const P1 P, const Box b, double* rec, double* xnew, unsigned int* ticket, int s) {
  __shared__ double2 ringv[kRingRows * kRing][2];   // the three components of a point value
  __shared__ double2 upv[kAoGroups][8];             // a group's values of the plane below, [zone][component]
  __shared__ int2 pub[2][kAoGroups];                // a level's zones: ring slot, box index (-1: none)
  __shared__ int plane;
  if (threadIdx.x == 0) plane = (int)atomicAdd(ticket, 1u);
  __syncthreads();
  const int kr = plane;
  if (kr >= b.nk) return;
  const double sm = P.a.smallnum;
  const int Z = (blockDim.x - 64) / kAoLanes, g = threadIdx.x / kAoLanes, ln = threadIdx.x % kAoLanes;
  const int m = ln < 10 ? ln : 9;  // lanes 10 to 15 repeat mode 9 with weight 0
  const int ur = ln < 15 ? ln / 3 : 4, uc = ln < 15 ? ln % 3 : 2;  // the value below that this lane reads
  const int levels = b.ni + s * (b.nj - 1);
  struct Index {
    int4 near;
    int nn, below, ir, jr;
    bool on;
  };
  struct Zone {
    Index x;
    double2 G[5], p01, p2w, e01, e2, i01, i2f;
    double acc[3], up;
  };
  auto box_index = [&](int ir, int jr) { return ir + (int64_t)b.ni * (jr + (int64_t)b.nj * kr); };
  if (g >= Z) {
    // the last wave sends each level's point values on after the level: a
    // store's acknowledgement counts before the loads that a wave put out
    // after it, so the waves that form the values send none
    for (int l = 0; l < (levels + 2) / 3 * 3; ++l) {
      ring_barrier();
      for (int e = threadIdx.x % 64; e < 3 * Z; e += 64) {
        const int2 w = pub[l & 1][e / 3];
        if (w.y >= 0)
          __hip_atomic_store(xnew + 4 * (int64_t)w.y + e % 3, ((const double*)ringv[w.x])[e % 3], __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    return;
  }
  // group g's zone of level l: its row, if it has one there, and the indices
  // of its record
  auto place = [&](int l, Index& I) {
    const int jmax = l / s;
    I.on = false;
    if (l >= levels || jmax < g) return;
    I.jr = jmax - (jmax - g) % Z;
    I.ir = l - s * I.jr;
    if (I.jr >= b.nj || I.ir >= b.ni) return;
    I.on = true;
    const int* ix = (const int*)(rec + box_index(I.ir, I.jr) * kAoRec + kAoIx);
    I.below = ix[ur];
    I.nn = ix[5];
    I.near = *(const int4*)(ix + 8);
  };
  // the loads of the zone's record and of its values below go out
  auto issue = [&](const Index& I, Zone& Q) {
    Q.x = I;
    Q.x.on = I.on && I.nn >= 0;
    if (!Q.x.on) return;
    Q.up = 0.0;
    if (I.below >= 0) Q.up = ao_load(xnew + 4 * (int64_t)I.below + uc);
    const double* R = rec + box_index(I.ir, I.jr) * kAoRec;
    const double2* g2 = (const double2*)(R + kAoG + 10 * m);
#pragma unroll
    for (int r = 0; r < 5; ++r) Q.G[r] = g2[r];
    const double2* p2 = (const double2*)(R + kAoPo + 4 * m);
    Q.p01 = p2[0];
    Q.p2w = p2[1];
    const double2* e2 = (const double2*)(R + kAoEe + 4 * (m < 4 ? m : 0));
    Q.e01 = e2[0];
    Q.e2 = e2[1];
    const double2* i2 = (const double2*)(R + kAoMi);
    Q.i01 = i2[0];
    Q.i2f = i2[1];
  };
  auto add = [&](Zone& Q, double gv, double2 v01, double v2) {
    Q.acc[0] += gv * v01.x;
    Q.acc[1] += gv * v01.y;
    Q.acc[2] += gv * v2;
  };
  // the plane below's values arrive and enter the sum
  auto settle = [&](Zone& Q) {
    if (!Q.x.on) return;
    while (ao_empty(Q.up)) {
      __builtin_amdgcn_s_sleep(1);
      Q.up = ao_load(xnew + 4 * (int64_t)Q.x.below + uc);
    }
    ((double*)upv[g])[ln] = Q.up;
    wave_sync();
    Q.acc[0] = Q.p01.x;
    Q.acc[1] = Q.p01.y;
    Q.acc[2] = Q.p2w.x;
    double2 u[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) u[r] = upv[g][r];
    add(Q, Q.G[0].x, u[0], u[1].x);
    add(Q, Q.G[0].y, make_double2(u[1].y, u[2].x), u[2].y);
    add(Q, Q.G[1].x, u[3], u[4].x);
    add(Q, Q.G[1].y, make_double2(u[4].y, u[5].x), u[5].y);
    add(Q, Q.G[2].x, u[6], u[7].x);
    wave_sync();
  };
  auto newest = [&](Zone& Q, int code, double gv) {
    if (code >= 0) {
      add(Q, gv, ringv[code][0], ringv[code][1].x);
    } else {
      double v[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double* p = xnew + 4 * (int64_t)(-2 - code) + c;
        v[c] = ao_load(p);
        while (ao_empty(v[c])) v[c] = ao_load(p);
      }
      add(Q, gv, make_double2(v[0], v[1]), v[2]);
    }
  };
  auto form = [&](Zone& Q, int l) {
    if (!Q.x.on) {
      if (ln == 0) pub[l & 1][g].y = -1;
      return;
    }
    if (Q.x.nn > 0) newest(Q, Q.x.near.x, Q.G[2].y);
    if (Q.x.nn > 1) newest(Q, Q.x.near.y, Q.G[3].x);
    if (Q.x.nn > 2) newest(Q, Q.x.near.z, Q.G[3].y);
    if (Q.x.nn > 3) newest(Q, Q.x.near.w, Q.G[4].x);
    const int64_t t = box_index(Q.x.ir, Q.x.jr);
    for (int r = 4; r < Q.x.nn; ++r) {  // tri-corner strips only
      const double* R = rec + t * kAoRec;
      newest(Q, ((const int*)(R + kAoIx))[8 + r], R[kAoGf + 10 * (r - 4) + m]);
    }
    const double f = Q.i2f.y, x1 = 1.0 - f, gh = f * 0.6 + x1 * 0.95, gl = 1.0 - gh;
    const double obg = 1.0 / gh, gr = gl / gh;
    const double e[3] = {ln < 4 ? Q.e01.x : 0.0, ln < 4 ? Q.e01.y : 0.0, ln < 4 ? Q.e2.x : 0.0};
    const double lo[3] = {Q.i01.x, Q.i01.y, Q.i2f.x};
    const double w = ln < 10 ? Q.p2w.y : 0.0;
    double o[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double p = Q.acc[c] * obg - e[c] * gr, hi = row_sum(p * p * w), tau = fabs(hi - lo[c]);
      const double wlo = gl * (1.0 + tau / (lo[c] + sm)), whi = gh * (1.0 + tau / (hi + sm));
      const double aa = 1.0 / (wlo + whi);
      o[c] = (whi * aa * p + wlo * aa * e[c]) * x1;
    }
    if (ln == 0) {  // the point value
#pragma unroll
      for (int c = 0; c < 3; ++c) o[c] = e[c] * f + o[c];
      const int slot = (Q.x.jr % kRingRows) * kRing + Q.x.ir % kRing;
      ringv[slot][0] = make_double2(o[0], o[1]);
      ringv[slot][1].x = o[2];
      pub[l & 1][g] = make_int2(slot, (int)t);
    }
    if (ln < 10) {  // the modes take the place of the rows that have been read
      double2* v = (double2*)(rec + t * kAoRec + kAoOut + 4 * ln);
      v[0] = make_double2(o[0], o[1]);
      v[1].x = o[2];
    }
  };
  // three zones in turn: at level l, l + 2's loads go out, l's values are
  // formed and l + 1's loads, put out a level ago, are waited for
  Zone A, B, C;
  Index ia, ib, ic;
  place(0, ia);
  place(1, ib);
  place(2, ic);
  issue(ia, A);
  issue(ib, B);
  settle(A);
#pragma unroll 1
  for (int l = 0; l < levels; l += 3) {
    place(l + 3, ia);
    issue(ic, C);
    form(A, l);
    settle(B);
    ring_barrier();
    place(l + 4, ib);
    issue(ia, A);
    form(B, l + 1);
    settle(C);
    ring_barrier();
    place(l + 5, ic);
    issue(ib, B);
    form(C, l + 2);
    settle(A);
    ring_barrier();
  }
}

// the active zones' modes from their records into E, once no zone reads the
// old point values: the sweep's own stores then stay within a zone's record
// (30 words together) instead of 30 places far apart
__global__ void __launch_bounds__(256) k_ao_e_put(const P1 P, const Box b, const double* __restrict__ rec) {
  const int64_t t = tid();
  int i, j, k;
  if (!b.decode(t, i, j, k) || !P.active(i, j, 1)) return;
  const int64_t z = P.zi(i, j, k);
  const double2* R = (const double2*)(rec + t * kAoRec + kAoOut);
#pragma unroll
  for (int m = 0; m < 10; ++m) {
    const double2 v = R[2 * m];
    P.a.Ex_zc[z + P.NZ * m] = v.x;
    P.a.Ey_zc[z + P.NZ * m] = v.y;
    P.a.Ez_zc[z + P.NZ * m] = R[2 * m + 1].x;
  }
}

}  // namespace csp1

extern "C" int cs_limit_all_slopes_p12(const cs_p12_patch* q, void* stream_) {
  if (!q || !q->moments) {
    cs::set_error("cs_limit_all_slopes_p12: null patch or moments");
    return CS_E_INVALID;
  }
  return run_p1(&q->p1, stream_, nullptr, nullptr, 0, q->moments);
}

extern "C" int cs_limit_all_slopes_p12_timed(const cs_p12_patch* q, void* stream_, float* kernel_ms) {
  if (!q || !q->moments || !kernel_ms) {
    cs::set_error("cs_limit_all_slopes_p12_timed: null patch, moments or kernel_ms");
    return CS_E_INVALID;
  }
  return run_p1(&q->p1, stream_, kernel_ms, nullptr, 0, q->moments);
}
