// cs_p1_common.h -- small dense kernels shared by the P1 reconstruction of one
// patch (cs_slopes_p1.hip) and the P1 stage over the six sectors of a shell
// (cs_p1_stage.hip): the adjugate 3 x 3 inverse of the WENO stencils
// (410limit_all_slopes_p1.f:2421-3761), the constrained least squares of the
// zone B (410...f:4643-5360), and the 3-state HLL edge field of the tri-corners (631...f:1-216).
#pragma once
#include <hip/hip_runtime.h>

namespace csp1 {

// A word written back only where its bits have changed: the conserved words
// that a conversion leaves as they were (density, momentum and B of a zone
// above the floors) are not sent to memory again.  The conversion kernels are
// bound by memory: the stage's k_prim on 160^2 x 48 631 -> 477 us (7 of 28
// words a zone saved), the patch update with cleanup and time step on
// 128^2 x 48 336 -> 317 us.
__device__ __forceinline__ void put_changed(double& w, double v, double was) {
  if (__double_as_longlong(v) != __double_as_longlong(was)) w = v;
}

// WENO (410...f:2421-3761, 5437-7100): each stencil's 3 x 3 offset matrix
// inverted by its adjugate, with the reference's sign(det) / max(1e-32, |det|)
__device__ __forceinline__ void inv3(const double (&m)[3][3], double (&r)[3][3]) {
  const double a11 = m[0][0], a12 = m[0][1], a13 = m[0][2], a21 = m[1][0], a22 = m[1][1], a23 = m[1][2],
               a31 = m[2][0], a32 = m[2][1], a33 = m[2][2];
  const double det =
      -(a13 * a22 * a31) + a12 * a23 * a31 + a13 * a21 * a32 - a11 * a23 * a32 - a12 * a21 * a33 + a11 * a22 * a33;
  const double od = (signbit(det) ? -1.0 : 1.0) / fmax(1.0e-32, fabs(det));
  r[0][0] = (-(a23 * a32) + a22 * a33) * od;
  r[0][1] = (a13 * a32 - a12 * a33) * od;
  r[0][2] = (-(a13 * a22) + a12 * a23) * od;
  r[1][0] = (a23 * a31 - a21 * a33) * od;
  r[1][1] = (-(a13 * a31) + a11 * a33) * od;
  r[1][2] = (a13 * a21 - a11 * a23) * od;
  r[2][0] = (-(a22 * a31) + a21 * a32) * od;
  r[2][1] = (a12 * a31 - a11 * a32) * od;
  r[2][2] = (-(a12 * a21) + a11 * a22) * od;
}

// packed lower triangle
#define LIX(r, c) ((r) * ((r) + 1) / 2 + (c))

// Step 8.d: the ADP constrained least squares for the 12 linear B
// coefficients of a zone (410...f:4643-5360): the six face means are matched
// exactly (constraint rows n (x) (1, r) at the face centroids, the normal of
// the face's first point), the face-point B at points 2 and 4 of each face
// and the 12 WENO modes in least squares; then the energy takes the change
// of magnetic energy (:5336-5357).  The reference solves the 18 x 18 KKT
// system by LU; here six unknowns are eliminated.  In a frame of the zone
// (the mean of its x-face normals, the mean of its y-face normals made
// orthogonal to it, their cross product: a rotation R), the six
// face-mean constraints fix each B component's mean and its derivative along
// its own axis, the pivots (b0x, Gxx, b0y, Gyy, b0z, Gzz) = e - W x_f of the
// six other coefficients x_f (Gaussian elimination of the 6 x 6 pivot block,
// which in this frame is close to block diagonal, [[1, h], [1, -h]] per
// component).  The least-squares rows (the face points 2 and 4 of each face,
// the 12 WENO modes) in x_f are then a 6 x 6 normal system.  B' = R B and
// rho' = R rho, so n . B(rho) = n' . B'(rho') and the WENO rows' squared
// distance is unchanged: the minimiser is the one of the 12-unknown form.
// About 100 live words instead of a 12 x 12 Cholesky factor and a 6 x 12
// block in LDS, so two waves fit per SIMD, and no LDS.
// con(f, n, r): face f's face B, and its first normal and scaled centroid
// offset; pnt(f, t, n, r): the face-point B, normal and scaled offset of its
// point 2 + 2 t; mode(c, m): mode m of the WENO B component c.  Faces 0 right
// x, 1 left x, 2 up y, 3 down y, 4 top z, 5 bottom z.  x: the 12 coefficients.
__device__ __forceinline__ void put6(double* a, int f, double v) {
#pragma unroll
  for (int q = 0; q < 6; ++q) a[q] = f == q ? v : a[q];
}
__device__ __forceinline__ void rot3(const double* R, const double* v, double* o) {
#pragma unroll
  for (int r = 0; r < 3; ++r) o[r] = R[3 * r] * v[0] + R[3 * r + 1] * v[1] + R[3 * r + 2] * v[2];
}
// the row n' (x) (1, rho') split into the pivot and the free coefficients
__device__ __forceinline__ void split_row(const double* n, const double* r, double* rp, double* rf) {
  rp[0] = n[0];
  rp[1] = n[0] * r[0];
  rp[2] = n[1];
  rp[3] = n[1] * r[1];
  rp[4] = n[2];
  rp[5] = n[2] * r[2];
  rf[0] = n[0] * r[1];
  rf[1] = n[0] * r[2];
  rf[2] = n[1] * r[0];
  rf[3] = n[1] * r[2];
  rf[4] = n[2] * r[0];
  rf[5] = n[2] * r[1];
}
template <class Con, class Pnt, class Mode>
__device__ __forceinline__ void adp_clsq(const Con& con, const Pnt& pnt, const Mode& mode, double* x) {
  // pass 1: the constraint rows (the first point's normal at the centroid) and the face B
  double cn[3][6], cr[3][6], cd[6];
#pragma unroll 1
  for (int f = 0; f < 6; ++f) {
    double n[3], r[3];
    const double d = con(f, n, r);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      put6(cn[c], f, n[c]);
      put6(cr[c], f, r[c]);
    }
    put6(cd, f, d);
  }
  // the zone's frame
  double R[9];
  {
    double a[3], e2[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      a[c] = cn[c][0] + cn[c][1];
      e2[c] = cn[c][2] + cn[c][3];
    }
    double t = 1.0 / sqrt(a[0] * a[0] + a[1] * a[1] + a[2] * a[2]);
#pragma unroll
    for (int c = 0; c < 3; ++c) a[c] *= t;
    t = e2[0] * a[0] + e2[1] * a[1] + e2[2] * a[2];
#pragma unroll
    for (int c = 0; c < 3; ++c) e2[c] -= t * a[c];
    t = 1.0 / sqrt(e2[0] * e2[0] + e2[1] * e2[1] + e2[2] * e2[2]);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      e2[c] *= t;
      R[c] = a[c];
      R[3 + c] = e2[c];
    }
    R[6] = a[1] * e2[2] - a[2] * e2[1];
    R[7] = a[2] * e2[0] - a[0] * e2[2];
    R[8] = a[0] * e2[1] - a[1] * e2[0];
  }
  // the pivot block and its right-hand sides [free | d], eliminated in place
  double Ap[6][6], Wd[6][7];
#pragma unroll
  for (int f = 0; f < 6; ++f) {
    double n[3], r[3], nn[3], rr[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      n[c] = cn[c][f];
      r[c] = cr[c][f];
    }
    rot3(R, n, nn);
    rot3(R, r, rr);
    double rf[6];
    split_row(nn, rr, Ap[f], rf);
#pragma unroll
    for (int q = 0; q < 6; ++q) Wd[f][q] = rf[q];
    Wd[f][6] = cd[f];
  }
#pragma unroll
  for (int c = 0; c < 6; ++c) {
    const double od = 1.0 / Ap[c][c];
#pragma unroll
    for (int r = c + 1; r < 6; ++r) {
      const double m = Ap[r][c] * od;
#pragma unroll
      for (int q = c + 1; q < 6; ++q) Ap[r][q] -= m * Ap[c][q];
#pragma unroll
      for (int q = 0; q < 7; ++q) Wd[r][q] -= m * Wd[c][q];
    }
  }
#pragma unroll
  for (int r = 5; r >= 0; --r) {
    const double od = 1.0 / Ap[r][r];
#pragma unroll
    for (int q = 0; q < 7; ++q) {
      double t = Wd[r][q];
#pragma unroll
      for (int c = r + 1; c < 6; ++c) t -= Ap[r][c] * Wd[c][q];
      Wd[r][q] = t * od;
    }
  }
  // pass 2: the least-squares rows in the free coefficients
  double N[21], h[6];
#pragma unroll
  for (int q = 0; q < 21; ++q) N[q] = 0.0;
#pragma unroll
  for (int q = 0; q < 6; ++q) h[q] = 0.0;
#pragma unroll 1
  for (int f = 0; f < 6; ++f) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      double n[3], r[3], nn[3], rr[3];
      double tgt = pnt(f, t, n, r);
      rot3(R, n, nn);
      rot3(R, r, rr);
      double rp[6], red[6];
      split_row(nn, rr, rp, red);
#pragma unroll
      for (int q = 0; q < 6; ++q) {
        tgt -= rp[q] * Wd[q][6];
#pragma unroll
        for (int c = 0; c < 6; ++c) red[c] -= rp[q] * Wd[q][c];
      }
#pragma unroll
      for (int r2 = 0; r2 < 6; ++r2) {
        h[r2] += red[r2] * tgt;
#pragma unroll
        for (int c = 0; c <= r2; ++c) N[LIX(r2, c)] += red[r2] * red[c];
      }
    }
  }
  // the WENO modes u, in the zone's frame: b0' = R b0, G' = R G R^T
  double up[6], uf[6];
  {
    double b0[3], G[3][3], t[3][3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      b0[c] = mode(c, 0);
#pragma unroll
      for (int q = 0; q < 3; ++q) G[c][q] = mode(c, 1 + q);
    }
    double bp[3];
    rot3(R, b0, bp);
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int q = 0; q < 3; ++q) t[r][q] = R[3 * r] * G[0][q] + R[3 * r + 1] * G[1][q] + R[3 * r + 2] * G[2][q];
    double Gp[3][3];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int q = 0; q < 3; ++q) Gp[r][q] = t[r][0] * R[3 * q] + t[r][1] * R[3 * q + 1] + t[r][2] * R[3 * q + 2];
    up[0] = bp[0];
    up[1] = Gp[0][0];
    up[2] = bp[1];
    up[3] = Gp[1][1];
    up[4] = bp[2];
    up[5] = Gp[2][2];
    uf[0] = Gp[0][1];
    uf[1] = Gp[0][2];
    uf[2] = Gp[1][0];
    uf[3] = Gp[1][2];
    uf[4] = Gp[2][0];
    uf[5] = Gp[2][1];
  }
  // the WENO rows: free ones directly, pivot ones through x_p = e - W x_f
#pragma unroll
  for (int q = 0; q < 6; ++q) {
    N[LIX(q, q)] += 1.0;
    h[q] += uf[q];
  }
#pragma unroll
  for (int q = 0; q < 6; ++q) {
    const double tgt = up[q] - Wd[q][6];
#pragma unroll
    for (int r2 = 0; r2 < 6; ++r2) {
      h[r2] -= Wd[q][r2] * tgt;
#pragma unroll
      for (int c = 0; c <= r2; ++c) N[LIX(r2, c)] += Wd[q][r2] * Wd[q][c];
    }
  }
  // 6 x 6 Cholesky with reciprocal diagonals, then the two solves
#pragma unroll
  for (int c = 0; c < 6; ++c) {
    double d = N[LIX(c, c)];
#pragma unroll
    for (int q = 0; q < c; ++q) d -= N[LIX(c, q)] * N[LIX(c, q)];
    const double od = 1.0 / sqrt(d);
    N[LIX(c, c)] = od;
#pragma unroll
    for (int r = c + 1; r < 6; ++r) {
      double t = N[LIX(r, c)];
#pragma unroll
      for (int q = 0; q < c; ++q) t -= N[LIX(r, q)] * N[LIX(c, q)];
      N[LIX(r, c)] = t * od;
    }
  }
#pragma unroll
  for (int r = 0; r < 6; ++r) {
    double t = h[r];
#pragma unroll
    for (int q = 0; q < r; ++q) t -= N[LIX(r, q)] * h[q];
    h[r] = t * N[LIX(r, r)];
  }
#pragma unroll
  for (int r = 5; r >= 0; --r) {
    double t = h[r];
#pragma unroll
    for (int q = r + 1; q < 6; ++q) t -= N[LIX(q, r)] * h[q];
    h[r] = t * N[LIX(r, r)];
  }
  // the pivots, then back to the global frame: b0 = R^T b0', G = R^T G' R
  double xp[6];
#pragma unroll
  for (int q = 0; q < 6; ++q) {
    double t = Wd[q][6];
#pragma unroll
    for (int c = 0; c < 6; ++c) t -= Wd[q][c] * h[c];
    xp[q] = t;
  }
  {
    const double bp[3] = {xp[0], xp[2], xp[4]};
    const double Gp[3][3] = {{xp[1], h[0], h[1]}, {h[2], xp[3], h[3]}, {h[4], h[5], xp[5]}};
    double t[3][3];
#pragma unroll
    for (int c = 0; c < 3; ++c) x[4 * c] = R[c] * bp[0] + R[3 + c] * bp[1] + R[6 + c] * bp[2];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int q = 0; q < 3; ++q) t[r][q] = R[r] * Gp[0][q] + R[3 + r] * Gp[1][q] + R[6 + r] * Gp[2][q];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int q = 0; q < 3; ++q) x[4 * r + 1 + q] = t[r][0] * R[q] + t[r][1] * R[3 + q] + t[r][2] * R[6 + q];
  }
}

// Two_D_RS_Ez_3State_HLL (620riemann_2d/631...f:1-216): three zones around an
// edge, the faces 13, 21, 32 between them at 120 degrees in the solver frame;
// the HLL field from the wave triangle A, B, C of the six speeds.
__device__ __forceinline__ double emf3_hll(const double* sr, const double* sl, const double* ez, const double* bn) {
  const double h3 = 0.5 * sqrt(3.0), r3 = 1.0 / sqrt(3.0);
  const double o1 = 1.0 / (sr[0] - sl[0]), o2 = 1.0 / (sr[1] - sl[1]), o3 = 1.0 / (sr[2] - sl[2]);
  const double Ax = (sl[0] + 2.0 * sr[1]) * r3, Ay = -sl[0], Bx = (sl[1] - sr[2]) * r3, By = sl[1] + sr[2];
  const double Cx = -(sr[0] + 2.0 * sl[2]) * r3, Cy = -sr[0];
  const double xc = (Ax + Bx + Cx) / 3.0, yc = (Ay + By + Cy) / 3.0;
  const double lx[3] = {Ax - Cx, Bx - Ax, Cx - Bx}, ly[3] = {Ay - Cy, By - Ay, Cy - By};
  const double px[3] = {Ax, Bx, Cx}, py[3] = {Ay, By, Cy};
  const double mx[3] = {0.5 * (Ax + Cx), 0.5 * (Bx + Ax), 0.5 * (Cx + Bx)},
               my[3] = {0.5 * (Ay + Cy), 0.5 * (By + Ay), 0.5 * (Cy + By)};
  double l[3], nx[3], ny[3], Sn[3];
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    l[q] = sqrt(lx[q] * lx[q] + ly[q] * ly[q]);
    nx[q] = ly[q] / l[q];
    ny[q] = -lx[q] / l[q];
    Sn[q] = nx[q] * px[q] + ny[q] * py[q];
  }
  const double s = 0.5 * (l[0] + l[1] + l[2]);
  const double area = sqrt(s * (s - l[0]) * (s - l[1]) * (s - l[2]));
  // zone fields in the solver frame, their components along each face
  const double Bx1 = (2.0 * bn[1] + bn[0]) * r3, Bx2 = (bn[1] - bn[2]) * r3, Bx3 = -(2.0 * bn[2] + bn[0]) * r3;
  const double By1 = -bn[0], By2 = bn[1] + bn[2];
  const double t21 = -0.5 * Bx1 + h3 * By1, t22 = -0.5 * Bx2 + h3 * By2;
  const double t32 = -0.5 * Bx2 - h3 * By2, t33 = -0.5 * Bx3 - h3 * By1;
  // the 1-D HLL state of each face: tangential B, E, the frame components
  const double Bt13 = (sr[0] * Bx3 - sl[0] * Bx1 + ez[2] - ez[0]) * o1;
  const double E13 = (sr[0] * ez[0] - sl[0] * ez[2] - sr[0] * sl[0] * (Bx3 - Bx1)) * o1;
  const double Bt21 = (sr[1] * t21 - sl[1] * t22 + ez[0] - ez[1]) * o2;
  const double E21 = (sr[1] * ez[1] - sl[1] * ez[0] - sr[1] * sl[1] * (t21 - t22)) * o2;
  const double Bt32 = (sr[2] * t32 - sl[2] * t33 + ez[1] - ez[2]) * o3;
  const double E32 = (sr[2] * ez[2] - sl[2] * ez[1] - sr[2] * sl[2] * (t32 - t33)) * o3;
  const double Es[3] = {E13, E21, E32};
  const double Bsx[3] = {Bt13, -0.5 * Bt21 + h3 * bn[1], -0.5 * Bt32 - h3 * bn[2]};
  const double Bsy[3] = {-bn[0], h3 * Bt21 + 0.5 * bn[1], -h3 * Bt32 + 0.5 * bn[2]};
  if (sl[0] >= 0.0 && sr[1] <= 0.0) return ez[0];
  if (sl[1] >= 0.0 && sr[2] <= 0.0) return ez[1];
  if (sl[2] >= 0.0 && sr[0] <= 0.0) return ez[2];
  if (sl[0] * (sr[0] + 2.0 * sl[2]) + sr[0] * (sl[0] + 2.0 * sr[1]) <= 0.0) return E13;
  if ((sl[1] + sr[2]) * (sl[0] + 2.0 * sr[1]) + (sl[1] - sr[2]) * sl[0] <= 0.0) return E21;
  if ((sl[1] + sr[2]) * (sr[0] + 2.0 * sl[2]) - (sl[1] - sr[2]) * sr[0] <= 0.0) return E32;
  // strongly interacting state: the face states' fluxes around the triangle
  double sx = 0.0, sy = 0.0, mxs = 0.0, mys = 0.0;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const double fx = ny[q] * Es[q] - Sn[q] * Bsx[q], fy = -nx[q] * Es[q] - Sn[q] * Bsy[q];
    sx += fx * l[q];
    sy += fy * l[q];
    mxs += (mx[q] - xc) * fy * l[q];
    mys += (my[q] - yc) * fx * l[q];
  }
  const double BSSx = sx / (-2.0 * area), BSSy = sy / (-2.0 * area);
  return 0.5 * ((-xc * BSSy - mxs / area) + (yc * BSSx + mys / area));
}

}  // namespace csp1
