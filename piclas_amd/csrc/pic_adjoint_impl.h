// Self-consistent step through a fixed linear field operator, and the
// hand-written adjoint of interpolate + push + deposit over K such steps.
// Included once, at the end of pic_stage.hip (it uses the handle and the
// launch helpers defined there).
//
// Forward step n (state x^n, v^n sorted by element):
//   rho^n   = Dep(x^n)                      shape-function deposition (rho component)
//   rbar^n  = A rho^n                       rbar_e = sum_ijk w_i w_j w_k rho_e,ijk / 8
//   En^n    = G rbar^n                      E at the unique corner nodes (G given)
//   E^n     = P En^n                        trilinear corner interpolation at the Gauss points
//   F^n     = ext + E^n(x^n)                InterpolateFieldToParticle
//   v^{n+1} = Boris(v^n, F^n),  x^{n+1} = x^n + v^{n+1} dt   (then tracking and re-sort)
// Loss after K steps: W = eps0/2 sum_e sum_ijk w_i w_j w_k / sJ |E^K|^2 with
// E^K = P G A Dep(x^K) (CalcPotentialEnergy of the final deposition).
//
// Reverse sweep, adjoints lx, lv held per particle id:
//   lE^K = eps0 w / sJ E^K ;  lrbar = G^T P^T lE ;  lx += Dep_x^T (A^T lrbar)
//   step n, backwards:  lv' = lv + dt lx ;  (lv, lF) = (dB/dv, dB/dF)^T lv' ;
//                        lx += (dE/dx)^T lF ;  lE^n = sum_p L(xi_p) lF_p ;
//                        lrbar = G^T P^T lE^n ;  lx += Dep_x^T (A^T lrbar)
// The states of every step are recomputed from checkpoints taken every
// `every` steps, segment by segment.

namespace {

// ---- field operator kernels ---------------------------------------------------
template <int N>
__global__ __launch_bounds__(kBlock) void k_elem_mean(int nElems, const double *PS, QuadArgs Q, double *rbar) {
  constexpr int n1 = N + 1, nd = n1 * n1 * n1;
  const int e = blockIdx.x * kBlock + threadIdx.x;
  if (e >= nElems) return;
  double acc = 0.0;
  for (int k = 0; k < n1; ++k)
    for (int j = 0; j < n1; ++j)
#pragma unroll
      for (int i = 0; i < n1; ++i) {
        const int r = (k * n1 + j) * n1 + i;
        acc = acc + Q.wGP[i] * Q.wGP[j] * Q.wGP[k] * PS[((size_t)e * nd + r) * 4 + 3];
      }
  rbar[e] = acc / 8.0;
}

// y = M x for a dense row-major M[rows][cols]: one wave per row, lane-strided
// partial sums reduced by a butterfly (a fixed order)
__global__ __launch_bounds__(kBlock) void k_matvec(int64_t rows, int64_t cols, const double *Mx, const double *x, double *y) {
  const int64_t r = (int64_t(blockIdx.x) * kBlock + threadIdx.x) / kWave;
  const int lane = lane_id();
  if (r >= rows) return;
  const double *m = Mx + r * cols;
  double acc = 0.0;
  for (int64_t c = lane; c < cols; c += kWave) acc += m[c] * x[c];
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) acc = acc + __shfl_xor(acc, off, kWave);
  if (lane == 0) y[r] = acc;
}

// trilinear weight of CGNS corner q at the Gauss point (a1, a2, a3 in [0,1])
__device__ inline double corner_weight(int q, double a1, double a2, double a3) {
  switch (q) {
    case 0: return (1 - a1) * (1 - a2) * (1 - a3);
    case 1: return a1 * (1 - a2) * (1 - a3);
    case 2: return a1 * a2 * (1 - a3);
    case 3: return (1 - a1) * a2 * (1 - a3);
    case 4: return (1 - a1) * (1 - a2) * a3;
    case 5: return a1 * (1 - a2) * a3;
    case 6: return a1 * a2 * a3;
    default: return (1 - a1) * a2 * a3;
  }
}

template <int N>
__global__ __launch_bounds__(kBlock) void k_node_to_dof(DevMesh M, const int32_t *elemNode, const double *En, double *E) {
  constexpr int n1 = N + 1, nd = n1 * n1 * n1;
  const int64_t g = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  if (g >= int64_t(M.nElems) * nd) return;
  const int e = int(g / nd), r = int(g % nd);
  const int i = r % n1, j = (r / n1) % n1, k = r / (n1 * n1);
  const double a1 = (M.xGP[i] + 1.0) / 2.0, a2 = (M.xGP[j] + 1.0) / 2.0, a3 = (M.xGP[k] + 1.0) / 2.0;
  const int32_t *u = elemNode + (size_t)e * 8;
  for (int c = 0; c < 3; ++c) {
    double v = 0.0;
    for (int q = 0; q < 8; ++q) v = v + corner_weight(q, a1, a2, a3) * En[(size_t)u[q] * 3 + c];
    E[g * 3 + c] = v;
  }
}

// ---- adjoint kernels --------------------------------------------------------------
// lE = eps0 w_i w_j w_k / sJ E   (gradient of the field energy)
template <int N>
__global__ __launch_bounds__(kBlock) void k_adj_energy(int nElems, const double *E, const double *sJ, QuadArgs Q, double *lE) {
  constexpr int n1 = N + 1, nd = n1 * n1 * n1;
  const int64_t g = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  if (g >= int64_t(nElems) * nd) return;
  const int r = int(g % nd);
  const int i = r % n1, j = (r / n1) % n1, k = r / (n1 * n1);
  const double f = 8.8541878176e-12 * (Q.wGP[i] * Q.wGP[j] * Q.wGP[k] / sJ[g]);
  for (int c = 0; c < 3; ++c) lE[g * 3 + c] = f * E[g * 3 + c];
}

// P^T in two steps.  Per element, one wave with the DOFs on its lanes: the 8
// corner sums lEc[e][q] = sum_dof corner_weight_q(dof) lE_dof.
template <int N>
__global__ __launch_bounds__(kBlock) void k_adj_corner(DevMesh M, const double *lE, double *lEc) {
  constexpr int n1 = N + 1, nd = n1 * n1 * n1;
  const int e = (blockIdx.x * kBlock + threadIdx.x) / kWave;
  const int lane = lane_id();
  if (e >= M.nElems) return;
  double s[8][3];
#pragma unroll
  for (int q = 0; q < 8; ++q)
#pragma unroll
    for (int c = 0; c < 3; ++c) s[q][c] = 0.0;
  for (int r = lane; r < nd; r += kWave) {
    const double a1 = (M.xGP[r % n1] + 1.0) / 2.0, a2 = (M.xGP[(r / n1) % n1] + 1.0) / 2.0;
    const double a3 = (M.xGP[r / (n1 * n1)] + 1.0) / 2.0;
    const double *l = lE + ((size_t)e * nd + r) * 3;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const double w = corner_weight(q, a1, a2, a3);
#pragma unroll
      for (int c = 0; c < 3; ++c) s[q][c] = s[q][c] + w * l[c];
    }
  }
#pragma unroll
  for (int q = 0; q < 8; ++q)
#pragma unroll
    for (int c = 0; c < 3; ++c) {
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) s[q][c] = s[q][c] + __shfl_xor(s[q][c], off, kWave);
      if (lane == 3 * q + c) lEc[(size_t)e * 24 + lane] = s[q][c];
    }
}
// Per unique node, the corner sums of its incidences in element order
__global__ __launch_bounds__(kBlock) void k_adj_node(int nNodes, const int32_t *off, const int32_t *inc,
                                                     const double *lEc, double *lEn) {
  const int u = blockIdx.x * kBlock + threadIdx.x;
  if (u >= nNodes) return;
  double a[3] = {0.0, 0.0, 0.0};
  for (int q = off[u]; q < off[u + 1]; ++q)
    for (int c = 0; c < 3; ++c) a[c] = a[c] + lEc[(size_t)inc[q] * 3 + c];
  for (int c = 0; c < 3; ++c) lEn[(size_t)u * 3 + c] = a[c];
}

// Dep_x^T: for every particle, the derivative of sum_dof lrho_dof rho_dof
// with respect to its position; lrho_dof = lrbar_e w_i w_j w_k / 8 (A^T).
// rho_dof = sum_p f_p S^alpha, S = 1 - |x_p + shift - x_dof|^2 / R^2 (>= 0).
__global__ __launch_bounds__(kBlock) void k_adj_sf(DevMesh M, DevParts P, int64_t n, SFArgs A, const int32_t *srcOff,
                                                   const int32_t *tgt, const uint8_t *tgtShift, const double *lrbar,
                                                   QuadArgs Q, double *lx) {
  const int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  if (i >= n) return;
  const int e = P.elem[i];
  if (e < 0) return;
  const int sp = P.spec[i];
  const double q0 = M.charge[sp];
  if (!(fabs(q0) > 0.0)) return;
  const double f = q0 * M.mpf[sp] * A.w_sf;
  const int n1 = M.N + 1, nd = M.nDof;
  const double x0[3] = {P.x[i], P.y[i], P.z[i]};
  double g[3] = {0.0, 0.0, 0.0};
  for (int q = srcOff[e]; q < srcOff[e + 1]; ++q) {
    const int t = tgt[q];
    const int si = tgtShift[q];
    const double p[3] = {x0[0] + A.sh[si][0], x0[1] + A.sh[si][1], x0[2] + A.sh[si][2]};
    const double lr = lrbar[t] / 8.0;
    const double *xg = M.xGPe + (size_t)t * nd * 3;
    for (int r = 0; r < nd; ++r) {
      const double d0 = p[0] - xg[r * 3], d1 = p[1] - xg[r * 3 + 1], d2 = p[2] - xg[r * 3 + 2];
      const double r2 = d0 * d0 + d1 * d1 + d2 * d2;
      if (r2 > A.r2_sf) continue;
      const double S = 1. - A.r2_sf_inv * r2;
      double Sa1 = 1.0;   // S^(alpha-1)
      for (int ex = 2; ex <= A.alpha; ++ex) Sa1 = Sa1 * S;
      const int ii = r % n1, jj = (r / n1) % n1, kk = r / (n1 * n1);
      const double c = lr * Q.wGP[ii] * Q.wGP[jj] * Q.wGP[kk] * f * A.alpha * Sa1 * (-2.0 * A.r2_sf_inv);
      g[0] += c * d0; g[1] += c * d1; g[2] += c * d2;
    }
  }
  const int id = P.id[i];
  lx[(size_t)id * 3 + 0] += g[0];
  lx[(size_t)id * 3 + 1] += g[1];
  lx[(size_t)id * 3 + 2] += g[2];
}

// The same for N = 3 on axis-aligned tensor grids of Gauss points, where with
// u = x / R the argument S = 1 - (u_i - pu)^2 - (v_j - pv)^2 - (w_k - pw)^2
// splits by axis: 12 squares per target replace 64 distances, and the
// gradient sums factor into sums over i, j and k, 4 FP64 operations per DOF
// where the general kernel takes some 25 and a branch.  A plane of 16 DOFs
// that no lane's particle reaches is skipped (the particles of a wave are
// neighbours: they are sorted by element and z).
template <int ALPHA>
__global__ __launch_bounds__(kBlock) void k_adj_sf_cart(DevMesh M, DevParts P, int64_t n, SFArgs A, const int32_t *srcOff,
                                                        const int32_t *tgt, const uint8_t *tgtShift, const double *lrbar,
                                                        QuadArgs Q, double *lx) {
#pragma clang fp contract(fast)
  const int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  if (i >= n) return;
  const int e = P.elem[i];
  if (e < 0) return;
  const int sp = P.spec[i];
  const double q0 = M.charge[sp];
  if (!(fabs(q0) > 0.0)) return;
  const double x0[3] = {P.x[i], P.y[i], P.z[i]};
  const double Ri = A.r_inv;
  double g[3] = {0.0, 0.0, 0.0};
  for (int q = srcOff[e]; q < srcOff[e + 1]; ++q) {
    const int t = tgt[q];
    const int si = tgtShift[q];
    const double *xg = M.xGPe + (size_t)t * 64 * 3;
    const double px = x0[0] + A.sh[si][0], py = x0[1] + A.sh[si][1], pz = x0[2] + A.sh[si][2];
    double du[4], dv[4], dw[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      du[c] = (px - xg[c * 3]) * Ri;
      dv[c] = (py - xg[4 * c * 3 + 1]) * Ri;
      dw[c] = (pz - xg[16 * c * 3 + 2]) * Ri;
    }
    // squared distance to the DOF box across the planes: du runs monotonically
    auto gap = [](const double *d) {
      const double lo = fmin(d[0], d[3]), hi = fmax(d[0], d[3]);
      return fmax(fmax(lo, -hi), 0.0);
    };
    const double gu = gap(du), gv = gap(dv);
    const double dxy = gu * gu + gv * gv;
    double s2[4], wx[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      s2[c] = du[c] * du[c];
      wx[c] = Q.wGP[c] * du[c];
    }
    double gx = 0.0, gy = 0.0, gz = 0.0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const double zk = dw[k] * dw[k];
      // (a margin over the rounding of S; S = 0 beyond it)
      if (!__any(dxy + zk < 1.0 + 1e-9)) continue;
      double A1 = 0.0, AX = 0.0, AY = 0.0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const double D = (1.0 - zk) - dv[j] * dv[j];
        double si1 = 0.0, six = 0.0;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const double S = clamp01(D - s2[c]);   // (S <= 1: the clamp is free)
          double Sa = S;   // S^(alpha-1)
          if (ALPHA == 0) {
            for (int ex = 3; ex <= A.alpha; ++ex) Sa = Sa * S;
          } else {
#pragma unroll
            for (int ex = 3; ex <= ALPHA; ++ex) Sa = Sa * S;
          }
          si1 += Q.wGP[c] * Sa;
          six += wx[c] * Sa;
        }
        A1 += Q.wGP[j] * si1;
        AX += Q.wGP[j] * six;
        AY += (Q.wGP[j] * dv[j]) * si1;
      }
      gx += Q.wGP[k] * AX;
      gy += Q.wGP[k] * AY;
      gz += (Q.wGP[k] * dw[k]) * A1;
    }
    const double lr = lrbar[t];
    g[0] += lr * gx; g[1] += lr * gy; g[2] += lr * gz;
  }
  // lr / 8 * f * alpha * (-2 / R^2) * d, with d = R (du, dv, dw)
  const double f = q0 * M.mpf[sp] * A.w_sf;
  const double c = f * A.alpha * (-0.25 * Ri);
  const int id = P.id[i];
  lx[(size_t)id * 3 + 0] += c * g[0];
  lx[(size_t)id * 3 + 1] += c * g[1];
  lx[(size_t)id * 3 + 2] += c * g[2];
}

__device__ inline void cross3(const double a[3], const double b[3], double c[3]) {
  c[0] = a[1] * b[2] - a[2] * b[1];
  c[1] = a[2] * b[0] - a[0] * b[2];
  c[2] = a[0] * b[1] - a[1] * b[0];
}
__device__ inline double dot3(const double a[3], const double b[3]) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]; }

// Adjoint of the velocity update of boris_push: the forward pass at (v, E),
// then backwards through it, so that l (adjoint of the new velocity) gives
// lv = (dv'/dv)^T l and lE = (dv'/dE)^T l (the external B carries none).
__device__ inline void boris_vel_adjoint(double q, double m, const double E[3], const double B[3], double dt,
                                         const double v[3], const double l[3], double lv[3], double lE[3]) {
  const double c2i = c2_inv();
  const double c1 = (q * dt) / (m * 2.);
  const double g0 = 1.0 / sqrt(1.0 - dot3(v, v) * c2i);
  double vm[3], ub[3] = {0.0, 0.0, 0.0}, t[3], vp[3], cr[3], vn[3], w[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) vm[c] = v[c] * g0 + c1 * E[c];
  const double gm = sqrt(1.0 + dot3(vm, vm) * c2i);
  const double Bn = sqrt(dot3(B, B));
  if (Bn > 0.0)
#pragma unroll
    for (int c = 0; c < 3; ++c) ub[c] = B[c] / Bn;
  const double th = c1 / gm * Bn;
  const double tf = tan(th);
#pragma unroll
  for (int c = 0; c < 3; ++c) t[c] = tf * ub[c];
  cross3(vm, t, w);
#pragma unroll
  for (int c = 0; c < 3; ++c) vp[c] = vm[c] + w[c];
  const double f2 = 2.0 / (1.0 + dot3(t, t));
  cross3(vp, t, cr);
#pragma unroll
  for (int c = 0; c < 3; ++c) vn[c] = (vm[c] + f2 * cr[c]) + c1 * E[c];
  const double rd = 1.0 / sqrt(1.0 + dot3(vn, vn) * c2i);
  // v' = vn rd, rd = (1 + vn.vn / c^2)^(-1/2)
  double ln[3], lc[3], lvp[3], lt[3], lm[3];
  const double k0 = dot3(l, vn) * rd * rd * rd * c2i;
#pragma unroll
  for (int c = 0; c < 3; ++c) ln[c] = l[c] * rd - k0 * vn[c];
  // vn = vm + f2 vp x t + c1 E
  const double lf2 = dot3(ln, cr);
#pragma unroll
  for (int c = 0; c < 3; ++c) { lE[c] = c1 * ln[c]; lm[c] = ln[c]; lc[c] = f2 * ln[c]; }
  cross3(t, lc, lvp);
  cross3(lc, vp, lt);
  const double lT = -lf2 * f2 * f2;   // f2 = 2 / (1 + t.t)
#pragma unroll
  for (int c = 0; c < 3; ++c) lt[c] += lT * t[c];
  // vp = vm + vm x t
  cross3(t, lvp, w);
#pragma unroll
  for (int c = 0; c < 3; ++c) lm[c] += lvp[c] + w[c];
  cross3(lvp, vm, w);
#pragma unroll
  for (int c = 0; c < 3; ++c) lt[c] += w[c];
  // t = tan(th) ub, th = c1 Bn / gm, gm = sqrt(1 + vm.vm / c^2)
  const double lth = dot3(lt, ub) * (1.0 + tf * tf);
  const double kg = -lth * th / (gm * gm) * c2i;
#pragma unroll
  for (int c = 0; c < 3; ++c) lm[c] += kg * vm[c];
  // vm = v g0 + c1 E, g0 = (1 - v.v / c^2)^(-1/2)
  const double kv = dot3(lm, v) * c2i * g0 * g0 * g0;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    lE[c] += c1 * lm[c];
    lv[c] = lm[c] * g0 + kv * v[c];
  }
}

// Lagrange basis on the Gauss nodes and its derivative in product form, with
// c_i = 1 / prod_{m != i} (x_i - x_m) (no division)
template <int NP>
__device__ inline void lagrange_d(double x, const double *xg, const double *c, double *L, double *dL) {
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    double l = c[i], dl = 0.0;
#pragma unroll
    for (int m = 0; m < NP; ++m) {
      if (m == i) continue;
      const double d = x - xg[m];
      dl = dl * d + l;
      l = l * d;
    }
    L[i] = l;
    dL[i] = dl;
  }
}

// Reverse of one step for every particle of the stored step-n state:
// lv' = lv + dt lx ;  (lv, lF) = J_B^T lv' ;  lx += (dE/dx)^T lF.
// Writes lF and xi (sorted order) for the field scatter.  AFFINE: every
// element is a parallelepiped (xi and dxi/dx from the affine map).
template <int N, bool AFFINE>
__global__ __launch_bounds__(kBlock) void k_adj_push(DevMesh M, DevParts P, int64_t n, double dt, double *lx, double *lv,
                                                     double *lF, double *xiOut) {
#pragma clang fp contract(fast)
  constexpr int n1 = N + 1, nd = n1 * n1 * n1;
  const int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  if (i >= n) return;
  const int e = P.elem[i];
  const int id = P.id[i];
  const int sp = P.spec[i];
  const double q = M.charge[sp], m = M.mass[sp];
  const double x[3] = {P.x[i], P.y[i], P.z[i]};
  double lvp[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) lvp[c] = lv[(size_t)id * 3 + c] + dt * lx[(size_t)id * 3 + c];
  double xi[3] = {0, 0, 0};
  double lFo[3] = {0, 0, 0};
  double lvo[3] = {lvp[0], lvp[1], lvp[2]};
  if (fabs(q) > 0.0) {
    // the field of the forward step at this particle
    if (AFFINE) {
      affine_xi(M, e, x, xi);
    } else {
      ref_newton_start<N>(M, e, x, xi);
      ref_elem_newton(M, e, x, xi, true);
    }
    double L[3][n1], dL[3][n1];
#pragma unroll
    for (int d = 0; d < 3; ++d) lagrange_d<n1>(xi[d], M.xGP, M.cGP, L[d], dL[d]);
    const double *Ue = M.E + (size_t)e * nd * 3;
    double U[3] = {0, 0, 0}, dU[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};   // dU[c][d] = dE_c/dxi_d
#pragma unroll 1
    for (int k = 0; k < n1; ++k) {
      double s[3] = {0, 0, 0}, s0[3] = {0, 0, 0}, s1[3] = {0, 0, 0};
#pragma unroll
      for (int j = 0; j < n1; ++j) {
        double a[3] = {0, 0, 0}, b[3] = {0, 0, 0};
#pragma unroll
        for (int ii = 0; ii < n1; ++ii) {
          const double *u = Ue + ((k * n1 + j) * n1 + ii) * 3;
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            a[c] += u[c] * L[0][ii];
            b[c] += u[c] * dL[0][ii];
          }
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          s[c] += a[c] * L[1][j];
          s0[c] += b[c] * L[1][j];
          s1[c] += a[c] * dL[1][j];
        }
      }
      // (L and dL of the third direction by a select: k is a loop counter)
      double Lk = L[2][0], dLk = dL[2][0];
#pragma unroll
      for (int c = 1; c < n1; ++c)
        if (k == c) { Lk = L[2][c]; dLk = dL[2][c]; }
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        U[c] += s[c] * Lk;
        dU[c][0] += s0[c] * Lk;
        dU[c][1] += s1[c] * Lk;
        dU[c][2] += s[c] * dLk;
      }
    }
    const double Bx[3] = {M.ext[3], M.ext[4], M.ext[5]};
    const double F[3] = {M.ext[0] + U[0], M.ext[1] + U[1], M.ext[2] + U[2]};
    const double v0[3] = {P.vx[i], P.vy[i], P.vz[i]};
    boris_vel_adjoint(q, m, F, Bx, dt, v0, lvp, lvo, lFo);
    // lx_a += sum_c lF_c dE_c/dx_a = sum_d (sum_c lF_c dU[c][d]) dxi_d/dx_a
    double h[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) h[d] = lFo[0] * dU[0][d] + lFo[1] * dU[1][d] + lFo[2] * dU[2][d];
    double Ji[3][3];   // dxi/dx
    if (AFFINE) {
      const double *a = M.affine + (size_t)e * 12 + 3;
#pragma unroll
      for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int c = 0; c < 3; ++c) Ji[d][c] = a[3 * d + c];
    } else {
      // J[a][b] = dx_a/dxi_b of the element map at xi, inverted
      double Lc[3][2];
#pragma unroll
      for (int d = 0; d < 3; ++d) lagrange<2>(xi[d], M.xiCL, M.wBaryCL, Lc[d]);
      const double *dX = M.dXCL + (size_t)e * 72;
      double J[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
      for (int k = 0; k < 2; ++k)
        for (int j = 0; j < 2; ++j)
          for (int ii = 0; ii < 2; ++ii) {
            const double b2 = Lc[0][ii] * Lc[1][j] * Lc[2][k];
            const double *dp = dX + ((k * 2 + j) * 2 + ii) * 9;
            for (int a = 0; a < 3; ++a)
              for (int b = 0; b < 3; ++b) J[a][b] += dp[a * 3 + b] * b2;
          }
      const double det = get_det(J), sd = 1.0 / det;
      Ji[0][0] = (J[1][1] * J[2][2] - J[1][2] * J[2][1]) * sd;
      Ji[0][1] = (J[0][2] * J[2][1] - J[0][1] * J[2][2]) * sd;
      Ji[0][2] = (J[0][1] * J[1][2] - J[0][2] * J[1][1]) * sd;
      Ji[1][0] = (J[1][2] * J[2][0] - J[1][0] * J[2][2]) * sd;
      Ji[1][1] = (J[0][0] * J[2][2] - J[0][2] * J[2][0]) * sd;
      Ji[1][2] = (J[0][2] * J[1][0] - J[0][0] * J[1][2]) * sd;
      Ji[2][0] = (J[1][0] * J[2][1] - J[1][1] * J[2][0]) * sd;
      Ji[2][1] = (J[0][1] * J[2][0] - J[0][0] * J[2][1]) * sd;
      Ji[2][2] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) * sd;
    }
#pragma unroll
    for (int c = 0; c < 3; ++c)
      lx[(size_t)id * 3 + c] += h[0] * Ji[0][c] + h[1] * Ji[1][c] + h[2] * Ji[2][c];
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    lv[(size_t)id * 3 + c] = lvo[c];
    lF[i * 3 + c] = lFo[c];
    xiOut[i * 3 + c] = xi[c];
  }
}

// lE^n_dof = sum over the element's particles of L_ijk(xi_p) lF_p: a workgroup
// per element, its waves taking batches of 64 particles in turn.  One lane
// per particle forms the three bases once (formed by every DOF lane for
// every particle they were the kernel's time), then the lanes are the DOFs
// and add the batch from LDS; the waves' sums are added in wave order.
template <int N>
__global__ __launch_bounds__(kBlock) void k_adj_scatter(DevMesh M, const int32_t *start, const double *lF,
                                                        const double *xi, double *lE) {
#pragma clang fp contract(fast)
  constexpr int n1 = N + 1, nd = n1 * n1 * n1, nch = (nd + kWave - 1) / kWave, nw = kBlock / kWave;
  constexpr int kRow = 3 * n1 + 3;
  // the batches, then the waves' sums
  constexpr int kSums = nch * kWave * 3;
  constexpr int kB = N <= 4 ? kWave : 32;   // particles per batch (the bases of higher degrees take more room)
  __shared__ double lds[nw][kB * kRow > kSums ? kB * kRow : kSums];
  const int e = blockIdx.x, wib = threadIdx.x / kWave, lane = lane_id();
  double (*L)[kRow] = reinterpret_cast<double (*)[kRow]>(lds[wib]);
  double a[nch][3];
#pragma unroll
  for (int ch = 0; ch < nch; ++ch)
#pragma unroll
    for (int c = 0; c < 3; ++c) a[ch][c] = 0.0;
  const int s1 = start[e + 1];
  for (int base = start[e] + wib * kB; base < s1; base += nw * kB) {
    const int p = base + lane, cnt = min(kB, s1 - base);
    if (lane < cnt) {
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        double l[n1];
        lagrange_prod<n1>(xi[(size_t)p * 3 + d], M.xGP, M.cGP, l);
#pragma unroll
        for (int q = 0; q < n1; ++q) L[lane][d * n1 + q] = l[q];
        L[lane][3 * n1 + d] = lF[(size_t)p * 3 + d];
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int j = 0; j < cnt; ++j) {
      const double f0 = L[j][3 * n1], f1 = L[j][3 * n1 + 1], f2 = L[j][3 * n1 + 2];
#pragma unroll
      for (int ch = 0; ch < nch; ++ch) {
        const int r = min(ch * kWave + lane, nd - 1);
        const double w = L[j][r % n1] * L[j][n1 + (r / n1) % n1] * L[j][2 * n1 + r / (n1 * n1)];
        a[ch][0] += w * f0;
        a[ch][1] += w * f1;
        a[ch][2] += w * f2;
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
#pragma unroll
  for (int ch = 0; ch < nch; ++ch)
#pragma unroll
    for (int c = 0; c < 3; ++c) lds[wib][(ch * kWave + lane) * 3 + c] = a[ch][c];
  __syncthreads();
  for (int r = threadIdx.x; r < nd * 3; r += kBlock) {
    double sum = lds[0][r];
#pragma unroll
    for (int k = 1; k < nw; ++k) sum += lds[k][r];
    lE[(size_t)e * nd * 3 + r] = sum;
  }
}

// The sorted particle state (positions, velocities, element, id, species and
// the segment table) from one set of arrays to another, in one launch
struct StateCopy {
  const double *sx[6];
  double *dx[6];
  const int32_t *selem, *sid, *sstart;
  int32_t *delem, *did, *dstart;
  const uint8_t *sspec;
  uint8_t *dspec, *dnew;   // dnew: IsNewPart, cleared when given
};
__global__ __launch_bounds__(kBlock) void k_copy_state(int64_t n, int nStart, StateCopy C) {
  const int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  if (i < nStart) C.dstart[i] = C.sstart[i];
  if (i >= n) return;
#pragma unroll
  for (int c = 0; c < 6; ++c) C.dx[c][i] = C.sx[c][i];
  C.delem[i] = C.selem[i];
  C.did[i] = C.sid[i];
  C.dspec[i] = C.sspec[i];
  if (C.dnew) C.dnew[i] = 0;
}

__global__ void k_copy_f64(const double *a, double *b, int64_t n) {
  const int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  if (i < n) b[i] = a[i];
}

// ---- host side ------------------------------------------------------------------
// most memory for the fields of the forward steps
constexpr size_t kFieldBytes = size_t(16) << 30;

// device memory that the call can do without: null where there is none
double *try_alloc(pic_handle *h, size_t count) {
  void *q = nullptr;
  if (hipMalloc(&q, count * sizeof(double)) != hipSuccess) {
    (void)hipGetLastError();   // (not left for the next check)
    return nullptr;
  }
  h->allocs.push_back(q);
  return static_cast<double *>(q);
}
template <typename T>
void release(pic_handle *h, T *&p) {
  if (!p) return;
  h->allocs.erase(std::find(h->allocs.begin(), h->allocs.end(), static_cast<void *>(p)));
  (void)hipFree(p);
  p = nullptr;
}
void release_fields(pic_handle *h) {
  for (double *&E : h->adj.Es) release(h, E);
  h->adj.Es.clear();
}

int alloc_state(pic_handle *h, StepState &S) {
  int rc = 0;
  rc |= dalloc(h, &S.x, size_t(h->cap) * 6);
  rc |= dalloc(h, &S.elem, h->cap);
  rc |= dalloc(h, &S.id, h->cap);
  rc |= dalloc(h, &S.spec, h->cap);
  rc |= dalloc(h, &S.start, h->hm.nElems + 1);
  if (rc) {   // all or nothing: a later call tries again
    (void)hipGetLastError();
    release(h, S.x); release(h, S.elem); release(h, S.id); release(h, S.spec); release(h, S.start);
  }
  return rc;
}

// What every call of pic_adjoint needs: the checkpoints, and for gradients
// the states of one segment (the first one's slot holds the state after the
// last step) and the adjoint vectors.
int alloc_required(pic_handle *h, int nck, int every, bool backward) {
  Adjoint &a = h->adj;
  if (int(a.ck.size()) < nck) a.ck.resize(nck);
  for (int c = 0; c < nck; ++c)
    if (!a.ck[c].x && alloc_state(h, a.ck[c])) return PIC_EHIP;
  if (!backward) return 0;
  if (int(a.seg.size()) < every) a.seg.resize(every);
  for (int c = 0; c < every; ++c)
    if (!a.seg[c].x && alloc_state(h, a.seg[c])) return PIC_EHIP;
  for (double **v : {&a.lx, &a.lv, &a.lF, &a.xi})
    if (!*v && dalloc(h, v, size_t(h->cap) * 3)) {
      (void)hipGetLastError();
      return PIC_EHIP;
    }
  return 0;
}

// The fields of K steps of nE3 values, if they fit kFieldBytes (or
// PIC_ADJOINT_FIELD_BYTES) and half of the memory that is free, and the
// allocations succeed; else none are held.
bool keep_fields(pic_handle *h, int K, size_t nE3) {
  std::vector<double *> &Es = h->adj.Es;
  if (int(Es.size()) >= K) return true;
  size_t limit = kFieldBytes, avail = 0, total = 0;
  if (const char *k = std::getenv("PIC_ADJOINT_FIELD_BYTES")) limit = std::strtoull(k, nullptr, 10);
  const size_t bytes = nE3 * sizeof(double);
  if (hipMemGetInfo(&avail, &total) == hipSuccess) limit = std::min(limit, Es.size() * bytes + avail / 2);
  while (int(Es.size()) < K) {
    double *E = (Es.size() + 1) * bytes <= limit ? try_alloc(h, nE3) : nullptr;
    if (!E) {
      release_fields(h);
      return false;
    }
    Es.push_back(E);
  }
  return true;
}

void copy_state(pic_handle *h, const StateCopy &C, int64_t n) {
  const int nStart = h->hm.nElems + 1;
  hipLaunchKernelGGL(k_copy_state, dim3(grid_for(std::max<int64_t>(n, nStart))), dim3(kBlock), 0, h->stream, n, nStart, C);
}

int save_state(pic_handle *h, StepState &S) {
  const size_t cap = size_t(h->cap);
  StateCopy C{};
  const double *src[6] = {h->P.x, h->P.y, h->P.z, h->P.vx, h->P.vy, h->P.vz};
  for (int c = 0; c < 6; ++c) { C.sx[c] = src[c]; C.dx[c] = S.x + c * cap; }
  C.selem = h->P.elem; C.sid = h->P.id; C.sspec = h->P.spec; C.sstart = h->start;
  C.delem = S.elem; C.did = S.id; C.dspec = S.spec; C.dstart = S.start;
  copy_state(h, C, h->n);
  HIPCHK(hipGetLastError());
  S.n = h->n;
  return 0;
}

int restore_state(pic_handle *h, const StepState &S) {
  const size_t cap = size_t(h->cap);
  StateCopy C{};
  double *dst[6] = {h->P.x, h->P.y, h->P.z, h->P.vx, h->P.vy, h->P.vz};
  for (int c = 0; c < 6; ++c) { C.sx[c] = S.x + c * cap; C.dx[c] = dst[c]; }
  C.selem = S.elem; C.sid = S.id; C.sspec = S.spec; C.sstart = S.start;
  C.delem = h->P.elem; C.did = h->P.id; C.dspec = h->P.spec; C.dstart = h->start;
  C.dnew = h->P.isNew;
  copy_state(h, C, S.n);
  HIPCHK(hipGetLastError());
  h->recFresh = false;
  h->n = S.n;
  return 0;
}

// a DevParts view of a stored state
DevParts view_of(pic_handle *h, const StepState &S) {
  DevParts v{};
  const size_t cap = size_t(h->cap);
  v.x = S.x; v.y = S.x + cap; v.z = S.x + 2 * cap;
  v.vx = S.x + 3 * cap; v.vy = S.x + 4 * cap; v.vz = S.x + 5 * cap;
  v.elem = S.elem; v.id = S.id; v.spec = S.spec;
  return v;
}

QuadArgs quad_of(pic_handle *h) {
  QuadArgs Q{};
  for (int i = 0; i <= h->hm.N; ++i) Q.wGP[i] = h->hm.wGP[i];
  return Q;
}

// E = P G A rho of the current deposition (h->PS) into E
int field_from_source(pic_handle *h, double *E) {
  const int ne = h->hm.nElems, N = h->hm.N;
  QuadArgs Q = quad_of(h);
  LAUNCH_N(k_elem_mean, N, dim3(grid_for(ne)), ne, h->PS, Q, h->adj.rbar);
  const int64_t rows = int64_t(h->hm.nUnique) * 3;
  hipLaunchKernelGGL(k_matvec, dim3(grid_for(rows * kWave)), dim3(kBlock), 0, h->stream, rows, int64_t(ne), h->adj.G,
                     h->adj.rbar, h->adj.En);
  LAUNCH_N(k_node_to_dof, N, dim3(grid_for(int64_t(ne) * h->hm.nDof)), h->M, h->adj.elemNode, h->adj.En, E);
  HIPCHK(hipGetLastError());
  return 0;
}

// interpolate, push, track and re-sort in the field E
int sc_push(pic_handle *h, double dt, const double *E) {
  const int64_t n = h->n;
  const int32_t *nDev = h->start + h->hm.nElems;
  DevMesh M = h->M;
  M.E = E;
  if (int rc = push_track(h, M, n, dt, nDev, false)) return rc;
  h->recFresh = false;
  HIPCHK(hipGetLastError());
  return enqueue_sort(h, n, false);
}

// one self-consistent step: deposit, field (into E), push/track, re-sort
int sc_step(pic_handle *h, double dt, double *E) {
  if (h->par.tracking != PIC_TRACK_TRIA) return fail(PIC_EINVAL, "self-consistent steps: TriaTracking only");
  if (int rc = run_deposition(h, false)) return rc;
  if (int rc = field_from_source(h, E)) return rc;
  const int64_t n0 = h->n;
  if (int rc = sc_push(h, dt, E)) return rc;
  if (int rc = read_count(h)) return rc;
  if (h->n != n0) return fail(PIC_ETRACK, "self-consistent steps: particles left the domain (periodic meshes only)");
  return 0;
}

// loss of the current state: field energy of the field of its deposition
int sc_loss(pic_handle *h, double *loss) {
  if (int rc = run_deposition(h, false)) return rc;
  if (int rc = field_from_source(h, h->E)) return rc;
  double w = 0.0;
  if (int rc = elem_integral(h, 1, &w)) return rc;
  *loss = w * 8.8541878176e-12 * 0.5;
  return 0;
}

// lrbar = G^T P^T lE, then lx += Dep_x^T(A^T lrbar) at the state in h->P / view
int adj_field_to_x(pic_handle *h, const DevParts &V, int64_t n) {
  const int N = h->hm.N;
  LAUNCH_N(k_adj_corner, N, dim3(grid_for(int64_t(h->hm.nElems) * kWave)), h->M, h->adj.lE, h->adj.lEc);
  hipLaunchKernelGGL(k_adj_node, dim3(grid_for(h->hm.nUnique)), dim3(kBlock), 0, h->stream, h->hm.nUnique,
                     h->adj.nodeOff, h->adj.nodeInc, h->adj.lEc, h->adj.lEn);
  const int64_t rows = h->hm.nElems, cols = int64_t(h->hm.nUnique) * 3;
  hipLaunchKernelGGL(k_matvec, dim3(grid_for(rows * kWave)), dim3(kBlock), 0, h->stream, rows, cols, h->adj.GT,
                     h->adj.lEn, h->adj.lrbar);
  QuadArgs Q = quad_of(h);
  auto kp = !h->sf.cartesian ? k_adj_sf : h->sf.alpha == 2 ? k_adj_sf_cart<2> : h->sf.alpha == 3 ? k_adj_sf_cart<3>
                                                                                     : k_adj_sf_cart<0>;
  hipLaunchKernelGGL(kp, dim3(grid_for(std::max<int64_t>(n, 1))), dim3(kBlock), 0, h->stream, h->M, V, n, h->sf,
                     h->adj.srcOff, h->adj.tgt, h->adj.tgtShift, h->adj.lrbar, Q, h->adj.lx);
  HIPCHK(hipGetLastError());
  return 0;
}

}  // namespace

extern "C" {

int pic_set_field_operator(pic_handle *h, const double *G) {
  if (!h || !G) return fail(PIC_EINVAL, "pic_set_field_operator: null argument");
  if (h->par.deposition != PIC_DEPO_SF) return fail(PIC_EINVAL, "pic_set_field_operator: shape_function deposition only");
  if (h->par.tracking != PIC_TRACK_TRIA) return fail(PIC_EINVAL, "pic_set_field_operator: TriaTracking only");
  if (h->par.precision != PIC_PREC_FP64) return fail(PIC_EINVAL, "pic_set_field_operator: FP64 only");
  if (set_device(h)) return PIC_EHIP;
  const int ne = h->hm.nElems, nu = h->hm.nUnique;
  const size_t rows = size_t(nu) * 3;
  Adjoint &a = h->adj;
  if (!a.G) {
    int rc = 0;
    rc |= dalloc(h, &a.G, rows * ne);
    rc |= dalloc(h, &a.GT, rows * ne);
    rc |= dalloc(h, &a.rbar, ne);
    rc |= dalloc(h, &a.lrbar, ne);
    rc |= dalloc(h, &a.En, rows);
    rc |= dalloc(h, &a.lEn, rows);
    rc |= dalloc(h, &a.lE, size_t(ne) * h->hm.nDof * 3);
    rc |= dalloc(h, &a.lEc, size_t(ne) * 24);
    rc |= upload(h, &a.elemNode, h->hm.elemNode);
    rc |= upload(h, &a.nodeOff, h->hm.nodeOff);
    rc |= upload(h, &a.nodeInc, h->hm.nodeInc);
    rc |= upload(h, &a.srcOff, h->hm.sfSrcOff);
    rc |= upload(h, &a.tgt, h->hm.sfTgt);
    rc |= upload(h, &a.tgtShift, h->hm.sfTgtShift);
    if (rc) return PIC_EHIP;
  }
  HIPCHK(hipMemcpy(a.G, G, rows * ne * sizeof(double), hipMemcpyHostToDevice));
  std::vector<double> T(rows * ne);
  for (size_t r = 0; r < rows; ++r)
    for (int e = 0; e < ne; ++e) T[size_t(e) * rows + r] = G[r * ne + e];
  HIPCHK(hipMemcpy(a.GT, T.data(), rows * ne * sizeof(double), hipMemcpyHostToDevice));
  return PIC_OK;
}

int pic_sc_time_step(pic_handle *h, double dt, int32_t nsteps, double *loss) {
  if (!h) return fail(PIC_EINVAL, "pic_sc_time_step: null handle");
  if (!h->adj.G) return fail(PIC_ESTATE, "pic_sc_time_step: call pic_set_field_operator first");
  if (int rc = require_particles(h)) return rc;
  if (set_device(h)) return PIC_EHIP;
  for (int it = 0; it < nsteps; ++it)
    if (int rc = sc_step(h, dt, h->E)) return rc;
  if (loss)
    if (int rc = sc_loss(h, loss)) return rc;
  HIPCHK(hipStreamSynchronize(h->stream));
  h->stagedValid = false;
  return PIC_OK;
}

int pic_adjoint(pic_handle *h, double dt, int32_t K, int32_t every, double *loss, double *dLdx0, double *dLdv0) {
  if (!h || !loss) return fail(PIC_EINVAL, "pic_adjoint: null argument");
  if (!h->adj.G) return fail(PIC_ESTATE, "pic_adjoint: call pic_set_field_operator first");
  if (K < 1 || every < 1) return fail(PIC_EINVAL, "pic_adjoint: K and the checkpoint interval must be >= 1");
  if (int rc = require_particles(h)) return rc;
  if (set_device(h)) return PIC_EHIP;
  Adjoint &a = h->adj;
  const int nck = (K + every - 1) / every;
  const bool backward = dLdx0 || dLdv0;
  const int64_t nE3 = int64_t(h->hm.nElems) * h->hm.nDof * 3;
  if (alloc_required(h, nck, every, backward)) {
    release_fields(h);   // (of an earlier call)
    if (int rc = alloc_required(h, nck, every, backward)) return rc;
  }
  // The field of every forward step is kept where there is room, so that the
  // reverse sweep recomputes positions and velocities only (a deposition
  // costs some ten pushes); else it keeps those of a segment and deposits
  // again, and runs the last steps again at the end.
  const bool keep = backward && keep_fields(h, K, size_t(nE3));
  if (backward && !keep)
    for (int c = 0; c < every; ++c)
      if (!a.seg[c].E && !(a.seg[c].E = try_alloc(h, nE3)))
        return fail(PIC_EHIP, "pic_adjoint: no device memory for the fields of a segment");
  // what the stage holds after K steps; without room, the last ones are run again
  if (keep && !a.finE) a.finE = try_alloc(h, nE3);
  if (keep && !a.PS) a.PS = try_alloc(h, nE3 / 3 * 4);
  const bool fin = keep && a.finE && a.PS;
  const int64_t n = h->n;
  // the steps start from running particles (no IsNewPart half step)
  hipLaunchKernelGGL(k_fill_u8, dim3(grid_for(std::max<int64_t>(n, 1))), dim3(kBlock), 0, h->stream, h->P.isNew, n,
                     uint8_t(0));
  const int N = h->hm.N;
  const int ne = h->hm.nElems;
  auto copy = [&](const double *src, double *dst, int64_t cnt) {
    hipLaunchKernelGGL(k_copy_f64, dim3(grid_for(cnt)), dim3(kBlock), 0, h->stream, src, dst, cnt);
  };
  // forward: checkpoints every `every` steps
  for (int it = 0; it < K; ++it) {
    if (it % every == 0)
      if (int rc = save_state(h, a.ck[it / every])) return rc;
    if (int rc = sc_step(h, dt, keep ? a.Es[it] : h->E)) return rc;
  }
  if (fin) {
    if (int rc = save_state(h, a.seg[0])) return rc;
    copy(a.Es[K - 1], a.finE, nE3);
    copy(h->PS, a.PS, nE3 / 3 * 4);
  }
  if (int rc = sc_loss(h, loss)) return rc;
  HIPCHK(hipStreamSynchronize(h->stream));
  if (!backward) return PIC_OK;
  // reverse: gradient of the field energy at step K
  QuadArgs Q = quad_of(h);
  hipLaunchKernelGGL(k_fill_f64, dim3(grid_for(int64_t(h->cap) * 3)), dim3(kBlock), 0, h->stream, a.lx, int64_t(h->cap) * 3);
  hipLaunchKernelGGL(k_fill_f64, dim3(grid_for(int64_t(h->cap) * 3)), dim3(kBlock), 0, h->stream, a.lv, int64_t(h->cap) * 3);
  LAUNCH_N(k_adj_energy, N, dim3(grid_for(int64_t(ne) * h->hm.nDof)), ne, h->E, h->sJ, Q, a.lE);
  if (int rc = adj_field_to_x(h, h->P, n)) return rc;
  // segments, last first: recompute the step states from the checkpoint, then reverse them
  for (int c = nck - 1; c >= 0; --c) {
    const int s0 = c * every, s1 = std::min(K, s0 + every);
    if (s1 - s0 > 1 || !keep)
      if (int rc = restore_state(h, a.ck[c])) return rc;
    for (int it = s0; it < s1; ++it) {
      if (it > s0)
        if (int rc = save_state(h, a.seg[it - s0])) return rc;
      double *E = keep ? a.Es[it] : a.seg[it - s0].E;
      if (!keep) {
        if (int rc = run_deposition(h, false)) return rc;
        if (int rc = field_from_source(h, E)) return rc;
      }
      if (it + 1 < s1)   // (the next checkpoint holds the state after the last)
        if (int rc = sc_push(h, dt, E)) return rc;
    }
    for (int it = s1 - 1; it >= s0; --it) {
      const StepState &S = it == s0 ? a.ck[c] : a.seg[it - s0];
      DevParts V = view_of(h, S);
      // the forward step read E^it: point the mesh view at the stored field
      DevMesh Mstep = h->M;
      Mstep.E = keep ? a.Es[it] : a.seg[it - s0].E;
      if (S.n > 0) {
        const dim3 grid(grid_for(S.n));
        if (Mstep.affine) { LAUNCH_N2(k_adj_push, N, true, grid, Mstep, V, S.n, dt, a.lx, a.lv, a.lF, a.xi); }
        else { LAUNCH_N2(k_adj_push, N, false, grid, Mstep, V, S.n, dt, a.lx, a.lv, a.lF, a.xi); }
      }
      LAUNCH_N(k_adj_scatter, N, dim3(ne), Mstep, S.start, a.lF, a.xi, a.lE);
      HIPCHK(hipGetLastError());
      if (int rc = adj_field_to_x(h, V, S.n)) return rc;
    }
  }
  // the stage ends in the state after K steps
  if (int rc = restore_state(h, fin ? a.seg[0] : a.ck[nck - 1])) return rc;
  if (fin) {
    copy(a.finE, h->E, nE3);
    copy(a.PS, h->PS, nE3 / 3 * 4);
  } else {
    for (int it = (nck - 1) * every; it < K; ++it)
      if (int rc = sc_step(h, dt, h->E)) return rc;
  }
  HIPCHK(hipStreamSynchronize(h->stream));
  const int64_t nt = h->nTotal;
  if (dLdx0) HIPCHK(hipMemcpy(dLdx0, a.lx, nt * 3 * sizeof(double), hipMemcpyDeviceToHost));
  if (dLdv0) HIPCHK(hipMemcpy(dLdv0, a.lv, nt * 3 * sizeof(double), hipMemcpyDeviceToHost));
  h->stagedValid = false;
  return PIC_OK;
}

}  // extern "C"
