// lbf_physics.h -- per-node physics shared by the fused and stage kernels.
#pragma once
#include "lbf_common.h"

namespace lbf {

template <class R>
struct NodeIn {  // collision input of one node
  R P, u, v, w, xx, yy, zz, xy, xz, yz;  // P, velocity, non-equilibrium Pi - u u
  R ax, ay, az;                          // force / rho_phi
  R om;                                  // relaxation rate
};

__device__ __forceinline__ int wrapg(int i, int n) {
  // periodic wrap for i in [-n, 2n)
  i = i < 0 ? i + n : i;
  return i >= n ? i - n : i;
}
__device__ __forceinline__ int clampi(int i, int lo, int hi) { return i < lo ? lo : (i > hi ? hi : i); }

__device__ __forceinline__ int8_t isf_at(const int8_t* isfh, int x, int y, int z, int nx, int ny, int nz) {
  // isfluid with the reference's 1-node halo; x,y,z unwrapped, clamped to [-1, n]
  x = clampi(x, -1, nx); y = clampi(y, -1, ny); z = clampi(z, -1, nz);
  return isfh[(size_t)(x + 1) + (size_t)(nx + 2) * ((size_t)(y + 1) + (size_t)(ny + 2) * (size_t)(z + 1))];
}

// One word per node of the haloed isfluid array, for the fused kernel: bit c
// (cidx of a velocity, 13 excepted) says that the node upstream of it, x - c,
// is solid; NODE_FLUID and NODE_WALL stand for isfluid != 0 and isfluid = -1.
// Only -1 nodes carry direction bits (nothing reads the others').
constexpr uint32_t NODE_FLUID = 1u << 31, NODE_WALL = 1u << 30;
__host__ __device__ inline size_t halo_nodes(const DevParams& dp) {
  return (size_t)(dp.nx + 2) * (dp.ny + 2) * (dp.nz + 2);
}

// ---------------------------------------------------------------------------
// Per-node rates shared by the moments stage, the collision and the near-wall
// closure: 1/rho_phi (two-component DENSRATIO; 1 otherwise), the kinematic
// viscosity (the density-weighted two-component mix, or visc1) and the plain
// relaxation rate 1/(3 nu + 1/2).  Computed once per node: the quarter-rate
// reciprocals are not repeated in the branches that use them.
template <class R>
struct NodeRates {
  R irho, visc, om0;
};
// STD (also below): the switches every two-component configuration sets,
// DENSRATIO with INTERFACE_INCOMP, no BUOYANCY_FORCING and no SMAGORINSKI (one
// component: no SMAGORINSKI), compiled in; std_switches() tells where it holds.
template <bool TWO, class R, bool STD = false>
__device__ __forceinline__ NodeRates<R> node_rates(const DevParams& dp, R phl) {
  const Phys<R>& ph = dp.ph<R>();
  NodeRates<R> r;
  r.irho = (TWO && (STD || dp.dens)) ? rcp(ph.rho_r * phl + ((R)1 - phl) * ph.rho_b) : (R)1;
  if (TWO) {
    // without DENSRATIO the reference's viscosity mix still reads rho_r/rho_b
    r.visc = (ph.rho_r * ph.visc1 * phl + ((R)1 - phl) * ph.visc2 * ph.rho_b) * r.irho;
    r.om0 = rcp(r.visc * (R)3 + (R)0.5);
  } else {
    r.visc = ph.visc1;
    r.om0 = ph.omega;
  }
  return r;
}

// ---------------------------------------------------------------------------
// Moments stage of one node (lb_cuda_moments_module.f90:104-339), in place on
// the loaded moments m; returns the stored force tF.  The terms along grad phi
// share their factors (surface tension and density-ratio pressure as one
// coefficient, (rho_r - rho_b) mask nu as one), and the divisions by rho_phi,
// the INTERFACE_INCOMP denominator and tau*cs^2 are multiplications by one
// reciprocal each, the first and last taken from the node's rates
// (nr = node_rates(dp, phl)).
// rflux: the REPULSIVE_FLUX flux of this node (locaux 6..8), or null.
template <bool TWO, class R, bool STD = false>
__device__ __forceinline__ void moments_stage(const DevParams& dp, const NodeRates<R>& nr, R phl, R gfx, R gfy,
                                              R gfz, R lap, R dvt, R uox, R uoy, R uoz, Mom<R>& m, R& tFx, R& tFy,
                                              R& tFz, const R* rflux = nullptr) {
  const Phys<R>& ph = dp.ph<R>();
  const R HALF = (R)0.5, ONE = (R)1;
  const bool dens = TWO && (STD || dp.dens != 0);
  const bool buoy = !STD && dp.buoy != 0, incomp = STD || dp.incomp != 0;
  const R rr = ph.rho_r, rb = ph.rho_b, dr = rr - rb;
  const R irho = dens ? nr.irho : ONE;
  R mask = 0, rhophi = ONE, Fx = ph.fx, Fy = ph.fy, Fz = ph.fz;
  if (TWO) mask = (R)4.0 * phl * (ONE - phl);
  if (dens) {
    rhophi = rr * phl + (ONE - phl) * rb;
    const R rf = buoy ? rhophi - (rr + rb) * HALF : rhophi;
    Fx = rf * ph.fx; Fy = rf * ph.fy; Fz = rf * ph.fz;
  }
  R kv = 0;
  if (TWO) {
    // 4 beta phi (phi - 1) (phi - 1/2) = -beta mask (phi - 1/2)
    R st = -(ph.beta * mask * (phl - HALF)) - ph.kapp * lap;
    if (dens) {
      st = st - mask * m.P * (dr * (R)(1.0 / 3.0));
      // visc / (tau cs^2) with tau = 3 visc + 1/2, as 3 visc / tau: 1/tau is
      // the node's plain relaxation rate
      kv = mask * (nr.visc * (R)3) * nr.om0 * dr;
    }
    Fx = Fx + st * gfx; Fy = Fy + st * gfy; Fz = Fz + st * gfz;
    if (rflux) {
      // REPULSIVE_FLUX (moments:148-160): rho_phi * flux clamped to +-1e-3, times rho_phi
      R fr[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        R mt = rflux[c] * rhophi;
        if (fabs(mt) > (R)1.0e-3) mt = (R)1.0e-3 * (mt < (R)0 ? (R)-1 : (R)1);
        fr[c] = mt * rhophi;
      }
      Fx = Fx + fr[0]; Fy = Fy + fr[1]; Fz = Fz + fr[2];
    }
  }
  tFx = Fx; tFy = Fy; tFz = Fz;
  if (dens) {
    const R pxx = m.xx - uox * uox, pyy = m.yy - uoy * uoy, pzz = m.zz - uoz * uoz;
    const R pxy = m.xy - uox * uoy, pxz = m.xz - uox * uoz, pyz = m.yz - uoy * uoz;
    Fx = Fx - kv * (pxx * gfx + pxy * gfy + pxz * gfz);
    Fy = Fy - kv * (pyy * gfy + pxy * gfx + pyz * gfz);
    Fz = Fz - kv * (pzz * gfz + pxz * gfx + pyz * gfy);
  }
  const R hi = HALF * irho;
  R u = m.u + Fx * hi, v = m.v + Fy * hi, w = m.w + Fz * hi;
  if (dens && incomp) {
    const R a = dr * (ph.tau_diff * lap - ph.sharp_c * dvt);
    const R iden = rcp(ONE - a * hi);
    u = u * iden; v = v * iden; w = w * iden;
    tFx = tFx - a * u; tFy = tFy - a * v; tFz = tFz - a * w;
    Fx = Fx - a * u; Fy = Fy - a * v; Fz = Fz - a * w;
  }
  m.u = u; m.v = v; m.w = w;
  const R hx = Fx * hi, hy = Fy * hi, hz = Fz * hi;
  m.xx = m.xx + (hx + hx) * u;
  m.yy = m.yy + (hy + hy) * v;
  m.zz = m.zz + (hz + hz) * w;
  m.xy = m.xy + (hy * u + hx * v);
  m.xz = m.xz + (hz * u + hx * w);
  m.yz = m.yz + (hz * v + hy * w);
  if (dens) {
    const R pxx = m.xx - u * u, pyy = m.yy - v * v, pzz = m.zz - w * w;
    const R pxy = m.xy - u * v, pxz = m.xz - u * w, pyz = m.yz - v * w;
    tFx = tFx - kv * (pxx * gfx + pxy * gfy + pxz * gfz);
    tFy = tFy - kv * (pyy * gfy + pxy * gfx + pyz * gfz);
    tFz = tFz - kv * (pzz * gfz + pxz * gfx + pyz * gfy);
  }
}

// ---------------------------------------------------------------------------
// Post-collision Hermite coefficients of one node on the tensor-product D3Q27
// basis, A[a + 3b + 9c] scaled by 1/2 for every index a, b, c >= 1 (a power of
// two: exact).  With that scaling the 1-D reconstruction (recon3) needs no
// factor on its first- and second-order inputs.  E_k and N_k of fused:668-702
// (k = 10..26, N_k as written there), grouped by common factors: with
// X1 = u/2, X2 = u^2/2 (Y, Z alike), q_ab the equally scaled (1-omega) Pn_ab
// (q_xx = (1-omega) Pn_xx / 2, q_xy = (1-omega) Pn_xy / 4) the orders 3..6
// take 62 multiply-adds where term by term they take about 150.
// Coefficients that are zero for !HO are not written.
template <bool HO, class R>
__device__ __forceinline__ void hermite27(const NodeIn<R>& n, R (&A)[27]) {
#define AI(a, b, c) A[(a) + 3 * (b) + 9 * (c)]
  const R om1 = (R)1 - n.om, oh = (R)0.5 * om1, oq = (R)0.25 * om1;
  const R u = n.u, v = n.v, w = n.w;
  const R X1 = (R)0.5 * u, Y1 = (R)0.5 * v, Z1 = (R)0.5 * w;
  const R X2 = u * X1, Y2 = v * Y1, Z2 = w * Z1;
  const R qxx = oh * n.xx, qyy = oh * n.yy, qzz = oh * n.zz;
  const R qxy = oq * n.xy, qxz = oq * n.xz, qyz = oq * n.yz;
  const R ax4 = (R)0.25 * n.ax, ay4 = (R)0.25 * n.ay, az4 = (R)0.25 * n.az;
  AI(0, 0, 0) = n.P;
  AI(1, 0, 0) = X1 + ax4; AI(0, 1, 0) = Y1 + ay4; AI(0, 0, 1) = Z1 + az4;
  AI(2, 0, 0) = X1 * (u + n.ax) + qxx; AI(0, 2, 0) = Y1 * (v + n.ay) + qyy; AI(0, 0, 2) = Z1 * (w + n.az) + qzz;
  AI(1, 1, 0) = X1 * AI(0, 1, 0) + (Y1 * ax4 + qxy);
  AI(1, 0, 1) = X1 * AI(0, 0, 1) + (Z1 * ax4 + qxz);
  AI(0, 1, 1) = Y1 * AI(0, 0, 1) + (Z1 * ay4 + qyz);
  if constexpr (HO) {
    const R exx = X2 + qxx, eyy = Y2 + qyy, ezz = Z2 + qzz;
    const R dxx = (R)2 * qxx, dyy = (R)2 * qyy, dxy = (R)2 * qxy, dxz = (R)2 * qxz, dyz = (R)2 * qyz;
    const R uxy = u * dxy, uxz = u * dxz, vxy = v * dxy, vyz = v * dyz, wxz = w * dxz, wyz = w * dyz;
    const R XY = X1 * Y1, XZ = X1 * Z1, YZ = Y1 * Z1, w3 = (R)3 * w;
    AI(2, 1, 0) = Y1 * exx + uxy; AI(2, 0, 1) = Z1 * exx + uxz;
    AI(1, 2, 0) = X1 * eyy + vxy; AI(1, 0, 2) = X1 * ezz + wxz;
    AI(0, 1, 2) = Y1 * ezz + wyz; AI(0, 2, 1) = Z1 * eyy + vyz;
    const R rz = X1 * qyz + Y1 * qxz;
    AI(1, 1, 1) = Z1 * (XY + qxy) + rz;
    AI(1, 1, 2) = XY * ezz + (w3 * rz + dxy * Z2);
    const R vuxy = v * uxy, ydx = Y2 * dxx;
    AI(2, 2, 0) = X2 * eyy + ((R)3 * vuxy + ydx);
    AI(2, 0, 2) = X2 * ezz + (w3 * uxz + Z2 * dxx);
    AI(0, 2, 2) = Y2 * ezz + (w3 * vyz + Z2 * dyy);
    const R my = X2 * qyz + Y1 * uxz, nx = X1 * vyz + Y2 * qxz;
    AI(2, 1, 1) = YZ * (X2 + dxx) + (w * uxy + my);
    AI(1, 2, 1) = XZ * (Y2 + dyy) + (w * vxy + nx);
    AI(2, 1, 2) = (X2 * Y1) * ezz + w3 * (qxx * YZ + (Z1 * uxy + my));
    AI(1, 2, 2) = (X1 * Y2) * ezz + w3 * (qyy * XZ + (Z1 * vxy + nx));
    const R l = X2 * vyz + Y2 * uxz;
    AI(2, 2, 1) = Z1 * (X2 * (Y2 + dyy) + ((R)5 * vuxy + (R)1.5 * ydx)) + l;
    AI(2, 2, 2) = (X2 * Y2) * ezz + (w3 * l + Z2 * (((R)1.5 * dyy) * X2 + ((R)7 * vuxy + (R)2 * ydx)));
  }
#undef AI
}

// Post-collision populations f[cidx(p,q,r)] of one node (the open-boundary
// closure's regularised populations; the D3Q19 collision of the fused kernel).
template <int LAT, bool HO, class R>
__device__ __forceinline__ void collide(const NodeIn<R>& n, R* f) {
  if constexpr (LAT == 27) {
    R A[27];
#pragma unroll
    for (int k = 0; k < 27; ++k) A[k] = 0;
    hermite27<HO, R>(n, A);
    // x pass: A[a][b][c] -> B[p][b][c]
    R B[27];
#pragma unroll
    for (int bc = 0; bc < 9; ++bc) recon3(A[3 * bc + 0], A[3 * bc + 1], A[3 * bc + 2], B[3 * bc + 0], B[3 * bc + 1], B[3 * bc + 2]);
    // y pass: B[p][b][c] -> A[p][q][c]
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int pp = 0; pp < 3; ++pp)
        recon3(B[pp + 0 + 9 * c], B[pp + 3 + 9 * c], B[pp + 6 + 9 * c], A[pp + 0 + 9 * c], A[pp + 3 + 9 * c], A[pp + 6 + 9 * c]);
    // z pass: A[p][q][c] -> f[p][q][r]
#pragma unroll
    for (int pq = 0; pq < 9; ++pq) recon3(A[pq], A[pq + 9], A[pq + 18], f[pq], f[pq + 9], f[pq + 18]);
  } else {
    const R om1 = (R)1 - n.om;
    const R u = n.u, v = n.v, w = n.w;
    // order <= 2 Hermite coefficients (post-collision, with half forcing)
    const R A000 = n.P;
    const R A100 = u + (R)0.5 * n.ax, A010 = v + (R)0.5 * n.ay, A001 = w + (R)0.5 * n.az;
    const R A200 = u * u + om1 * n.xx + u * n.ax;
    const R A020 = v * v + om1 * n.yy + v * n.ay;
    const R A002 = w * w + om1 * n.zz + w * n.az;
    const R A110 = u * v + om1 * n.xy + (R)0.5 * (u * n.ay + v * n.ax);
    const R A101 = u * w + om1 * n.xz + (R)0.5 * (u * n.az + w * n.ax);
    const R A011 = v * w + om1 * n.yz + (R)0.5 * (v * n.az + w * n.ay);
    // D3Q19: f_l = w_l [A0 + 3 c.A1 + 4.5 sum_ab (c_a c_b - delta/3) A2_ab]
#pragma unroll
    for (int r = -1; r <= 1; ++r)
#pragma unroll
      for (int q = -1; q <= 1; ++q)
#pragma unroll
        for (int p = -1; p <= 1; ++p) {
          const int c = cidx(p, q, r);
          if (!present<LAT>(p, q, r)) { f[c] = 0; continue; }
          const R wl = (R)weight<LAT>(p, q, r);
          R s = A000;
          if (p) s += (R)(3 * p) * A100;
          if (q) s += (R)(3 * q) * A010;
          if (r) s += (R)(3 * r) * A001;
          s += (R)(4.5 * (p * p - 1.0 / 3.0)) * A200;
          s += (R)(4.5 * (q * q - 1.0 / 3.0)) * A020;
          s += (R)(4.5 * (r * r - 1.0 / 3.0)) * A002;
          if (p * q) s += (R)(9 * p * q) * A110;
          if (p * r) s += (R)(9 * p * r) * A101;
          if (q * r) s += (R)(9 * q * r) * A011;
          f[c] = wl * s;
        }
  }
}

// relaxation rate of the fused / LB_int_boundary kernels: omega, or
// 1/(3 nu(phi) + 1/2) with nu(phi) the density-weighted viscosity mix;
// under SMAGORINSKI (fused:198-210, 603-616; boundary:145-160)
//   tau = 1/2 + (3 nu + sqrt((3 nu)^2 + C sqrt(2 Q) / rho_phi)) / 6,
// Q = Pneq:Pneq, C = 0.053*18.0 evaluated in single precision as the
// reference's default-real literals are.
template <bool TWO, class R, bool STD = false>
__device__ __forceinline__ R relax_rate(const DevParams& dp, const NodeRates<R>& nr, R pxx, R pyy, R pzz, R pxy,
                                        R pxz, R pyz) {
  if (!STD && dp.smag) {
    const R QQ = pxx * pxx + pyy * pyy + pzz * pzz + (R)2 * (pxy * pxy + pxz * pxz + pyz * pyz);
    const R C = (R)(0.053f * 18.0f);
    const R t3 = (R)3 * nr.visc;
    return rcp((R)0.5 + (R)(1.0 / 6.0) * ((R)3 * nr.visc + sqrt(t3 * t3 + C * sqrt((R)2 * QQ) * nr.irho)));
  }
  return nr.om0;
}

}  // namespace lbf
