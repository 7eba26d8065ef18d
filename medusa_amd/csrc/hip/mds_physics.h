// mds_physics.h -- pointwise device physics of the hydro sweep (gfx950).
//
// Two families:
//   *_x64  FP64, the reference's operation order (reconstruct.c:127-213,
//          riemann.c:4-62,178-499, fluid.c:4-53, rad_fluid.c:164-192,
//          step.c:205-223).  Built with -ffp-contract=off so that every
//          product and sum rounds exactly as in the reference CPU build.
//   *_f32  FP32-bulk: the same algorithms in single precision with the
//          well-conditioned local reconstruction (MDS_RC_* coefficients),
//          hardware reciprocal / square root, FMA contraction within an
//          expression: contract(on), by which the source decides what is
//          fused and every launch shape gives the same bits.  contract(fast)
//          leaves it to each kernel's own instruction selection (1% faster:
//          RT 256^3 1.90 ms a step against 1.92, KH 2048^2 211 us against
//          213), and 3D boxes then differed between the tile shapes.
//
// Velocity components beyond NV are identically zero and skipped; every
// skipped term is an exact +-0 contribution in the reference arithmetic.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define MDS_DEV __device__ __forceinline__

// ---------------------------------------------------------------------------
// geometry of one face as seen by a Riemann solve: area, scale[1+dir][dir],
// gcov[1+dir][0..2].  CART: unit metric, so every multiply/divide by scale or
// gcov is the identity and is dropped at compile time.
template <class R>
struct FaceGeo {
  R area;
  R scale;
  R gcov[3];
};

template <class R, int NV>
struct PState {          // reconstructed primitive state on one side of a face
  R rho, uu, v[3], P, G;
  R ye;                  // passive scalar (electron fraction), used when NS = 1
};

// slot of the passive scalar in conserved/flux records (decs.h:646: YE after U3)
#define MDS_YI 5

// field-wise select of one of two states
template <class R, int NV>
__device__ __forceinline__ PState<R, NV> pick_state(bool first, const PState<R, NV> &a, const PState<R, NV> &b)
{
  PState<R, NV> k;
  k.rho = first ? a.rho : b.rho;
  k.uu = first ? a.uu : b.uu;
  for (int d = 0; d < 3; d++) k.v[d] = first ? a.v[d] : b.v[d];
  k.P = first ? a.P : b.P;
  k.G = first ? a.G : b.G;
  k.ye = first ? a.ye : b.ye;
  return k;
}

template <class R, int NV>
struct Flux {
  R f[5];                // rho, E, m1..m3 (area weighted)
};

// ---------------------------------------------------------------------------
// FP64 quotients and roots
//
// The FP64 kernels are bound by vector issue, and a compiled division is 11
// instructions: two scalings for operands near the ends of the exponent
// range, the reciprocal (hardware estimate, two Newton steps), the quotient,
// its residual correction, and the fix-up of zeros, infinities and NaN.  The
// scalings only matter where an exponent leaves some +-960 or a quotient
// falls below the normal range, which no state of these units does, and the
// reciprocal belongs to the denominator alone.  Here the steps are separate,
// so that one reciprocal serves every quotient of its denominator (4
// instructions each); inside that range the bits are the compiled
// division's.  With the limiter's two cases and the two sides of the contact
// evaluated once on selected operands, KH 777 x 1003 went from 374 to 318 us
// a step, RT 150 x 122 x 203 from 3.63 to 3.07 ms, 40 columns from 19.5 to
// 17.2 us, the 160 x 32 x 64 star from 630 to 593 us, with the same bits.
// ---------------------------------------------------------------------------
MDS_DEV double drcp(double x)
{
  double r = __builtin_amdgcn_rcp(x);
  double e = __builtin_fma(-x, r, 1.0);
  r = __builtin_fma(r, e, r);
  e = __builtin_fma(-x, r, 1.0);
  return __builtin_fma(r, e, r);
}
// a / b with y = drcp(b)
MDS_DEV double div_y(double a, double b, double y)
{
  double q = a * y;
  q = __builtin_fma(__builtin_fma(-b, q, a), y, q);
  return __builtin_amdgcn_div_fixup(q, b, a);
}
MDS_DEV double div_x64(double a, double b) { return div_y(a, b, drcp(b)); }

// sqrt(x): the hardware's reciprocal root, one coupled Newton step for the
// root and half its reciprocal and two residual corrections (correctly
// rounded), without the compiled root's scaling of arguments below 2^-767
MDS_DEV double sqrt_x64(double x)
{
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, r, g);
  h = __builtin_fma(h, r, h);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  return (x == 0.0 || x == __builtin_huge_val()) ? x : g;
}

// ---------------------------------------------------------------------------
// FP64, reference operation order
// ---------------------------------------------------------------------------

// para_recon for one zone (reconstruct.c:142-201).  am, a0, ap: zone means;
// al_m..: volume moments alpha/beta/Gamma of zones i-1, i, i+1; xlo, xhi:
// faces of zone i.  den and den2 depend on the geometry only; the reference
// recomputes them per variable with identical operands, so hoisting them is
// bit-exact.
struct ReconGeo64 {
  double am, a0, ap;     // alpha
  double bm, b0, bp;     // beta
  double gm, g0, gp;     // Gamma
  double xlo, xhi;
  double den, den2;
  double y0;             // drcp(Gamma_0)
  int order = 3;         // hydro_interp_order: 3 para_recon, 2 lin_recon, 1 piecewise constant
};

__host__ MDS_DEV void recon_geo_x64(ReconGeo64 &g)
{
  double t012 = (g.am * g.b0) * g.gp;
  double t021 = (g.am * g.bp) * g.g0;
  double t102 = (g.a0 * g.bm) * g.gp;
  double t120 = (g.a0 * g.bp) * g.gm;
  double t201 = (g.ap * g.bm) * g.g0;
  double t210 = (g.ap * g.b0) * g.gm;
  g.den = 1.0 / (((((t012 + t120) + t201) - t021) - t102) - t210);
  double d2 = (g.xlo - g.xhi) * ((g.a0 + ((g.g0 * g.xlo) * g.xhi)) - (g.b0 * (g.xlo + g.xhi)));
  g.den2 = 1.0 / d2;
}

MDS_DEV void para_recon_x64(double qm, double q0, double qp, const ReconGeo64 &g,
                            double &al, double &ar)
{
  double dqm = q0 - qm;
  double dqp = qp - q0;
  if (dqm * dqp <= 0.0) { al = q0; ar = q0; return; }
  double dqc = qp - qm;
  double A = ((((dqm * g.bp) * g.gm) * g.g0) + g.gp * (((dqp * g.bm) * g.g0) - ((dqc * g.b0) * g.gm))) * g.den;
  double B = (-((((dqm * g.ap) * g.gm) * g.g0) + g.gp * (((dqp * g.am) * g.g0) - ((dqc * g.a0) * g.gm)))) * g.den;
  double C = q0 - div_y((g.a0 * A) + (g.b0 * B), g.g0, g.y0);
  double l = g.xlo * ((A * g.xlo) + B) + C;
  double r = g.xhi * ((A * g.xhi) + B) + C;
  double mean = (0.75 * qm) + (0.25 * q0);
  if (((q0 - l) * (l - mean)) < 0.0) l = mean;
  mean = (0.75 * qp) + (0.25 * q0);
  if (((mean - r) * (r - q0)) < 0.0) r = mean;
  double A2 = ((g.b0 * (r - l)) + g.g0 * (((q0 * (g.xlo - g.xhi)) - (r * g.xlo)) + (l * g.xhi))) * g.den2;
  double B2 = (((g.a0 * (l - r)) + ((g.g0 * (r - q0)) * (g.xlo * g.xlo))) + ((g.g0 * (q0 - l)) * (g.xhi * g.xhi))) * g.den2;
  double xz = div_x64(-B2, (2.0 * A2) + 1.0e-16);
  if (!__builtin_isfinite(xz)) xz = -1.0e-200;
  double xmid = 0.5 * (g.xlo + g.xhi);
  if (xz > g.xlo && xz < g.xhi) {
    // the extremum moves to the nearer face x, whose value f stays; the other
    // face (X) follows.  One evaluation for both cases, on selected operands.
    const bool up = xz > xmid;
    const double f = up ? r : l, x = up ? g.xhi : g.xlo, X = up ? g.xlo : g.xhi;
    const double A3 = div_x64(g.g0 * (q0 - f), g.a0 + (x * ((g.g0 * x) - (2.0 * g.b0))));
    const double B3 = (-2.0 * A3) * x;
    const double C3 = q0 - div_y((g.a0 * A3) + (g.b0 * B3), g.g0, g.y0);
    const double n = X * ((A3 * X) + B3) + C3;
    l = up ? n : l;
    r = up ? r : n;
  }
  al = l;
  ar = r;
}

// lin_recon for one zone (reconstruct.c:89-124): a limited linear profile
// through the zone's centroid x0 = beta/Gamma, the slope the smallest of the
// one-sided slopes to the neighbours' centroid-face midpoints and the centred
// slope; flat at a local extremum
MDS_DEV void lin_recon_x64(double qm, double q0, double qp, const ReconGeo64 &g, double &al, double &ar)
{
  const double xm = g.bm / g.gm;
  const double xp = g.bp / g.gp;
  const double x0 = g.b0 / g.g0;
  const double sm = (q0 - qm) / (x0 - (0.5 * (g.xlo + xm)));
  const double sp = (qp - q0) / ((0.5 * (g.xhi + xp)) - x0);
  if (sm * sp <= 0.0) { al = q0; ar = q0; return; }
  const double sc = (qp - qm) / (xp - xm);
  const double asm_ = fabs(sm), asp = fabs(sp), asc = fabs(sc);
  const double m1 = asm_ < asp ? asm_ : asp;                // MIN of decs.h:627, NaN order included
  const double A = (sc < 0.0 ? -1.0 : 1.0) * (m1 < asc ? m1 : asc);
  const double B = q0 - ((A * g.b0) / g.g0);
  al = (A * g.xlo) + B;
  ar = (A * g.xhi) + B;
}

// the reconstruction of hydro_interp_order (reconstruct.c:246-266): every
// zone of a launch shares the order, so the branch is uniform
MDS_DEV void recon_x64(double qm, double q0, double qp, const ReconGeo64 &g, double &al, double &ar)
{
  if (g.order == 3) para_recon_x64(qm, q0, qp, g, al, ar);
  else if (g.order == 2) lin_recon_x64(qm, q0, qp, g, al, ar);
  else { al = q0; ar = q0; }
}

// The quotients of Gamma alone in the wave-speed estimate, for a gamma law
// (G_l = G_r = G, so G_avg is G itself).  One set per launch, in scalar
// registers: a quotient of the same operands has the same bits wherever it
// is formed, so the faces' results do not change.
struct GamF64 {
  double ravg;  // (G - 1) / (2 G)
  double pex;   // (2 G) / (G - 1)
  double bgm;   // (G - 1) / (G + 1)
  double kq;    // (G + 1) / (2 G)
};
MDS_DEV double uniform_f64(double x)
{
  const long long v = __double_as_longlong(x);
  const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)v);
  const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(v >> 32));
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
MDS_DEV GamF64 gam_f64_uniform(double G)
{
  GamF64 k;
  k.ravg = uniform_f64((G - 1.0) / (2.0 * G));
  k.pex = uniform_f64((2.0 * G) / (G - 1.0));
  k.bgm = uniform_f64((G - 1.0) / (G + 1.0));
  k.kq = uniform_f64((G + 1.0) / (2.0 * G));
  return k;
}

// wave-speed estimate shared by HLLC/HLLE (riemann.c:210-303, 368-429);
// UNIG: G_l = G_r, with its quotients in *gk (a gamma law)
template <bool HLLC_FLOOR, bool UNIG = false>
MDS_DEV void wave_speeds_x64(double rl, double rr, double p_l, double p_r, double G_l, double G_r,
                             double u_l, double u_r, double cs_l, double cs_r,
                             double &sl, double &sr, double &ss, double &p_s, int &isshock,
                             const GamF64 *gk = nullptr)
{
  double p_max, p_min;
  if (p_l > p_r) { p_max = p_l; p_min = p_r; } else { p_max = p_r; p_min = p_l; }
  // pratio < 2 and (p_max - p_min) / p_min > 1/2 without the quotients: a
  // quotient of doubles rounds to the other side of 2 (or 1/2) only from
  // closer than a double can be to twice (half) another, so the products
  // decide alike; a negative p_min (an unphysical state) makes the first
  // quotient at most 1 and the second at most 0
  const bool neg = p_min < 0.0;
  const bool near = neg || p_max < 2.0 * p_min;
  isshock = (!neg && p_max - p_min > 0.5 * p_min) ? 1 : 0;
  p_s = (0.5 * (p_l + p_r)) - (((0.125 * (u_r - u_l)) * (rl + rr)) * (cs_l + cs_r));
  if (HLLC_FLOOR) p_s = (0 > p_s) ? 0.0 : p_s;
  else p_s = (p_s > 0.0) ? p_s : 0.0;
  if (near && p_s >= p_min && p_s <= p_max) {
  } else if (p_s < p_min) {
    double G_avg = 0.5 * (G_l + G_r);
    const double yl = drcp(cs_l), yr = drcp(cs_r);
    double plr = pow(div_x64(p_l, p_r), UNIG ? gk->ravg : div_x64(G_avg - 1.0, 2.0 * G_avg));
    double s0 = div_x64((div_y(plr * u_l, cs_l, yl) + div_y(u_r, cs_r, yr)) + div_x64(2.0 * (plr - 1.0), G_avg - 1.0),
                        div_y(plr, cs_l, yl) + div_y(1.0, cs_r, yr));
    const double el = UNIG ? gk->pex : div_x64(2.0 * G_l, G_l - 1.0);
    const double er = UNIG ? gk->pex : div_x64(2.0 * G_r, G_r - 1.0);
    p_s = 0.5 * ((p_l * pow(1.0 + (div_x64(G_l - 1.0, 2.0 * cs_l) * (u_l - s0)), el))
                 + (p_r * pow(1.0 + (div_x64(G_r - 1.0, 2.0 * cs_r) * (s0 - u_r)), er)));
    p_s = (p_s > 0.0) ? p_s : 0.0;
  } else {
    double a_l = div_x64(2.0, (G_l + 1.0) * rl);
    double a_r = div_x64(2.0, (G_r + 1.0) * rr);
    double b_l = (UNIG ? gk->bgm : div_x64(G_l - 1.0, G_l + 1.0)) * p_l;
    double b_r = (UNIG ? gk->bgm : div_x64(G_r - 1.0, G_r + 1.0)) * p_r;
    double g_l = sqrt_x64(div_x64(a_l, p_s + b_l));
    double g_r = sqrt_x64(div_x64(a_r, p_s + b_r));
    p_s = div_x64(((g_l * p_l) + (g_r * p_r)) - (u_r - u_l), g_l + g_r);
    p_s = (p_s > 0.0) ? p_s : 0.0;
  }
  double q_l = 1.0, q_r = 1.0;
  if (!(p_s <= p_l)) q_l = sqrt_x64(1.0 + ((UNIG ? gk->kq : div_x64(G_l + 1.0, 2.0 * G_l)) * (div_x64(p_s, p_l) - 1.0)));
  if (!(p_s <= p_r)) q_r = sqrt_x64(1.0 + ((UNIG ? gk->kq : div_x64(G_r + 1.0, 2.0 * G_r)) * (div_x64(p_s, p_r) - 1.0)));
  sl = u_l - (cs_l * q_l);
  sr = u_r + (cs_r * q_r);
  ss = div_x64(((p_r - p_l) + ((rl * u_l) * (sl - u_l))) - ((rr * u_r) * (sr - u_r)),
               (rl * (sl - u_l)) - (rr * (sr - u_r)));
}

// conserved state and physical flux of one side (riemann.c:4-37)
template <int NV, bool CART, int NS = 0>
MDS_DEV void p_uflux_x64(const PState<double, NV> &p, const FaceGeo<double> &g, int dir,
                         double u[6], double f[6])
{
  double vcov[3];
  for (int d = 0; d < NV; d++) vcov[d] = CART ? p.v[d] : g.gcov[d] * p.v[d];
  double v = p.v[dir];
  u[0] = p.rho;
  double vsq = 0.0;
  for (int d = 0; d < NV; d++) vsq += p.v[d] * vcov[d];
  double etot = ((0.5 * u[0]) * vsq) + p.uu;
  u[1] = etot;
  for (int d = 0; d < NV; d++) u[2 + d] = u[0] * vcov[d];
  if (NS) u[MDS_YI] = u[0] * p.ye;
  f[0] = u[0] * v;
  f[1] = v * (etot + p.P);
  for (int d = 0; d < NV; d++) f[2 + d] = f[0] * vcov[d];
  f[2 + dir] += p.P;
  if (NS) f[MDS_YI] = f[0] * p.ye;
}

// area-weighted physical flux (riemann.c:39-62)
template <int NV, bool CART, int NS = 0>
MDS_DEV void pflux_x64(const PState<double, NV> &p, const FaceGeo<double> &g, int dir, double f[6])
{
  double vcov[3];
  for (int d = 0; d < NV; d++) vcov[d] = CART ? p.v[d] : g.gcov[d] * p.v[d];
  double v = p.v[dir];
  f[0] = (g.area * p.rho) * v;
  for (int d = 0; d < NV; d++) f[2 + d] = f[0] * vcov[d];
  f[2 + dir] += g.area * p.P;
  double vsq = 0.0;
  for (int d = 0; d < NV; d++) vsq += p.v[d] * vcov[d];
  double etot = ((0.5 * p.rho) * vsq) + p.uu;
  f[1] = (g.area * v) * (etot + p.P);
  if (NS) f[MDS_YI] = f[0] * p.ye;
}

// HLLC (riemann.c:328-499).  Returns isshock.
template <int NV, bool CART, int NS = 0, bool UNIG = false>
MDS_DEV int hllc_x64(const PState<double, NV> &L, const PState<double, NV> &Rt,
                     const FaceGeo<double> &g, int dir, double flux[6], double &sig, const GamF64 *gk = nullptr)
{
  if (g.area < 1.0e-16) {
    sig = 1.0e-200;
    for (int q = 0; q < 2 + NV; q++) flux[q] = 0.0;
    if (NS) flux[MDS_YI] = 0.0;
    return 0;
  }
  double u_l = CART ? L.v[dir] : L.v[dir] * g.scale;
  double u_r = CART ? Rt.v[dir] : Rt.v[dir] * g.scale;
  double cs_l = sqrt_x64(div_x64(L.G * L.P, L.rho));
  double cs_r = sqrt_x64(div_x64(Rt.G * Rt.P, Rt.rho));
  double sl, sr, ss, p_s;
  int isshock;
  wave_speeds_x64<true, UNIG>(L.rho, Rt.rho, L.P, Rt.P, L.G, Rt.G, u_l, u_r, cs_l, cs_r, sl, sr, ss, p_s, isshock, gk);
  if (ss > sr) sr = 1.001 * ss;
  if (ss < sl) sl = 1.001 * ss;
  const double ysc = CART ? 1.0 : drcp(g.scale);
  double smax = (fabs(sl) > fabs(sr)) ? fabs(sl) : fabs(sr);
  sig = CART ? smax : div_y(smax, g.scale, ysc);
  if (sl > 0.0) { pflux_x64<NV, CART, NS>(L, g, dir, flux); return isshock; }
  if (sr < 0.0) { pflux_x64<NV, CART, NS>(Rt, g, dir, flux); return isshock; }
  double u[6], fx[6], Us[6], vs[3];
  // the side upwind of the contact, selected by value (a reference to one of
  // two locals would force both into scratch memory).  The right side's star
  // energy has its numerator and denominator negated in the reference
  // (riemann.c:470-480), which leaves every rounding and the quotient alike,
  // so one evaluation serves both sides.
  const bool left = ss > 0.0;
  const PState<double, NV> K = pick_state(left, L, Rt);
  const double sk = left ? sl : sr, uk = left ? u_l : u_r;
  const double den = sk - ss, yden = drcp(den);
  p_uflux_x64<NV, CART, NS>(K, g, dir, u, fx);
  Us[0] = div_y(K.rho * (sk - uk), den, yden);
  Us[1] = div_y(((u[1] * (sk - uk)) - (K.P * uk)) + (p_s * ss), den, yden);
  const double slr = CART ? sk : div_y(sk, g.scale, ysc);
  for (int d = 0; d < NV; d++) vs[d] = K.v[d];
  vs[dir] = CART ? ss : div_y(ss, g.scale, ysc);
  for (int d = 0; d < NV; d++) Us[2 + d] = (CART ? vs[d] : g.gcov[d] * vs[d]) * Us[0];
  if (NS) Us[MDS_YI] = Us[0] * K.ye;
  for (int q = 0; q < 2 + NV; q++) flux[q] = g.area * (fx[q] + (slr * (Us[q] - u[q])));
  if (NS) flux[MDS_YI] = g.area * (fx[MDS_YI] + (slr * (Us[MDS_YI] - u[MDS_YI])));
  return isshock;
}

// HLLE (riemann.c:178-325)
template <int NV, bool CART, int NS = 0, bool UNIG = false>
MDS_DEV void hlle_x64(const PState<double, NV> &L, const PState<double, NV> &Rt,
                      const FaceGeo<double> &g, int dir, double flux[6], double &sig, const GamF64 *gk = nullptr)
{
  if (g.area < 1.0e-16) {
    sig = 1.0e-200;
    for (int q = 0; q < 2 + NV; q++) flux[q] = 0.0;
    if (NS) flux[MDS_YI] = 0.0;
    return;
  }
  double u_l = CART ? L.v[dir] : L.v[dir] * g.scale;
  double u_r = CART ? Rt.v[dir] : Rt.v[dir] * g.scale;
  double cs_l = sqrt_x64(div_x64(L.G * L.P, L.rho));
  double cs_r = sqrt_x64(div_x64(Rt.G * Rt.P, Rt.rho));
  double sl, sr, ss, p_s;
  int isshock;
  wave_speeds_x64<false, UNIG>(L.rho, Rt.rho, L.P, Rt.P, L.G, Rt.G, u_l, u_r, cs_l, cs_r, sl, sr, ss, p_s, isshock, gk);
  double ul[6], ur[6], fl[6], fr[6];
  p_uflux_x64<NV, CART, NS>(L, g, dir, ul, fl);
  p_uflux_x64<NV, CART, NS>(Rt, g, dir, ur, fr);
  const double ysc = CART ? 1.0 : drcp(g.scale);
  double srs = CART ? sr : div_y(sr, g.scale, ysc);
  double sls = CART ? sl : div_y(sl, g.scale, ysc);
  double cmax = (srs > 0.0) ? srs : 0.0;
  double cmin = fabs((sls < 0.0) ? sls : 0.0);
  sig = (cmax > cmin) ? cmax : cmin;
  const double den = cmax + cmin, yden = drcp(den);
  for (int q = 0; q < 2 + NV; q++)
    flux[q] = div_y(g.area * (((cmin * fr[q]) + (cmax * fl[q])) - ((cmax * cmin) * (ur[q] - ul[q]))), den, yden);
  if (NS) {
    const int q = MDS_YI;
    flux[q] = div_y(g.area * (((cmin * fr[q]) + (cmax * fl[q])) - ((cmax * cmin) * (ur[q] - ul[q]))), den, yden);
  }
}

// fluid.c:4-25
template <int NV, bool CART>
MDS_DEV void p_to_u_x64(double rho, double uu, const double v[3], const double gcov[3], double u[5])
{
  double vcov[3];
  for (int d = 0; d < NV; d++) vcov[d] = CART ? v[d] : gcov[d] * v[d];
  u[0] = rho;
  double vsq = 0.0;
  for (int d = 0; d < NV; d++) {
    vsq += v[d] * vcov[d];
    u[2 + d] = u[0] * vcov[d];
  }
  u[1] = ((0.5 * u[0]) * vsq) + uu;
}

// fluid.c:27-53 (no floors)
template <int NV, bool CART>
MDS_DEV void u_to_p_x64(double u[5], const double gcon[3], double &rho, double &uu, double v[3])
{
  rho = u[0];
  const double y = drcp(u[0]);
  for (int d = 0; d < NV; d++) u[2 + d] = div_y(u[2 + d], u[0], y);
  for (int d = 0; d < NV; d++) v[d] = CART ? u[2 + d] : gcon[d] * u[2 + d];
  double vsq = 0.0;
  for (int d = 0; d < NV; d++) vsq += u[2 + d] * v[d];
  uu = u[1] - ((0.5 * rho) * vsq);
}

// step.c:205-223
template <int NV>
MDS_DEV double dt_source_control_x64(double uu, const double v[3], const double u[5], const double s[5])
{
  const double alpha = 0.02;
  double mdt = 1.0e100;
  double local_dt = div_x64(alpha * u[0], fabs(s[0]) + 1.0e-16);
  mdt = (mdt < local_dt) ? mdt : local_dt;
  local_dt = div_x64(alpha * u[1], fabs(s[1]) + 1.0e-16);
  mdt = (mdt < local_dt) ? mdt : local_dt;
  double momterm = 0.0;
  for (int d = 0; d < NV; d++) momterm += v[d] * s[2 + d];
  local_dt = div_x64(2.0 * uu, fabs(fabs(s[1]) - fabs(momterm)) + 1.0e-16);
  mdt = (mdt < local_dt) ? mdt : local_dt;
  return mdt;
}

// dt_source_control with reciprocals instead of divisions (FP32-bulk path,
// where the limit only needs to be close to the reference value)
template <int NV>
MDS_DEV double dt_source_control_fast(double uu, const double v[3], const double u[5], const double s[5]);

// ---------------------------------------------------------------------------
// FP32-bulk
// ---------------------------------------------------------------------------
struct ReconGeo32 {
  float clm, clp, crm, crp, mu1, kinv, inur, imu2;
};

MDS_DEV float frcp(float x) { return __builtin_amdgcn_rcpf(x); }
// hardware square root and reciprocal square root (v_sqrt_f32, v_rsq_f32,
// about 1 ulp): the FP32-bulk path needs no correctly rounded result, and the
// IEEE sequence costs some 16 VALU instructions per call.  Their arguments
// must stay in the FP32 normal range: the hardware flushes denormal inputs.
MDS_DEV float fsqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
MDS_DEV float frsqrt(float x) { return __builtin_amdgcn_rsqf(x); }
// x^y for x > 0 as 2^(y log2 x) (v_log_f32, v_exp_f32): three instructions
// instead of the library powf's range reduction; the relative error grows to
// a few 1e-7 for |y log2 x| near 10, within what FP32 storage already makes
MDS_DEV float fpow(float x, float y) { return __builtin_amdgcn_exp2f(y * __builtin_amdgcn_logf(x)); }

// para_recon in local coordinates: the same limiter, on the face values'
// offsets L, R from the zone mean.  With the parabola's slopes d0 = b1 and
// d1 = b1 + 2 b2 at the faces and D = R - L at the middle, its extremum lies
// inside the zone where d0 d1 < 0, in the upper half where d0 D > 0: no
// reciprocal, and 34 instructions against the 45 slots of the form that
// located it.  The FP32 kernels are bound by vector issue: with the shorter
// star pressure and star flux below, KH 2048^2 went from 282 to 248 us a step,
// RT 256^3 from 2.28 to 1.98 ms.  Against 64-bit runs the errors are what they
// were (KH 1.09e-7 -> 1.06e-7, tubes 1.31e-7 -> 1.23e-7, all variables).
MDS_DEV void para_recon_f32(float qm, float q0, float qp, const ReconGeo32 &g, float &al, float &ar)
{
#pragma clang fp contract(on)
  const float dqm = q0 - qm;
  const float dqp = qp - q0;
  // a local extremum or a uniform stretch, where whole wavefronts skip the rest
  if (dqm * dqp <= 0.0f) { al = q0; ar = q0; return; }
  float L = g.clm * dqm + g.clp * dqp;
  float R = g.crm * dqm + g.crp * dqp;
  // outside the span of the zone mean and 3/4 of the step to the neighbour
  if (L * (L + 0.75f * dqm) > 0.0f) L = -0.75f * dqm;
  if (R * (R - 0.75f * dqp) > 0.0f) R = 0.75f * dqp;
  const float D = R - L;
  const float b2 = (-L - D * g.mu1) * g.kinv;
  const float d0 = D - b2, d1 = D + b2;
  const bool in = d0 * d1 < 0.0f, up = d0 * D > 0.0f;
  const float Ln = R - R * g.inur, Rn = L - L * g.imu2;
  if (in && up) L = Ln;
  if (in && !up) R = Rn;
  al = q0 + L;
  ar = q0 + R;
}

// Gamma-only factors of the FP32 wave-speed estimate.  A gamma law needs one
// set per launch: gam_f32_uniform makes it once and keeps it in scalar
// registers, and the shock and rarefaction branches then take no reciprocal
// of Gamma per face.
struct GamF32 {
  float ravg;  // (G - 1) rcp(2 G): exponent of the two-rarefaction pressure ratio
  float hgm1;  // (G - 1) / 2
  float pex;   // 2 G rcp(G - 1): power of the two-rarefaction star pressure
  float bgm;   // (G - 1) rcp(G + 1): the two-shock b / p
  float sgp1;  // sqrt((G + 1) / 2): the two-shock velocity scale
  float kq;    // (G + 1) rcp(2 G): the shock factor's slope
};
MDS_DEV float uniform_f32(float x) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x))); }
MDS_DEV GamF32 gam_f32_uniform(float G)
{
  GamF32 k;
  k.ravg = uniform_f32((G - 1.0f) * frcp(2.0f * G));
  k.hgm1 = uniform_f32((G - 1.0f) * 0.5f);
  k.pex = uniform_f32(2.0f * G * frcp(G - 1.0f));
  k.bgm = uniform_f32((G - 1.0f) * frcp(G + 1.0f));
  k.sgp1 = uniform_f32(fsqrt(0.5f * (G + 1.0f)));
  k.kq = uniform_f32((G + 1.0f) * frcp(2.0f * G));
  return k;
}

// both precisions' sets for a gamma law (a kernel uses the one it needs)
struct GamSet {
  GamF32 f32;
  GamF64 f64;
};
MDS_DEV GamSet gam_set_uniform(double G)
{
  GamSet k;
  k.f32 = gam_f32_uniform((float)G);
  k.f64 = gam_f64_uniform(G);
  return k;
}

// EAGER: both pressure reciprocals up front, serving the rarefactions and
// both shock factors (faster where shock factors are common, as on Cartesian
// boxes); otherwise the shock factors divide only where a wavefront needs them.
// UNIG: G_l = G_r, with its factors in *gk (a gamma law).  rs_l, rs_r:
// rsqrt(rho), which the sound speeds have formed already.
template <bool EAGER = false, bool UNIG = false>
MDS_DEV void wave_speeds_f32(float rl, float rr, float p_l, float p_r, float G_l, float G_r,
                             float u_l, float u_r, float cs_l, float cs_r, float rs_l, float rs_r,
                             float &sl, float &sr, float &ss, float &p_s, int &isshock,
                             const GamF32 *gk = nullptr)
{
#pragma clang fp contract(on)
  const float p_max = fmaxf(p_l, p_r), p_min = fminf(p_l, p_r);
  const float du = u_r - u_l;
  float ipl = 0.0f, ipr = 0.0f;
  if constexpr (EAGER) {
    ipl = frcp(p_l);
    ipr = frcp(p_r);
  }
  isshock = (p_max - p_min > 0.5f * p_min) ? 1 : 0;
  p_s = 0.5f * (p_l + p_r) - 0.125f * du * (rl + rr) * (cs_l + cs_r);
  p_s = fmaxf(p_s, 0.0f);
  if (p_max < 2.0f * p_min && p_s >= p_min && p_s <= p_max) {
  } else if (p_s < p_min) {
    const float plr = fpow(p_l * (EAGER ? ipr : frcp(p_r)),
                           UNIG ? gk->ravg : (0.5f * (G_l + G_r) - 1.0f) * frcp(G_l + G_r));
    if constexpr (UNIG) {
      // both sides' star pressures in one: with one Gamma the left and the
      // right isentrope meet at p_l [(c_l + c_r - h du) / (c_l + c_r plr)]^pex,
      // which is what their mean is; the bracket as one less its distance
      // from one, which the power would multiply the rounding of
      p_s = p_l * fpow(1.0f - (gk->hgm1 * du + cs_r * (plr - 1.0f)) * frcp(cs_l + cs_r * plr), gk->pex);
    } else {
      const float icl = frcp(cs_l), icr = frcp(cs_r);
      const float igm1 = frcp(0.5f * (G_l + G_r) - 1.0f);
      const float s0 = (plr * u_l * icl + u_r * icr + 2.0f * (plr - 1.0f) * igm1) * frcp(plr * icl + icr);
      const float hl = (G_l - 1.0f) * 0.5f, hr = (G_r - 1.0f) * 0.5f;
      const float el = 2.0f * G_l * frcp(G_l - 1.0f), er = 2.0f * G_r * frcp(G_r - 1.0f);
      p_s = 0.5f * (p_l * fpow(1.0f + hl * icl * (u_l - s0), el) + p_r * fpow(1.0f + hr * icr * (s0 - u_r), er));
    }
    p_s = fmaxf(p_s, 0.0f);
  } else {
    // the two-shock weights sqrt(2 / ((G + 1) rho) / (p_s + b)) as products of
    // reciprocal roots: the quotient itself falls below the FP32 normal range
    // at stellar-core densities and pressures, where the hardware roots flush
    // it to zero.  With one Gamma their common sqrt(2 / (G + 1)) moves to du.
    const float b_l = (UNIG ? gk->bgm : (G_l - 1.0f) * frcp(G_l + 1.0f)) * p_l;
    const float b_r = (UNIG ? gk->bgm : (G_r - 1.0f) * frcp(G_r + 1.0f)) * p_r;
    float g_l = rs_l * frsqrt(p_s + b_l);
    float g_r = rs_r * frsqrt(p_s + b_r);
    float dv = du;
    if constexpr (UNIG) {
      dv = du * gk->sgp1;
    } else {
      g_l *= frsqrt(0.5f * (G_l + 1.0f));
      g_r *= frsqrt(0.5f * (G_r + 1.0f));
    }
    p_s = (g_l * p_l + g_r * p_r - dv) * frcp(g_l + g_r);
    p_s = fmaxf(p_s, 0.0f);
  }
  const float kl = UNIG ? gk->kq : (G_l + 1.0f) * frcp(2.0f * G_l);
  const float kr = UNIG ? gk->kq : (G_r + 1.0f) * frcp(2.0f * G_r);
  float q_l = (p_s <= p_l) ? 1.0f : fsqrt(1.0f + kl * (p_s * (EAGER ? ipl : frcp(p_l)) - 1.0f));
  float q_r = (p_s <= p_r) ? 1.0f : fsqrt(1.0f + kr * (p_s * (EAGER ? ipr : frcp(p_r)) - 1.0f));
  // the waves' speeds against the gas and the mass fluxes through them
  const float w_l = cs_l * q_l, w_r = cs_r * q_r;
  const float m_l = rl * w_l, m_r = rr * w_r;
  sl = u_l - w_l;
  sr = u_r + w_r;
  ss = (p_l - p_r + u_l * m_l + u_r * m_r) * frcp(m_l + m_r);
}

// Conserved state and per-unit-area physical flux of one side in FP32 (the
// FP64 caller applies the FP64 area).
template <int NV, bool CART, int NS = 0>
MDS_DEV void p_uflux_f32(const PState<float, NV> &p, const FaceGeo<float> &g, int dir, float u[6], float f[6])
{
#pragma clang fp contract(on)
  float vcov[3];
  for (int d = 0; d < NV; d++) vcov[d] = CART ? p.v[d] : g.gcov[d] * p.v[d];
  float v = p.v[dir];
  u[0] = p.rho;
  float vsq = 0.0f;
  for (int d = 0; d < NV; d++) vsq += p.v[d] * vcov[d];
  float etot = 0.5f * p.rho * vsq + p.uu;
  u[1] = etot;
  for (int d = 0; d < NV; d++) u[2 + d] = p.rho * vcov[d];
  f[0] = p.rho * v;
  f[1] = v * (etot + p.P);
  for (int d = 0; d < NV; d++) f[2 + d] = f[0] * vcov[d];
  f[2 + dir] += p.P;
  if (NS) { u[MDS_YI] = p.rho * p.ye; f[MDS_YI] = f[0] * p.ye; }
}

// HLLC in FP32; flux per unit area.  Returns isshock.  UNIG: a gamma law,
// whose wave-speed factors *gk carries.
template <int NV, bool CART, int NS = 0, bool UNIG = false>
MDS_DEV int hllc_f32(const PState<float, NV> &L, const PState<float, NV> &Rt,
                     const FaceGeo<float> &g, int dir, float flux[6], float &sig, const GamF32 *gk = nullptr)
{
#pragma clang fp contract(on)
  float u_l = CART ? L.v[dir] : L.v[dir] * g.scale;
  float u_r = CART ? Rt.v[dir] : Rt.v[dir] * g.scale;
  const float rs_l = frsqrt(L.rho), rs_r = frsqrt(Rt.rho);
  float cs_l = fsqrt(L.G * L.P) * rs_l;
  float cs_r = fsqrt(Rt.G * Rt.P) * rs_r;
  float sl, sr, ss, p_s;
  int isshock;
  wave_speeds_f32<CART, UNIG>(L.rho, Rt.rho, L.P, Rt.P, L.G, Rt.G, u_l, u_r, cs_l, cs_r, rs_l, rs_r, sl, sr, ss, p_s,
                              isshock, gk);
  if (ss > sr) sr = 1.001f * ss;
  if (ss < sl) sl = 1.001f * ss;
  float iscale = CART ? 1.0f : frcp(g.scale);
  sig = fmaxf(fabsf(sl), fabsf(sr)) * iscale;
  // One evaluation for every face, no divergent exits: the physical flux of
  // the upwind state (the left state where sl > 0, the right where sr < 0,
  // else the side of the contact), plus the star-state term where neither
  // wave is supersonic (riemann.c:437-495).  The term is selected, not
  // weighted, so an undefined star state of a supersonic face stays out.
  // The transverse velocities (and Ye) do not change across the waves, so
  // their fluxes are the mass flux times the upwind value.
  const bool sup_l = sl > 0.0f, sup_r = sr < 0.0f, star = !(sup_l || sup_r);
  const bool left = sup_l || (!sup_r && ss > 0.0f);
  const PState<float, NV> K = pick_state(left, L, Rt);
  const float sk = left ? sl : sr, uk = left ? u_l : u_r;
  float vcov[3], vsq = 0.0f;
  for (int d = 0; d < NV; d++) {
    vcov[d] = CART ? K.v[d] : g.gcov[d] * K.v[d];
    vsq += K.v[d] * vcov[d];
  }
  const float vn = K.v[dir], etot = 0.5f * K.rho * vsq + K.uu;
  const float iden = frcp(sk - ss);
  // the star state's differences from the upwind state, which vanish exactly
  // where the gas rests: formed as rho (sk - uk) / (sk - ss) less rho, the
  // rounding of the reciprocal was a mass flux of eps rho c in uniform gas,
  // and spherical columns drifted by it
  const float rel = (ss - uk) * iden;
  const float dr = K.rho * rel;
  const float de = etot * rel + (p_s * ss - K.P * uk) * iden;
  const float slr = sk * iscale, vs = ss * iscale;
  const float f0 = K.rho * vn, f1 = vn * (etot + K.P), fn = f0 * vcov[dir] + K.P;
  const float dm = K.rho * (vs - vn) + vs * dr;
  flux[0] = star ? f0 + slr * dr : f0;
  flux[1] = star ? f1 + slr * de : f1;
  flux[2 + dir] = star ? fn + slr * (CART ? dm : g.gcov[dir] * dm) : fn;
  for (int d = 0; d < NV; d++)
    if (d != dir) flux[2 + d] = flux[0] * vcov[d];
  if (NS) flux[MDS_YI] = flux[0] * K.ye;
  return isshock;
}

template <int NV, bool CART, int NS = 0, bool UNIG = false>
MDS_DEV void hlle_f32(const PState<float, NV> &L, const PState<float, NV> &Rt,
                      const FaceGeo<float> &g, int dir, float flux[6], float &sig, const GamF32 *gk = nullptr)
{
#pragma clang fp contract(on)
  float u_l = CART ? L.v[dir] : L.v[dir] * g.scale;
  float u_r = CART ? Rt.v[dir] : Rt.v[dir] * g.scale;
  const float rs_l = frsqrt(L.rho), rs_r = frsqrt(Rt.rho);
  float cs_l = fsqrt(L.G * L.P) * rs_l;
  float cs_r = fsqrt(Rt.G * Rt.P) * rs_r;
  float sl, sr, ss, p_s;
  int isshock;
  wave_speeds_f32<CART, UNIG>(L.rho, Rt.rho, L.P, Rt.P, L.G, Rt.G, u_l, u_r, cs_l, cs_r, rs_l, rs_r, sl, sr, ss, p_s,
                              isshock, gk);
  float ul[6], ur[6], fl[6], fr[6];
  p_uflux_f32<NV, CART, NS>(L, g, dir, ul, fl);
  p_uflux_f32<NV, CART, NS>(Rt, g, dir, ur, fr);
  float iscale = CART ? 1.0f : frcp(g.scale);
  float cmax = fmaxf(sr * iscale, 0.0f);
  float cmin = fabsf(fminf(sl * iscale, 0.0f));
  sig = fmaxf(cmax, cmin);
  float iden = frcp(cmax + cmin);
  for (int q = 0; q < 2 + NV; q++) flux[q] = (cmin * fr[q] + cmax * fl[q] - cmax * cmin * (ur[q] - ul[q])) * iden;
  if (NS) {
    const int q = MDS_YI;
    flux[q] = (cmin * fr[q] + cmax * fl[q] - cmax * cmin * (ur[q] - ul[q])) * iden;
  }
}

// ---------------------------------------------------------------------------
// helpers
// ---------------------------------------------------------------------------
// positive double -> order-preserving 64-bit key for atomicMin
MDS_DEV unsigned long long dt_key(double v) { return (unsigned long long)__double_as_longlong(v); }

// Running minimum keys shared by a whole launch.  One same-address atomic per
// wavefront serializes at the L2 and can cost more than the kernel's own
// work, so a wavefront reads the current minimum (device-coherent load, the
// L2 copy) when it starts and goes on only if its value beats it; then it
// reads it again, since all wavefronts of a launch's first round have seen
// the minimum as the step's reset left it, and by the time they finish most
// of them no longer improve on it (the first stage of the 320 x 64 x 128 star
// spent 125 of its 560 us in those atomics; a step went from 1190 to 994 us,
// the 160 x 32 x 64 star's in FP64 from 587 to 467, KH 2048^2 from 245 to
// 220).  A stale read is larger than the true
// minimum, so no needed update is lost.
MDS_DEV unsigned long long min_key_seen(unsigned long long *p)
{
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
MDS_DEV void fold_min_key(unsigned long long *p, unsigned long long seen, double v)
{
  const unsigned long long k = dt_key(v);
  if (k < seen && k < min_key_seen(p)) atomicMin(p, k);
}

// Device health: lanes of the wavefront whose new state is unphysical --
// a non-finite or non-positive density, a non-finite internal energy, and
// with the gamma law a negative one (negative pressure).  Call with every
// lane of the wavefront active; returns the wave-uniform count.
MDS_DEV unsigned bad_state_lanes(bool valid, double rho, double uu, bool gamma_law)
{
  const double inf = __builtin_huge_val();
  const bool ok = (rho > 0.0) && (rho < inf) && (uu > -inf) && (uu < inf) && (!gamma_law || uu >= 0.0);
  return (unsigned)__popcll(__ballot(valid && !ok));
}

// Cross-lane neighbours with whole-wave DPP shifts (GFX9 wave_shr:1 /
// wave_shl:1): lane l reads lane l-1 (from_below) or l+1 (from_above); the
// edge lane keeps its own value.  Must be called with every lane active.
MDS_DEV int dpp_shr1(int v) { return __builtin_amdgcn_update_dpp(v, v, 0x138, 0xf, 0xf, false); }
MDS_DEV int dpp_shl1(int v) { return __builtin_amdgcn_update_dpp(v, v, 0x130, 0xf, 0xf, false); }
MDS_DEV float lane_from_below(float v) { return __int_as_float(dpp_shr1(__float_as_int(v))); }
MDS_DEV float lane_from_above(float v) { return __int_as_float(dpp_shl1(__float_as_int(v))); }
MDS_DEV int lane_from_below(int v) { return dpp_shr1(v); }
MDS_DEV int lane_from_above(int v) { return dpp_shl1(v); }
MDS_DEV double lane_from_below(double v)
{
  long long b = __double_as_longlong(v);
  int lo = dpp_shr1((int)(b & 0xffffffffll)), hi = dpp_shr1((int)(b >> 32));
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
MDS_DEV double lane_from_above(double v)
{
  long long b = __double_as_longlong(v);
  int lo = dpp_shl1((int)(b & 0xffffffffll)), hi = dpp_shl1((int)(b >> 32));
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

MDS_DEV double wave_max(double v)
{
  for (int off = 32; off > 0; off >>= 1) {
    double o = __shfl_xor(v, off, 64);
    v = (o > v) ? o : v;
  }
  return v;
}

MDS_DEV double wave_min(double v)
{
  for (int off = 32; off > 0; off >>= 1) {
    double o = __shfl_xor(v, off, 64);
    v = (o < v) ? o : v;
  }
  return v;
}

// The FP32-bulk source limit: hardware reciprocal estimates (v_rcp_f64, no
// Newton steps).  The limit bounds dt; a relative error near 1e-8 in it is
// far below what FP32 state storage already changes.
template <int NV>
MDS_DEV double dt_source_control_fast(double uu, const double v[3], const double u[5], const double s[5])
{
  double mdt = (0.02 * u[0]) * __builtin_amdgcn_rcp(fabs(s[0]) + 1.0e-16);
  double t = (0.02 * u[1]) * __builtin_amdgcn_rcp(fabs(s[1]) + 1.0e-16);
  mdt = fmin(mdt, t);
  double momterm = 0.0;
  for (int d = 0; d < NV; d++) momterm += v[d] * s[2 + d];
  t = (2.0 * uu) * __builtin_amdgcn_rcp(fabs(fabs(s[1]) - fabs(momterm)) + 1.0e-16);
  return fmin(mdt, t);
}
