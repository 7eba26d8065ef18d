// mds_gravity.h -- GR effective monopole gravity (gravity.c:142-375 with
// GR_MONOPOLE, no radiation: the radiation pressure, energy and v.F shell
// terms are zero), evaluated by one workgroup per problem.
//
// Input: the volume-weighted shell sums of rho, P, u and v^1 in the
// problem's GR block (DevProb::gr, MDS_GR_* arrays of n1 + 1 doubles), and
// the host-made shell geometry (face radius, (4 pi) r^3, dr/dx, shell
// volume).  Output: the zone-centred field gz[0..n1), the TOV factor Gamma
// and mass at the faces (Gamma is kept: the next call starts from it), and
// the lapses exp(phi / c^2) at the faces and zone centres.
//
// Steps, in the reference's order and operation order:
//   averages  sum * (1 / V_shell)                           (gravity.c:277-287)
//   Gamma     first call: the Newtonian estimate             (gravity.c:292-301)
//             passes over the faces ii = 1..n1 until the outer TOV mass moves
//             by less than 1e-10 (at most 21 passes)       (gravity.c:303-336)
//   g         face gravity with the pressure and inertia terms (gravity.c:339-346)
//   lapse     potential integrated inwards from -G M / r_out (gravity.c:349-352)
//   zone      g and the potential linear in x across each zone at the volume
//             centroid beta/Gamma; lapses exponentiated     (gravity.c:355-375)
// The pass over the faces is a recurrence (Gamma at face ii needs the mass
// below it, and that the Gammas below), lower triangular and weakly coupled:
// a mass enters Gamma only through 2 G m / (r c^2).  One thread walking it
// was the whole cost of the field (two passes of 640 faces, some 0.4 us a
// face).  The workgroup solves it a tile of one face per thread at a time
// instead: the mass is a prefix sum of the current Gammas, Gamma follows
// from it, and the two alternate until no face moves by more than two units
// in the last place, which takes a few rounds (a round makes at least one
// more face final, so NT rounds end it whatever the state is).  24 columns
// of 640 zones with the table EOS: 591 us a call before, 26 us now.
#pragma once
#include "mds_internal.h"

#define MDS_GR_MAXPASS 20

namespace gr {

constexpr double GNEWT = 6.67384e-8;       // constants.h
constexpr double CLIGHT = 2.99792458e10;   // constants.h:10

__device__ __forceinline__ double *arr(const DevProb &pb, int k) { return pb.gr + (size_t)k * (pb.n[0] + 1); }

// zone moments beta and Gamma of radial zone i (ghost zones included)
__device__ __forceinline__ double mom_be(const DevProb &pb, int i) { return pb.mom[0][3 * (i + MDS_NG) + 1]; }
__device__ __forceinline__ double mom_ga(const DevProb &pb, int i) { return pb.mom[0][3 * (i + MDS_NG) + 2]; }

// DPP move of a double: lanes without a source keep 0
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_or_zero(double v)
{
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffll), CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// inclusive sums over the lanes of a wavefront (row shifts by 1, 2, 4, 8,
// then the last lane of each row of 16 and of the first half to those above)
__device__ __forceinline__ double wave_scan(double v)
{
  v += dpp_or_zero<0x111, 0xf>(v);
  v += dpp_or_zero<0x112, 0xf>(v);
  v += dpp_or_zero<0x114, 0xf>(v);
  v += dpp_or_zero<0x118, 0xf>(v);
  v += dpp_or_zero<0x142, 0xa>(v);
  v += dpp_or_zero<0x143, 0xc>(v);
  return v;
}

// Sums over the threads of a workgroup below this one, the total in `sum`.
// One barrier: the callers alternate `par`, so a slow wavefront still reads
// one half of the totals while the next call fills the other.
template <int NT>
__device__ __forceinline__ double block_scan(double v, double &sum, double (&tot)[2][NT / 64], int par)
{
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const double s = wave_scan(v);
  if (lane == 63) tot[par][w] = s;
  __syncthreads();
  double below = 0.0;
  sum = 0.0;
#pragma unroll
  for (int k = 0; k < NT / 64; k++) {
    if (k == w) below = sum;
    sum += tot[par][k];
  }
  return below + (s - v);
}

}  // namespace gr

// The field of one problem from its shell sums (see above); NT threads.
template <int NT>
__device__ void gr_monopole_block(const DevProb &pb, double *gz)
{
  using namespace gr;
  const int n1 = pb.n[0];
  const int tid = threadIdx.x;
  const double c2 = CLIGHT * CLIGHT;
  const double dx = pb.dx[0];
  double *redge = arr(pb, MDS_GR_REDGE), *r34 = arr(pb, MDS_GR_R34), *drdx = arr(pb, MDS_GR_DRDX);
  double *vsh = arr(pb, MDS_GR_VSH), *gtov = arr(pb, MDS_GR_GTOV), *mr = arr(pb, MDS_GR_MR);
  double *le = arr(pb, MDS_GR_LAPSE_E), *lc = arr(pb, MDS_GR_LAPSE), *gf = arr(pb, MDS_GR_GFACE);
  double *rho = arr(pb, MDS_GR_RHO), *pg = arr(pb, MDS_GR_P), *uu = arr(pb, MDS_GR_U), *vv = arr(pb, MDS_GR_V);

  // volume averages over the exact shell volume
  for (int i = tid; i < n1; i += NT) {
    const double iv = 1.0 / vsh[i];
    rho[i] *= iv;
    pg[i] *= iv;
    uu[i] *= iv;
    vv[i] *= iv;
  }
  __syncthreads();

  __shared__ double s_tot[2][NT / 64];
  __shared__ int s_moved[2][NT / 64];
  const int lane = tid & 63, wv = tid >> 6;
  int par = 0;                          // alternates with every block_scan
  // M_star = sum V rho, and on the first call Gamma from the Newtonian mass
  // (gravity.c:292-301)
  const bool first = !pb.grst[0];
  double mstar = 0.0;
  for (int base = 1; base <= n1; base += NT) {
    const int ii = base + tid;
    const double v = ii <= n1 ? vsh[ii - 1] * rho[ii - 1] : 0.0;
    double sum;
    const double below = block_scan<NT>(v, sum, s_tot, par);
    par ^= 1;
    if (first && ii <= n1) gtov[ii] = sqrt(1.0 - ((2.0 * GNEWT) * (mstar + (below + v))) / (c2 * redge[ii]));
    mstar += sum;
  }
  __syncthreads();                      // every thread has read grst[0]
  if (tid == 0) {
    mr[0] = 0.0;
    if (first) {
      gtov[0] = 1.0;
      pb.grst[0] = 1;
    }
  }
  __syncthreads();

  // Gamma at the centroid of the zone above face ii is gl + (g - gl) th from
  // the Gammas gl, g of the faces ii - 1 and ii, so the mass at face ii is
  //   m_ii = sum_{q <= ii} a_q g_{q-1} + b_q g_q,  a = V w (1 - th), b = V w th
  auto shell = [&](int ii, double &a, double &b) {
    const double xl = pb.startx[0] + ii * dx;
    const double th = (mom_be(pb, ii) / mom_ga(pb, ii) - xl) / dx;
    const double vw = vsh[ii - 1] * (rho[ii - 1] + uu[ii - 1] / c2);
    a = vw * (1.0 - th);
    b = vw * th;
  };
  double mlast = 0.0;
  int iter = 0;
  while (true) {
    double gp = gtov[0], mp = 0.0;        // Gamma and mass at the face below the tile
    for (int base = 1; base <= n1; base += NT) {
      const int ii = base + tid;
      const bool live = ii <= n1;
      double a = 0.0, b = 0.0, an = 0.0, bn, go = 0.0, vq = 1.0, kq = 0.0, g = 0.0;
      if (live) {
        shell(ii, a, b);
        if (ii < n1) shell(ii + 1, an, bn);
        go = gtov[ii];
        const double ve = (ii < n1) ? 0.5 * (vv[ii - 1] + vv[ii]) : vv[ii - 1];
        const double vc = ve / CLIGHT;
        vq = 1.0 + vc * vc;
        kq = (2.0 * GNEWT) / (redge[ii] * c2);
        g = go;
      }
      // the first face's share of the Gamma below the tile
      double ab;
      {
        double bb;
        shell(base, ab, bb);
      }
      const double mb = mp + ab * gp;
      const double e = b + an;            // g_ii's share of the masses above face ii
      bool moved = true;
      double m = 0.0;
      for (int round = 0; round <= NT; round++) {
        const unsigned long long any = __ballot(moved);
        if (lane == 0) s_moved[par][wv] = any != 0;
        double sum;
        const double t = mb + block_scan<NT>(e * g, sum, s_tot, par);
        int go_on = 0;
#pragma unroll
        for (int k = 0; k < NT / 64; k++) go_on |= s_moved[par][k];
        par ^= 1;
        m = t + b * g;
        if (!go_on) break;
        const double gn = live ? sqrt(vq - kq * (t + b * go)) : 0.0;
        moved = !(fabs(gn - g) <= 4.5e-16 * fabs(gn));
        g = gn;
      }
      if (live) {
        gtov[ii] = g;
        mr[ii] = m;
      }
      __syncthreads();
      const int last = min(base + NT - 1, n1);
      gp = gtov[last];
      mp = mr[last];
    }
    int done = 0;
    if (iter > 0 && fabs(mlast - mp) / mp < 1.0e-10) done = 1;
    if (!done) {
      mlast = mp;
      iter++;
      if (iter > MDS_GR_MAXPASS) {
        done = 1;
        if (tid == 0) pb.grst[2] += 1;    // did not converge: the reference exits here
      }
    }
    if (done) break;
  }
  if (tid == 0) pb.grst[1] = iter;

  // face gravity with the pressure and inertia terms (gravity.c:339-346)
  for (int ii = tid; ii <= n1; ii += NT) {
    double g = 0.0;
    if (ii > 0) {
      const int a = ii - 1, b = ii < n1 ? ii : ii - 1;
      const double pe = ii < n1 ? 0.5 * (pg[a] + pg[b]) : pg[a];
      const double re = ii < n1 ? 0.5 * (rho[a] + rho[b]) : rho[a];
      const double ue = ii < n1 ? 0.5 * (uu[a] + uu[b]) : uu[a];
      const double rg = redge[ii] * gtov[ii];
      g = ((((-GNEWT * (mr[ii] + (r34[ii] * (pe + 0.0)) / c2)) / (rg * rg)) * (re + (ue + pe) / c2)) / re) * drdx[ii];
    }
    gf[ii] = g;
  }
  __syncthreads();

  // the potential, integrated inwards from -G M_star / r_out: sums from the
  // top, a tile of NT faces at a time
  double lp = (-GNEWT * mstar) / redge[n1];
  if (tid == 0) le[n1] = lp;
  for (int top = n1 - 1; top >= 0; top -= NT) {
    const int ii = top - tid;
    const double v = ii >= 0 ? (0.5 * (gf[ii] + gf[ii + 1])) * dx : 0.0;
    double sum;
    const double below = block_scan<NT>(v, sum, s_tot, par);
    par ^= 1;
    if (ii >= 0) le[ii] = lp + (below + v);
    lp += sum;
  }
  __syncthreads();

  // zone values: g and the potential at the volume centroid, then the lapses
  for (int i = tid; i < n1; i += NT) {
    const double xl = pb.startx[0] + i * dx;
    const double be = mom_be(pb, i), ga = mom_ga(pb, i);
    double A = (gf[i + 1] - gf[i]) / dx;
    double B = gf[i] - A * xl;
    gz[i] = (A * be) / ga + B;
    A = (le[i + 1] - le[i]) / dx;
    B = le[i] - A * xl;
    lc[i] = exp(((A * be) / ga + B) / c2);
  }
  __syncthreads();
  for (int i = tid; i <= n1; i += NT) le[i] = exp(le[i] / c2);
}
