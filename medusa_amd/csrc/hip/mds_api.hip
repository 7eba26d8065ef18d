// mds_api.hip -- C-ABI of the hydro sweep: context, device residency, the
// device-side dt policy, hipGraph replay, compensated totals and the
// pointwise parity entry points.  See include/mds_hydro.h.
#include <hip/hip_runtime.h>
#include <stdio.h>
#include <string.h>
#include <stdarg.h>
#include <stdlib.h>
#include <vector>
#include <atomic>
#include <new>
#include <algorithm>
#include "mds_internal.h"
#include "mds_physics.h"
#include "mds_clock.h"
#include "../common/mds_stage.h"
#include "mds_eos.h"
#include "../../../include/mds_eos.h"
#include "../common/mds_mp.h"


extern "C" hipError_t mds_launch_sweep1d(int fp32, int nv, int sph, int tab, int mono, const Sweep1DArgs *a,
                                         const void *sp, const void *sph_, int stage, hipStream_t st);
extern "C" hipError_t mds_launch_slab_fill(int fp32, const DevProb *probs, int nprob, long long items,
                                           void *const *state, const DevEos *eos, int tab, int nv, hipStream_t st);
extern "C" hipError_t mds_launch_monopole(int fp32, int mono, int tab, int nprob, int nmax, const DevProb *prob,
                                          const DevClock *clock, const DevEos *eos, const void *st, double *grav,
                                          hipStream_t s);
hipError_t mds_eos_to_device(const mds_eos_table *t, DevEos *d, void **alloc);
extern "C" hipError_t mds_launch_sph3d(const Sph3Launch *L, const DevProb *pb, DevClock *clock,
                                       unsigned long long *counters, const DevEos *eos, const void *sp,
                                       const void *sph, int stage, hipStream_t st);
extern "C" hipError_t mds_launch_sweep2d(int fp32, int nv, const Sweep2DArgs *a, const void *sp,
                                         const void *sph, int stage, hipStream_t st);
extern "C" hipError_t mds_launch_sweep3d(int fp32, int ty, int hshare, const Sweep3DArgs *a, const void *sp,
                                         const void *sph, int stage, hipStream_t st);

struct mds_ctx {
  int precision = 0;
  int nprob = 0;
  int ndim = 1;
  int nv = 1;
  int sph = 0;
  long long nzone = 0;
  RunParams rp{};
  double tmax = 0.0;
  hipStream_t st = nullptr;
  // host copies
  std::vector<DevProb> hprob;
  std::vector<long long> zstart;        // prefix sums of interior zones (nprob+1)
  std::vector<int> nvars;
  // device
  void *p[6] = {nullptr}, *ph[6] = {nullptr};    // rho, u, v1..v3, Ye (Ye with a table EOS)
  int nstate = 5;                  // state arrays per copy (6 with a table EOS)
  int tab = 0;                     // tabulated EOS (Ye carried)
  DevEos deos{};
  void *eos_alloc = nullptr;
  int mono = 0;                    // monopole gravity (MDS_MONOPOLE_NEWTON or MDS_MONOPOLE_GR)
  double *dgrav = nullptr;         // monopole field at zone centres (FP64), packed like the state
  double *dgr = nullptr;           // GR: every problem's block of MDS_GR_COUNT x (n1 + 1) doubles
  size_t gr_doubles = 0;
  int *dgrst = nullptr;            // GR: 4 ints of state per problem
  int sph3 = 0;                    // 3D spherical grid (direction-split stage)
  Sph3Launch s3{};                 // its work buffers
  DevProb *dprob = nullptr;
  DevClock *dclock = nullptr;
  DevClock *dclock2 = nullptr;     // 1D two-stage: second clocks and running minima of folded steps (mds_clock.h)
  unsigned long long *dmind = nullptr;
  int2 *dseg = nullptr;            // 1D segment table of the single-stage kernels
  int nseg = 0;
  int2 *dseg2 = nullptr;           // 1D segment table of the two-stage kernel
  int nseg2 = 0;
  int2 *dseg3 = nullptr;           // the same for two zones per lane (FP32-bulk)
  int nseg3 = 0;
  int nmax1d = 0;                  // 1D: zones of the largest column
  int can_fuse1d = 0;              // 1D and no problem periodic in x
  int fuse1d = 0;                  // use the two-stage 1D kernel (p -> ph, then swap); 2: two zones per lane
  int par = 0;                     // buffer parity: which allocation p currently names
  unsigned char *dflags = nullptr;
  unsigned long long *dcount = nullptr;
  long long *dzstart = nullptr;
  std::vector<void *> geo_allocs;
  int chunk2d = 24;
  int ty3d = 4;
  int ncu = 0;                          // compute units of the device
  int dev = 0;                          // the device the context was created on
  int grid1d = 0;                       // 1D grid: 0 one wavefront per segment, 1 persistent
  int halo3d = 0;                       // 3D: 1 = the output wavefronts also load the halo rows
  int kc3d = 16;
  int has_slab = 0;                     // some problem has a PROB or EXTRAP side
  long long slab_items = 0;             // most ghost zones of PROB/EXTRAP sides in one problem
  std::vector<int> prob_pending;        // per problem: PROB sides whose values were never set
  // time-dependent PROB hooks (mds_set_prob_bounds_t), per problem, and
  // pinned host staging of their values per side and stage
  std::vector<mds_prob_bounds_t_fn> tdep_fn;
  std::vector<void *> tdep_user;
  std::vector<double *> tdep_buf;                 // [prob][3 dirs][2 sides][2 stages], or null
  int ntdep = 0;
  std::vector<int> hdj, hdk;            // dendritic grid: dj and dk with ghosts (the grid's layout)
  // one step, per buffer parity, then groups of folded steps, per parity
  hipGraph_t graph[4] = {nullptr, nullptr, nullptr, nullptr};
  hipGraphExec_t gexec[4] = {nullptr, nullptr, nullptr, nullptr};
  // pinned staging of the state's way back, two halves of MDS_PIN_BYTES, made
  // by the first download
  char *pin = nullptr;
  long long pin_half = 0;
  hipEvent_t pin_ev[2] = {nullptr, nullptr};
  char err[512] = {0};
};

static void drop_graphs(mds_ctx *c)
{
  for (int k = 0; k < 4; k++) {
    if (c->gexec[k]) { hipGraphExecDestroy(c->gexec[k]); c->gexec[k] = nullptr; }
    if (c->graph[k]) { hipGraphDestroy(c->graph[k]); c->graph[k] = nullptr; }
  }
}

static int set_err(mds_ctx *c, int code, const char *fmt, ...)
{
  if (c) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(c->err, sizeof(c->err), fmt, ap);
    va_end(ap);
  }
  return code;
}

#define HIPCHK(ctx, call)                                                              \
  do {                                                                                 \
    hipError_t e_ = (call);                                                            \
    if (e_ != hipSuccess)                                                              \
      return set_err((ctx), MDS_EDEVICE, "%s failed: %s", #call, hipGetErrorString(e_)); \
  } while (0)

// ---------------------------------------------------------------------------
// small device kernels
// ---------------------------------------------------------------------------

// the dt policy (mds_clock.h), one thread per problem
__global__ void dt_policy_kernel(DevClock *ck, int nprob, RunParams rp)
{
  int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= nprob) return;
  DevClock c = ck[p];
  if (dt_policy(c, __longlong_as_double((long long)c.mindt), rp)) c.mindt = dt_key(1.0e100);   // step() resets min_dt (step.c:49)
  ck[p] = c;
}

// first estimate_dt zone bound from the initial state (main.c:181 then step.c:177-187)
template <class R>
__global__ void init_dt_kernel(const DevProb *prob, DevClock *ck, const long long *zstart, int nprob,
                               StateArrays<R> sp, int tab, DevEos eos)
{
  long long z = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  bool live = z < zstart[nprob];
  if (!live) z = zstart[nprob] - 1;       // keep every lane active for the wave reduction
  int lo = 0, hi = nprob - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (zstart[mid] <= z) lo = mid; else hi = mid - 1;
  }
  const DevProb &pb = prob[lo];
  long long q = z - zstart[lo];
  double rho = sp.v[0][pb.off + q], uu = sp.v[1][pb.off + q];
  double cs;
  if (tab) {
    double press, gam1, lt;
    eos_fill_x64(eos, rho, uu, (double)sp.v[5][pb.off + q], press, gam1, cs, lt);
  } else {
    double press = (pb.gam - 1.0) * uu;
    cs = sqrt((pb.gam * press) / rho);
  }
  int i = (int)(q % pb.n[0]);
  int j = (int)((q / pb.n[0]) % pb.n[1]);
  const int kz = (int)(q / ((long long)pb.n[0] * pb.n[1]));
  double loc = 0.0;
  for (int d = 0; d < pb.ndim; d++) {
    double sc = 1.0;
    if (pb.sph && pb.ndim >= 2)
      sc = pb.zone[(size_t)(MDS_ZS_SCALE0 + d) * (pb.n[0] + 2 * MDS_NG) * (pb.n[1] + 2 * MDS_NG)
                   + (size_t)(j + MDS_NG) * (pb.n[0] + 2 * MDS_NG) + (i + MDS_NG)];
    else if (pb.sph && d == 0) sc = pb.zone[(size_t)(i + MDS_NG) * MDS_ZG_COUNT + MDS_ZG_SCALE0];
    double v = sp.v[2 + d][pb.off + q];
    double ldx = pb.dx[d];                                  // DJS / DKS widths (step.c:179-181)
    if (pb.lj && d == 1) ldx *= (double)(1 << dend_lj(pb, i));
    if (pb.lj && d == 2 && dend_valid(pb, i, j, 0)) ldx *= (double)(1 << dend_lk(pb, i, j));
    loc += (fabs(v) + (cs / sc)) / ldx;
  }
  double b = 1.0 / loc;
  if (pb.lj && !dend_valid(pb, i, j, kz)) b = 1.0e300;
  // one atomic per wavefront when the whole wavefront belongs to one problem
  int p0 = __shfl(lo, 0, 64);
  if (__all(lo == p0)) {
    double m = wave_min(b);
    if ((threadIdx.x & 63) == 0) fold_min_key(&ck[lo].mindt, min_key_seen(&ck[lo].mindt), m);
  } else {
    atomicMin(&ck[lo].mindt, dt_key(b));
  }
}

// Neumaier-compensated block partials of rho*V and E*V over one problem.
template <class R>
__global__ void totals_kernel(const DevProb *prob, int p, long long nz, int nv, StateArrays<R> sp,
                              double *partial)
{
  const DevProb &pb = prob[p];
  double s[2] = {0.0, 0.0}, cmp[2] = {0.0, 0.0};
  for (long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x; q < nz;
       q += (long long)gridDim.x * blockDim.x) {
    double rho = sp.v[0][pb.off + q], uu = sp.v[1][pb.off + q];
    double vol = pb.volume;
    double g[3] = {1.0, 1.0, 1.0};
    if (pb.lj && !dend_valid(pb, (int)(q % pb.n[0]), (int)((q / pb.n[0]) % pb.n[1]),
                             (int)(q / ((long long)pb.n[0] * pb.n[1]))))
      continue;
    if (pb.sph && pb.ndim >= 2) {
      const int i = (int)(q % pb.n[0]), j = (int)((q / pb.n[0]) % pb.n[1]);
      const size_t fs = (size_t)(pb.n[0] + 2 * MDS_NG) * (pb.n[1] + 2 * MDS_NG);
      const double *zs = pb.zone + (size_t)(j + MDS_NG) * (pb.n[0] + 2 * MDS_NG) + (i + MDS_NG);
      vol = zs[MDS_ZS_VOLUME * fs];
      g[0] = zs[MDS_ZS_GCOV0 * fs]; g[1] = zs[(MDS_ZS_GCOV0 + 1) * fs]; g[2] = zs[(MDS_ZS_GCOV0 + 2) * fs];
    } else if (pb.sph) {
      const double *zg = pb.zone + (size_t)(q + MDS_NG) * MDS_ZG_COUNT;
      vol = zg[MDS_ZG_VOLUME];
      g[0] = zg[MDS_ZG_GCOV00]; g[1] = zg[MDS_ZG_GCOV01]; g[2] = zg[MDS_ZG_GCOV02];
    }
    double vsq = 0.0;
    for (int d = 0; d < nv; d++) { double v = sp.v[2 + d][pb.off + q]; vsq += v * (g[d] * v); }
    double val[2] = {rho * vol, (((0.5 * rho) * vsq) + uu) * vol};
    for (int k = 0; k < 2; k++) {
      double t = s[k] + val[k];
      if (fabs(s[k]) >= fabs(val[k])) cmp[k] += (s[k] - t) + val[k];
      else cmp[k] += (val[k] - t) + s[k];
      s[k] = t;
    }
  }
  __shared__ double sh[4][256];
  sh[0][threadIdx.x] = s[0]; sh[1][threadIdx.x] = cmp[0];
  sh[2][threadIdx.x] = s[1]; sh[3][threadIdx.x] = cmp[1];
  __syncthreads();
  if (threadIdx.x == 0) {
    double S[2] = {0, 0}, C[2] = {0, 0};
    for (int t = 0; t < (int)blockDim.x; t++)
      for (int k = 0; k < 2; k++) {
        double vals[2] = {sh[2 * k][t], sh[2 * k + 1][t]};
        for (int m = 0; m < 2; m++) {
          double tt = S[k] + vals[m];
          if (fabs(S[k]) >= fabs(vals[m])) C[k] += (S[k] - tt) + vals[m];
          else C[k] += (vals[m] - tt) + S[k];
          S[k] = tt;
        }
      }
    partial[4 * blockIdx.x + 0] = S[0];
    partial[4 * blockIdx.x + 1] = C[0];
    partial[4 * blockIdx.x + 2] = S[1];
    partial[4 * blockIdx.x + 3] = C[1];
  }
}

// ---------------------------------------------------------------------------
// helpers
// ---------------------------------------------------------------------------
static size_t rsize(const mds_ctx *c) { return c->precision == MDS_FP32_BULK ? sizeof(float) : sizeof(double); }

template <class R>
static StateArrays<R> arrays(void *const v[5])
{
  StateArrays<R> s;
  for (int k = 0; k < 6; k++) s.v[k] = (R *)v[k];
  return s;
}

static int upload_geo(mds_ctx *c, const void *src, size_t bytes, const void **dst)
{
  void *d = nullptr;
  HIPCHK(c, hipMalloc(&d, bytes));
  c->geo_allocs.push_back(d);
  HIPCHK(c, hipMemcpy(d, src, bytes, hipMemcpyHostToDevice));
  *dst = d;
  return 0;
}

extern "C" void mds_default_run_params(mds_run_params *rp)
{
  rp->cfl = 0.9;
  rp->dt_init_safety = 0.1;
  rp->dt_grow_safety = 1.1;
  rp->dtmin = 1.0e-200;
  rp->dtmax = 1.0e200;
  rp->initial_dt = 1.0e100;
  rp->tmax = 0.0;
  rp->hydro_interp_order = 3;
}

extern "C" const char *mds_last_error(const mds_ctx *ctx) { return ctx ? ctx->err : "null context"; }

extern "C" void *mds_stream(mds_ctx *ctx) { return ctx ? (void *)ctx->st : nullptr; }

extern "C" int mds_destroy(mds_ctx *c)
{
  if (!c) return MDS_OK;
  if (c->st) hipStreamSynchronize(c->st);
  if (c->s3.side) hipStreamSynchronize(c->s3.side);
  drop_graphs(c);
  for (int k = 0; k < 6; k++) { if (c->p[k]) hipFree(c->p[k]); if (c->ph[k]) hipFree(c->ph[k]); }
  if (c->eos_alloc) hipFree(c->eos_alloc);
  if (c->dgrav) hipFree(c->dgrav);
  if (c->dgr) hipFree(c->dgr);
  for (double *b : c->tdep_buf) if (b) hipHostFree(b);
  if (c->dgrst) hipFree(c->dgrst);
  for (int d = 0; d < 3; d++) if (c->s3.F[d]) hipFree(c->s3.F[d]);
  if (c->s3.P) hipFree(c->s3.P);
  if (c->s3.G) hipFree(c->s3.G);
  if (c->s3.CS) hipFree(c->s3.CS);
  if (c->s3.tg) hipFree(c->s3.tg);
  if (c->s3.ms) hipFree(c->s3.ms);
  if (c->s3.part) hipFree(c->s3.part);
  for (int k = 0; k < 5; k++) if (c->s3.ev[k]) hipEventDestroy(c->s3.ev[k]);
  if (c->s3.side) hipStreamDestroy(c->s3.side);
  if (c->s3.grav) hipFree(c->s3.grav);
  for (void *g : c->geo_allocs) hipFree(g);
  if (c->dprob) hipFree(c->dprob);
  if (c->pin) hipHostFree(c->pin);
  for (auto &e : c->pin_ev) if (e) hipEventDestroy(e);
  if (c->dclock) hipFree(c->dclock);
  if (c->dclock2) hipFree(c->dclock2);
  if (c->dmind) hipFree(c->dmind);
  if (c->dseg) hipFree(c->dseg);
  if (c->dseg2) hipFree(c->dseg2);
  if (c->dseg3) hipFree(c->dseg3);
  if (c->dflags) hipFree(c->dflags);
  if (c->dcount) hipFree(c->dcount);
  if (c->dzstart) hipFree(c->dzstart);
  if (c->st) hipStreamDestroy(c->st);
  delete c;
  return MDS_OK;
}

// Radial and theta faces of a dendritic grid whose 4-zone pencils cross a
// level change (prolongation / restriction, step.c:1159-1265), as (i, j, k, 0)
// with k the face's own phi index; every other face of the grid is handled by
// the regular flux kernels.
static int build_dendritic_lists(mds_ctx *c, const mds_grid *g, Sph3Launch &L)
{
  const int n1 = g->n[0], n2 = g->n[1], n3 = g->n[2], NG = MDS_NG, S1 = n2 + 2 * NG;
  auto dj = [&](int i) { return g->dj[i + NG]; };
  auto dk = [&](int i, int j) { return g->dk[(size_t)(i + NG) * S1 + j + NG]; };
  std::vector<int4> rad, th;
  for (int i = 0; i <= n1; i++) {
    const int nj = n2 / dj(i);
    bool jreg = true;
    for (int s = -2; s < 2; s++) jreg = jreg && dj(i + s) == dj(i);
    for (int j = 0; j < nj; j++) {
      bool reg = jreg;
      for (int s = -2; s < 2 && reg; s++) reg = dk(i + s, j) == dk(i, j);
      if (reg) continue;
      for (int k = 0; k < n3 / dk(i, j); k++) rad.push_back(make_int4(i, j, k, 0));
    }
  }
  for (int i = 0; i < n1; i++) {
    const int nj = n2 / dj(i);
    for (int j = 0; j <= nj; j++) {
      const int dkf = dk(i, j) < dk(i, j - 1) ? dk(i, j) : dk(i, j - 1);
      bool reg = true;
      for (int s = -2; s < 2; s++) reg = reg && dk(i, j + s) == dkf;
      if (reg) continue;
      for (int k = 0; k < n3 / dkf; k++) th.push_back(make_int4(i, j, k, 0));
    }
  }
  // order each list by the storage address of its faces' zones, (k, j, i)
  // with i fastest: a wavefront's faces then share the cache lines of the
  // i-fastest state arrays (the faces of one row of a theta level change lie
  // side by side in i; radial faces of neighbouring shells share rows)
  auto by_address = [](const int4 &a, const int4 &b) {
    if (a.z != b.z) return a.z < b.z;
    if (a.y != b.y) return a.y < b.y;
    return a.x < b.x;
  };
  std::sort(rad.begin(), rad.end(), by_address);
  std::sort(th.begin(), th.end(), by_address);
  std::vector<int4> *lists[2] = {&rad, &th};
  for (int t = 0; t < 2; t++) {
    L.nirr[t] = (long long)lists[t]->size();
    L.irr[t] = nullptr;
    if (!L.nirr[t]) continue;
    int rc1 = upload_geo(c, lists[t]->data(), lists[t]->size() * sizeof(int4), (const void **)&L.irr[t]);
    if (rc1) return rc1;
  }
  return 0;
}

// Multipole gravity: the host tables on the device and the stage work arrays.
static int build_multipole(mds_ctx *c, const mds_grid *g, int lmax, Sph3Launch &L)
{
  mds_mp_tab t;
  const int rc = mds_mp_tab_build(g, lmax, &t);
  if (rc) return set_err(c, rc, "multipole gravity tables");
  MpDev &M = L.mp;
  memset(&M, 0, sizeof(M));
  M.lmax = t.lmax;
  M.mmax = t.mmax;
  M.nlm = t.nlm;
  M.maxklev = t.maxklev;
  std::vector<short2> lms;
  for (int l = 0; l <= lmax; l++) {
    const int mm = l < t.mmax ? l : t.mmax;
    for (int m = -mm; m <= mm; m++) lms.push_back(make_short2((short)MDS_MP_LM(l, m), (short)l));
  }
  M.nlist = (int)lms.size();
  const long long rows = (long long)g->n[1] * g->n[2];
  M.npart = (int)((rows + 4 * MDS_MP_ROWS - 1) / (4 * MDS_MP_ROWS));
  const int NJ = t.maxjlev + 1, NK = t.maxklev + 1, n1 = g->n[0], n2 = g->n[1], n3 = g->n[2], L1 = lmax + 1;
  int e = MDS_OK;
  auto up = [&](const void *h, size_t bytes, const void **d) {
    if (e == MDS_OK) e = upload_geo(c, h, bytes, d);
  };
  up(lms.data(), lms.size() * sizeof(short2), (const void **)&M.lms);
  up(t.S, sizeof(double) * (size_t)t.nS, (const void **)&M.S);
  up(t.Soff, sizeof(long long) * NJ * NK, (const void **)&M.Soff);
  up(t.Y, sizeof(double) * (size_t)(n2 + 1) * (n3 + 1) * t.nlm, (const void **)&M.Y);
  up(t.rc, sizeof(double) * (size_t)n1 * L1, (const void **)&M.rc);
  up(t.rd, sizeof(double) * (size_t)n1 * L1, (const void **)&M.rd);
  up(t.Cf, sizeof(double) * (size_t)(n1 + 1) * L1, (const void **)&M.Cf);
  up(t.Df, sizeof(double) * (size_t)(n1 + 1) * L1, (const void **)&M.Df);
  up(t.rm, sizeof(double) * (size_t)(n1 + 1), (const void **)&M.rm);
  up(t.wx, sizeof(double) * 2 * (size_t)n1, (const void **)&M.wx);
  up(t.wy, sizeof(double) * 2 * (size_t)NJ * n2, (const void **)&M.wy);
  up(t.wz, sizeof(double) * 2 * (size_t)NK * n3, (const void **)&M.wz);
  mds_mp_tab_free(&t);
  if (e) return e;
  auto work = [&](size_t bytes, double **d) {
    void *m = nullptr;
    if (e == MDS_OK && hipMalloc(&m, bytes) != hipSuccess) e = set_err(c, MDS_ENOMEM, "multipole work arrays");
    if (e == MDS_OK) { c->geo_allocs.push_back(m); hipMemset(m, 0, bytes); *d = (double *)m; }
  };
  work(sizeof(double) * 2 * (size_t)M.nlist * M.npart * n1, &M.part);
  work(sizeof(double) * (size_t)M.nlist * n1, &M.C);
  work(sizeof(double) * (size_t)M.nlist * n1, &M.D);
  work(sizeof(double) * (size_t)(n1 + 1) * (n2 + 1) * (n3 + 1), &M.phi);
  work(sizeof(double) * 6 * (size_t)n1 * n2 * n3, &M.src);
  if (e == MDS_OK) L.mpl = lmax;
  return e;
}

// ---------------------------------------------------------------------------
// launch shapes
// ---------------------------------------------------------------------------
// A marching kernel's piece of `len` rows (planes) costs len + 2 of them (the
// window's start), and a piece shares its compute unit's issue slots with the
// others there: few long pieces leave units idle and latencies bare, many
// short ones repeat their starts.  The costs below are relative times per row
// (plane), read off sweeps over the pieces on one MI355X.

static bool gen3d(const mds_ctx *c);

// 2D, rows per wavefront.  A row of one wavefront per SIMD waits for its own
// latencies, so the second costs little (FP32: 5.0, 7.4, 8.3 and 10.2 us for 1
// to 4 wavefronts; FP64 19.6 and 29.8 us for 1 and 2); from there the work
// counts.  With the fixed 24 rows of before a 300^2 box took 140 us a step in
// FP32 where 2 rows take 36, 64^2 in FP64 471 and 49, 777 x 1003 in FP64 511
// (8 rows, the best of the shapes tried: 298) and 270 at 7 rows.
static double cost2d(const mds_ctx *c, int rows)
{
  static const double t32[4] = {1.96, 2.9, 3.25, 4.0}, t64[2] = {1.4, 2.13};
  const int fp32 = c->precision == MDS_FP32_BULK, held = fp32 ? 4 : 2;
  const DevProb &h = c->hprob[0];
  const double w = (double)((h.n[0] + MDS_SEG1D - 1) / MDS_SEG1D) * ((h.n[1] + rows - 1) / rows);
  const double r = w / (4.0 * std::max(1, c->ncu));
  const double t = r <= held ? (fp32 ? t32 : t64)[std::max(0, (int)ceil(r) - 1)]
                             : std::max(r + 0.3, held + 1.0);     // a second round of wavefronts
  return (rows + 2) * t;
}

// 3D, planes per workgroup of a tile shape.  FP32 tiles of 4 rows without halo
// wavefronts run three to a compute unit (12.7 us a plane for one, 17.3 for
// three, then 5.4 us each); every other tile fills its unit.  The FP64 tiles
// of 4 rows with halo wavefronts take 36 us a plane, those of 8 without 58,
// which decides between the two on small boxes.
static double cost3d(const mds_ctx *c, int ty, int kc, int hs)
{
  const int fp32 = c->precision == MDS_FP32_BULK;
  const DevProb &h = c->hprob[0];
  const double w = (double)((h.n[0] + MDS_SEG1D - 1) / MDS_SEG1D) * ((h.n[1] + ty - 1) / ty) * ((h.n[2] + kc - 1) / kc);
  const double r = w / std::max(1, c->ncu);
  if (fp32 && ty == 4 && hs)
    return (kc + 2) * (r <= 3.0 ? 12.7 + 2.3 * std::max(0.0, r - 1.0) : std::max(22.0, 5.4 * (r + 0.8)));
  return (kc + 2) * (ty == 4 ? 36.0 : 58.0) * (r <= 8.0 ? std::max(1.0, ceil(r)) : r + 0.5);
}

static const int rows2d[] = {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16, 18, 20, 24, 32, 48, 64};
static const int planes3d[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64};

// The cheapest rows per wavefront.
static int rows_for(const mds_ctx *c)
{
  int best = 1;
  for (int v : rows2d)
    if (v <= c->hprob[0].n[1] && cost2d(c, v) < cost2d(c, best)) best = v;
  return best;
}

// The cheapest planes per workgroup of a tile shape.
static int planes_for(const mds_ctx *c, int ty, int hs)
{
  int best = 1;
  for (int kc : planes3d)
    if (kc <= c->hprob[0].n[2] && cost3d(c, ty, kc, hs) < cost3d(c, ty, best, hs)) best = kc;
  return best;
}

// The shapes of a new context.  Boxes: the cheapest by the costs above; FP32
// boxes in tiles of 4 rows without halo wavefronts, the fastest at every size
// (256^3: 1.93 ms a step against 2.1 to 3.7 for the others; 150 x 122 x 203:
// 0.50 ms, 0.87 with the fixed shape of before), FP64 boxes in the cheaper of
// 4 rows with and 8 without (24^3: 77 us, 622 before; 256^3: 11.4 ms, 13.3).
// FP32 columns: two zones per lane once one zone per lane is more wavefronts
// than the device holds (1024 columns: 107 us against 143; below that the
// wavefronts' latency counts, which one zone per lane has less of).
static void default_shapes(mds_ctx *c)
{
  if (c->sph3) return;
  if (c->ndim == 1) {
    if (c->fuse1d && c->precision == MDS_FP32_BULK && c->nseg2 > 16 * std::max(1, c->ncu)) c->fuse1d = 2;
  } else if (c->ndim == 2) {
    c->chunk2d = rows_for(c);
  } else {
    c->ty3d = 4;
    c->halo3d = c->precision == MDS_FP32_BULK && !gen3d(c);
    c->kc3d = planes_for(c, c->ty3d, c->halo3d);
    if (c->precision != MDS_FP32_BULK && !gen3d(c)) {
      const int kc = planes_for(c, 8, 1);
      if (cost3d(c, 8, kc, 1) < cost3d(c, 4, c->kc3d, 0)) { c->ty3d = 8; c->halo3d = 1; c->kc3d = kc; }
    }
  }
}

static int create_impl(mds_ctx *c, const mds_problem *probs, int nprob, const mds_run_params *rp)
{
  c->nprob = nprob;
  c->rp.cfl = rp->cfl;
  c->rp.dt_init_safety = rp->dt_init_safety;
  c->rp.dt_grow_safety = rp->dt_grow_safety;
  c->rp.dtmin = rp->dtmin;
  c->rp.dtmax = rp->dtmax;
  c->rp.initial_dt = rp->initial_dt;
  if (rp->hydro_interp_order < 1 || rp->hydro_interp_order > 3)
    return set_err(c, MDS_EINVAL, "hydro_interp_order must be 1, 2 or 3");
  if (rp->hydro_interp_order != 3 && c->precision == MDS_FP32_BULK)
    return set_err(c, MDS_ENOTIMPL, "FP32-bulk reconstructs with para_recon (hydro_interp_order 3) only");
  c->tmax = rp->tmax;
  c->ndim = probs[0].grid->ndim;
  c->sph = probs[0].grid->geom == MDS_GEOM_SPHERICAL;
  // auto: FP64 spherical columns carry all three velocity components (the
  // connection terms give the transverse ones round-off sources, so the
  // reference evolves them); FP32-bulk carries the ndim physical ones
  auto auto_nv = [&](const mds_problem &P) {
    if (P.nvel) return P.nvel;
    bool s = P.grid && P.grid->geom == MDS_GEOM_SPHERICAL;
    return (s && c->precision == MDS_FP64) ? 3 : (P.grid ? P.grid->ndim : 1);
  };
  c->nv = auto_nv(probs[0]);
  if (c->ndim > 1 && nprob != 1) return set_err(c, MDS_ENOTIMPL, "batches are supported for 1D columns only");
  // 3D grids and 2D/3D spherical grids evolve all three components: an
  // explicit other count is an error, not something to override
  if ((c->ndim == 3 || (c->sph && c->ndim >= 2)) && probs[0].nvel != 0 && probs[0].nvel != 3)
    return set_err(c, MDS_EINVAL, "3D and 2D/3D spherical grids carry three velocity components (nvel 0 or 3)");
  if (c->ndim == 1 && c->nv == 2) c->nv = 3;
  if (c->ndim == 2 && c->nv < 2) c->nv = 2;
  if (c->ndim == 3) c->nv = 3;
  // 2D (r, theta) grids run the 3D spherical kernels on one phi zone of 2 pi,
  // without phi faces and without the phi term of the zone dt
  c->sph3 = c->sph && c->ndim >= 2;
  if (c->sph3) c->nv = 3;
  if (c->sph && c->precision == MDS_FP64 && c->nv != 3)
    return set_err(c, MDS_EINVAL, "FP64 spherical columns carry three velocity components");
  if (c->sph && !c->sph3 && c->precision == MDS_FP32_BULK && c->nv != 1 && c->nv != 3)
    return set_err(c, MDS_EINVAL, "FP32-bulk spherical columns carry the radial velocity (nvel 1) or all three (nvel 3)");
  c->tab = probs[0].eos != nullptr;
  c->mono = probs[0].monopole;
  for (int p = 0; p < nprob; p++)
    if (probs[p].monopole < 0 || probs[p].monopole > MDS_MONOPOLE_GR)
      return set_err(c, MDS_EINVAL, "problem %d: monopole must be 0, MDS_MONOPOLE_NEWTON or MDS_MONOPOLE_GR", p);
  for (int p = 1; p < nprob; p++)
    if ((probs[p].eos != probs[0].eos) || (probs[p].monopole != c->mono))
      return set_err(c, MDS_EINVAL, "problem %d: every problem of a batch needs the same EOS and gravity", p);
  if (probs[0].multipole_lmax < 0 || probs[0].multipole_lmax > MDS_MULTIPOLE_LMAX)
    return set_err(c, MDS_EINVAL, "multipole_lmax must be in [0, %d]", MDS_MULTIPOLE_LMAX);
  if (probs[0].multipole_lmax > 0 &&
      (!c->mono || probs[0].grid->geom != MDS_GEOM_SPHERICAL || probs[0].grid->ndim < 2))
    return set_err(c, MDS_EINVAL, "multipole gravity needs monopole gravity on a 2D or 3D spherical grid");
  if ((c->tab || c->mono) && !c->sph)
    return set_err(c, MDS_ENOTIMPL, "tabulated EOS and monopole gravity are supported on spherical grids");
  if (c->tab) {
    const mds_eos_table *t = probs[0].eos;
    if (!t->data || t->nr < 2 || t->nt < 3 || t->ny < 2 || t->nt - 1 > (1 << 20))
      return set_err(c, MDS_EINVAL, "EOS table without data or with bad dimensions");
    HIPCHK(c, mds_eos_to_device(t, &c->deos, &c->eos_alloc));
    c->nstate = 6;
  }
  HIPCHK(c, hipStreamCreateWithFlags(&c->st, hipStreamNonBlocking));
  {
    int dev = 0;
    HIPCHK(c, hipGetDevice(&dev));
    HIPCHK(c, hipDeviceGetAttribute(&c->ncu, hipDeviceAttributeMultiprocessorCount, dev));
    c->dev = dev;
  }
  c->zstart.assign(nprob + 1, 0);
  c->hprob.resize(nprob);
  for (int p = 0; p < nprob; p++) {
    const mds_problem &P = probs[p];
    const mds_grid *g = P.grid;
    if (!g || g->ndim != c->ndim || (g->geom == MDS_GEOM_SPHERICAL) != (c->sph != 0))
      return set_err(c, MDS_EINVAL, "problem %d: every problem of a batch needs the same ndim and geometry", p);
    int nvp = auto_nv(P);
    if (c->ndim == 1 && nvp == 2) nvp = 3;
    if (c->ndim == 2 && nvp < 2) nvp = 2;
    if (c->ndim == 3 || c->sph3) nvp = 3;
    if (nvp != c->nv) return set_err(c, MDS_EINVAL, "problem %d: velocity component count differs in the batch", p);
    for (int d = 0; d < g->ndim; d++) {
      if (g->n[d] < 4) return set_err(c, MDS_EINVAL, "problem %d: need at least 4 zones per active direction", p);
      for (int side = 0; side < 2; side++) {
        int b = side ? P.bc_hi[d] : P.bc_lo[d];
        // SPHERICAL_ORIGIN: theta across the pole of 3D spherical grids, or
        // the inner radius through the origin of 1D and 3D spherical grids
        const bool phi_ok = g->ndim == 2 || (g->n[2] % 2) == 0;     // the phi + pi map
        const bool pole = c->sph3 && d == 1 && b == MDS_BC_SPHERICAL_ORIGIN && phi_ok;
        const bool origin = c->sph && d == 0 && side == 0 && b == MDS_BC_SPHERICAL_ORIGIN && (!c->sph3 || phi_ok);
        // ghost layers held on the device: PROB anywhere but the inner radius
        // and the angles of 3D spherical grids; EXTRAP in direction 0 (the
        // only direction the reference extrapolates), not at that inner radius
        const bool slab = (b == MDS_BC_PROB && (!c->sph3 || (d == 0 && side == 1))) ||
                          (b == MDS_BC_EXTRAP && d == 0 && (!c->sph3 || side == 1)) ||
                          (b == MDS_BC_DISK && d == 0 && side == 0 && !c->sph3);
        if (b != MDS_BC_OUTFLOW && b != MDS_BC_REFLECT && b != MDS_BC_PERIODIC && !pole && !origin && !slab)
          return set_err(c, MDS_ENOTIMPL, "problem %d: boundary code %d not supported on the device", p, b);
      }
    }
    if (g->dendritic) {
      if (!c->sph3 || !g->dj || !g->dk)
        return set_err(c, MDS_EINVAL, "problem %d: dendritic grids are built 2D or 3D spherical grids", p);
      // (2D grids have one phi zone and no phi boundary)
      if ((P.bc_lo[0] != MDS_BC_REFLECT && P.bc_lo[0] != MDS_BC_SPHERICAL_ORIGIN) ||
          (P.bc_hi[0] != MDS_BC_OUTFLOW && P.bc_hi[0] != MDS_BC_REFLECT && P.bc_hi[0] != MDS_BC_PROB &&
           P.bc_hi[0] != MDS_BC_EXTRAP) ||
          P.bc_lo[1] != MDS_BC_SPHERICAL_ORIGIN || P.bc_hi[1] != MDS_BC_SPHERICAL_ORIGIN ||
          (g->ndim == 3 && (P.bc_lo[2] != MDS_BC_PERIODIC || P.bc_hi[2] != MDS_BC_PERIODIC)))
        return set_err(c, MDS_ENOTIMPL,
                       "problem %d: dendritic grids need REFLECT or SPHERICAL_ORIGIN inner / OUTFLOW, REFLECT, PROB "
                       "or EXTRAP outer radius, the pole in theta and periodic phi", p);
      const int n1 = g->n[0], S1 = g->n[1] + 2 * MDS_NG;
      c->hdj.assign(g->dj, g->dj + (n1 + 2 * MDS_NG));
      c->hdk.assign(g->dk, g->dk + (size_t)(n1 + 2 * MDS_NG) * S1);
      if (P.bc_hi[0] == MDS_BC_EXTRAP) {
        // the reference extrapolates at the ghost's own (j, k): the two outer
        // shells must share their levels
        bool same = g->dj[n1 - 2 + MDS_NG] == g->dj[n1 - 1 + MDS_NG];
        for (int j = 0; same && j < g->n[1] / g->dj[n1 - 1 + MDS_NG]; j++)
          same = g->dk[(size_t)(n1 - 2 + MDS_NG) * S1 + j + MDS_NG] == g->dk[(size_t)(n1 - 1 + MDS_NG) * S1 + j + MDS_NG];
        if (!same)
          return set_err(c, MDS_ENOTIMPL, "problem %d: EXTRAP needs the two outer shells on one level", p);
      }
    }
    long long nz = (long long)g->n[0] * (g->ndim > 1 ? g->n[1] : 1) * (g->ndim > 2 ? g->n[2] : 1);
    c->zstart[p + 1] = c->zstart[p] + nz;
    DevProb &d = c->hprob[p];
    memset(&d, 0, sizeof(d));
    d.off = c->zstart[p];
    d.ndim = g->ndim;
    d.sph = c->sph;
    d.rcoord = g->rcoord;
    d.rtrans = g->rtrans;
    d.gam = P.gam;
    for (int k = 0; k < 3; k++) {
      d.n[k] = k < g->ndim ? g->n[k] : 1;
      d.bc_lo[k] = P.bc_lo[k];
      d.bc_hi[k] = P.bc_hi[k];
      d.g0[k] = P.g0[k];
      d.startx[k] = g->startx[k];
      d.dx[k] = g->dx[k];
      d.area[k] = g->area[k];
    }
    d.volume = g->volume;
    d.ivolume = g->volume != 0.0 ? 1.0 / g->volume : 0.0;
    for (int k = 0; k < 3; k++) d.idx[k] = 1.0 / d.dx[k];
    d.order = rp->hydro_interp_order;
    d.mono = c->mono;
    // one FP32 coefficient set for the whole column when the zones' sets
    // agree to 1e-5 (the moments of log-r and uniform grids differ only by
    // scale and shift; the spread left is the rounding of the FP64 moments,
    // which grows with n): the per-coefficient median of the reconstructed
    // zones -1 .. n
    {
      const int nzk = g->n[0] + 2 * MDS_NG;
      bool uni = true;
      std::vector<double> col(nzk - 2);
      for (int k = 0; k < MDS_RC_COUNT && uni; k++) {
        for (int q = 1; q < nzk - 1; q++) col[q - 1] = g->rcoef[0][(size_t)q * MDS_RC_COUNT + k];
        std::vector<double> srt(col);
        std::nth_element(srt.begin(), srt.begin() + srt.size() / 2, srt.end());
        const double med = srt[srt.size() / 2];
        for (double v : col) uni = uni && fabs(v - med) <= 1.0e-5 * fabs(med) + 1.0e-12;
        d.rcu_c[k] = (float)med;
      }
      d.rcu = uni ? 1 : 0;
    }
    // the transverse metric ratios and connection coefficients of a
    // spherical column, when every zone shares them to 1e-10 (a log-r column)
    d.tcu = 0;
    if (c->sph && !c->sph3 && g->zone) {
      const int nzk = g->n[0] + 2 * MDS_NG;
      const int cf[11] = {MDS_ZG_C000, MDS_ZG_C101, MDS_ZG_C202, MDS_ZG_C011, MDS_ZG_C110, MDS_ZG_C111,
                          MDS_ZG_C212, MDS_ZG_C022, MDS_ZG_C122, MDS_ZG_C220, MDS_ZG_C221};
      auto val = [&](int q, int t) -> double {
        const double *z = g->zone + (size_t)q * MDS_ZG_COUNT;
        switch (t) {
          case MDS_TC_G1: return z[MDS_ZG_GCOV01] / z[MDS_ZG_GCOV00];
          case MDS_TC_G2: return z[MDS_ZG_GCOV02] / z[MDS_ZG_GCOV00];
          case MDS_TC_GI1: return z[MDS_ZG_GCON1] * z[MDS_ZG_GCOV00];
          case MDS_TC_GI2: return z[MDS_ZG_GCON2] * z[MDS_ZG_GCOV00];
          case MDS_TC_F1: return z[MDS_ZG_GCOVF1] / z[MDS_ZG_GCOVF0];
          case MDS_TC_F2: return z[MDS_ZG_GCOVF2] / z[MDS_ZG_GCOVF0];
          default: return z[cf[t - MDS_TC_C000]];
        }
      };
      // zone values over the interior zones (the only ones updated), the
      // lower-face ratios over the faces 0 .. n (ghost records carry no
      // connection coefficients)
      bool uni = true;
      for (int t = 0; t < MDS_TC_COUNT && uni; t++) {
        const double ref = val(MDS_NG, t);
        double scale = fabs(ref);
        for (int tt = MDS_TC_C000; tt < MDS_TC_COUNT && t >= MDS_TC_C000; tt++) scale = fmax(scale, fabs(val(MDS_NG, tt)));
        const int q1 = (t == MDS_TC_F1 || t == MDS_TC_F2) ? nzk - MDS_NG : nzk - MDS_NG - 1;
        for (int q = MDS_NG; q <= q1 && uni; q++) {
          const double v = val(q, t);
          uni = std::isfinite(v) && fabs(v - ref) <= 1.0e-10 * scale;
        }
        d.tcu_c[t] = ref;
      }
      d.tcu = uni ? 1 : 0;
    }
    // ghost layers of the PROB and EXTRAP sides
    d.has_slab = 0;
    {
      long long items = 0;
      int pending = 0;
      for (int dd = 0; dd < g->ndim; dd++)
        for (int side = 0; side < 2; side++) {
          const int b = side ? P.bc_hi[dd] : P.bc_lo[dd];
          if (b != MDS_BC_PROB && b != MDS_BC_EXTRAP && b != MDS_BC_DISK) continue;
          const size_t bytes = sizeof(double) * MDS_NG * MDS_SLAB_NV * (size_t)slab_T(d, dd);
          void *m = nullptr;
          HIPCHK(c, hipMalloc(&m, bytes));
          c->geo_allocs.push_back(m);
          HIPCHK(c, hipMemset(m, 0, bytes));
          d.gs[dd][side] = (double *)m;
          d.has_slab = 1;
          items += MDS_NG * slab_T(d, dd);
          pending += b == MDS_BC_PROB;
        }
      c->has_slab |= d.has_slab;
      c->slab_items = std::max(c->slab_items, items);
      c->prob_pending.push_back(pending);
    }
    for (int k = 0; k < g->ndim; k++) {
      int nzk = g->n[k] + 2 * MDS_NG;
      std::vector<double> mom(3 * (size_t)nzk);
      std::vector<float> rcf((size_t)nzk * MDS_RC_COUNT);
      for (int q = 0; q < nzk; q++) {
        mom[3 * q + 0] = g->alpha[k][q];
        mom[3 * q + 1] = g->beta[k][q];
        mom[3 * q + 2] = g->Gamma[k][q];
      }
      for (size_t q = 0; q < rcf.size(); q++) rcf[q] = (float)g->rcoef[k][q];
      int rc1 = upload_geo(c, mom.data(), mom.size() * sizeof(double), (const void **)&d.mom[k]);
      if (rc1) return rc1;
      rc1 = upload_geo(c, rcf.data(), rcf.size() * sizeof(float), (const void **)&d.rc[k]);
      if (rc1) return rc1;
      if (c->precision != MDS_FP32_BULK && g->geom == MDS_GEOM_CARTESIAN && g->ndim > 1) {
        // the quotients of recon_geo_x64 and the faces of the zones that have
        // both neighbours
        std::vector<double> rg((size_t)nzk * MDS_RG_COUNT, 0.0);
        for (int q = 1; q < nzk - 1; q++) {
          const double *al = g->alpha[k] + q, *be = g->beta[k] + q, *ga = g->Gamma[k] + q;
          if (ga[-1] != g->dx[k] || ga[0] != g->dx[k] || ga[1] != g->dx[k])
            return set_err(c, MDS_EINVAL, "a Cartesian grid's Gamma moments are its zone width");
          ReconGeo64 z;
          z.am = al[-1]; z.bm = be[-1]; z.gm = ga[-1];
          z.a0 = al[0];  z.b0 = be[0];  z.g0 = ga[0];
          z.ap = al[1];  z.bp = be[1];  z.gp = ga[1];
          z.xlo = g->startx[k] + (q - MDS_NG) * g->dx[k];
          z.xhi = g->startx[k] + (q - MDS_NG + 1) * g->dx[k];
          recon_geo_x64(z);
          double *o = &rg[(size_t)q * MDS_RG_COUNT];
          o[MDS_RG_DEN] = z.den; o[MDS_RG_DEN2] = z.den2; o[MDS_RG_XLO] = z.xlo; o[MDS_RG_XHI] = z.xhi;
        }
        rc1 = upload_geo(c, rg.data(), rg.size() * sizeof(double), (const void **)&d.rg64[k]);
        if (rc1) return rc1;
      }
    }
    if (g->dendritic) {
      // level tables (log2 of dj, dk) and the theta / phi moments of every level
      const int N1 = g->n[0] + 2 * MDS_NG, N2 = g->n[1] + 2 * MDS_NG;
      std::vector<unsigned char> lj(N1), lk((size_t)N1 * N2, 0);
      auto lg = [](int f) { int l = 0; while (f >>= 1) l++; return l; };
      for (int q = 0; q < N1; q++) lj[q] = (unsigned char)lg(g->dj[q]);
      // the device table is i fastest (a wavefront runs along i)
      for (int i = 0; i < N1; i++)
        for (int j = 0; j < N2; j++) {
          const int f = g->dk[(size_t)i * N2 + j];
          lk[(size_t)j * N1 + i] = f > 0 ? (unsigned char)lg(f) : 0;
        }
      int rc1 = upload_geo(c, lj.data(), lj.size(), (const void **)&d.lj);
      if (rc1) return rc1;
      rc1 = upload_geo(c, lk.data(), lk.size(), (const void **)&d.lk);
      if (rc1) return rc1;
      const int nlev[2] = {g->maxjlev + 1, g->maxklev + 1};
      for (int t = 0; t < 2; t++) {
        const int nzk = g->n[t + 1] + 2 * MDS_NG;
        std::vector<double> mom(3 * (size_t)nzk * nlev[t]);
        std::vector<float> rcf((size_t)nzk * MDS_RC_COUNT * nlev[t]);
        for (size_t q = 0; q < (size_t)nzk * nlev[t]; q++) {
          mom[3 * q + 0] = g->lalpha[t][q];
          mom[3 * q + 1] = g->lbeta[t][q];
          mom[3 * q + 2] = g->lGamma[t][q];
        }
        for (size_t q = 0; q < rcf.size(); q++) rcf[q] = (float)g->lrcoef[t][q];
        rc1 = upload_geo(c, mom.data(), mom.size() * sizeof(double), (const void **)&d.lmom[t]);
        if (rc1) return rc1;
        rc1 = upload_geo(c, rcf.data(), rcf.size() * sizeof(float), (const void **)&d.lrc[t]);
        if (rc1) return rc1;
      }
    }
    if (c->sph) {
      if (!g->zone) return set_err(c, MDS_EINVAL, "problem %d: spherical grid without zone records", p);
      const int nzq = g->n[0] + 2 * MDS_NG;
      const size_t zbytes = c->sph3 ? (size_t)nzq * (g->n[1] + 2 * MDS_NG) * MDS_ZS_COUNT * sizeof(double)
                                    : (size_t)nzq * MDS_ZG_COUNT * sizeof(double);
      int rc1;
      if (c->sph3) {
        // field-major copy of the per-(i, j) records (the kernels read one field along i at a time)
        const size_t nrec = (size_t)nzq * (g->n[1] + 2 * MDS_NG);
        std::vector<double> soa(nrec * MDS_ZS_COUNT);
        for (size_t q = 0; q < nrec; q++)
          for (int f = 0; f < MDS_ZS_COUNT; f++) soa[(size_t)f * nrec + q] = g->zone[q * MDS_ZS_COUNT + f];
        rc1 = upload_geo(c, soa.data(), zbytes, (const void **)&d.zone);
      } else {
        rc1 = upload_geo(c, g->zone, zbytes, (const void **)&d.zone);
      }
      if (rc1) return rc1;
      if (c->precision == MDS_FP32_BULK && !c->sph3) {
        std::vector<ZoneF32> z32((size_t)nzq);
        for (int q = 0; q < nzq; q++) {
          const double *zg = g->zone + (size_t)q * MDS_ZG_COUNT;
          ZoneF32 &z = z32[q];
          memset(&z, 0, sizeof(z));
          z.ivol = zg[MDS_ZG_VOLUME] != 0.0 ? 1.0 / zg[MDS_ZG_VOLUME] : 0.0;
          z.area = zg[MDS_ZG_AREA0];
          z.gcov0 = zg[MDS_ZG_GCOV00];
          z.cp = (zg[MDS_ZG_C000] + zg[MDS_ZG_C101]) + zg[MDS_ZG_C202];
          z.c000 = (float)zg[MDS_ZG_C000];
          z.scalef = (float)zg[MDS_ZG_SCALEF];
          z.gcovf0 = (float)zg[MDS_ZG_GCOVF0];
          const double xlo = g->startx[0] + (q - MDS_NG) * g->dx[0];
          z.dcen = (float)(g->beta[0][q] / g->Gamma[0][q] - xlo);
        }
        rc1 = upload_geo(c, z32.data(), z32.size() * sizeof(ZoneF32), (const void **)&d.z32);
        if (rc1) return rc1;
      }
    }
  }
  c->nzone = c->zstart[nprob];
  size_t rs = rsize(c);
  for (int k = 0; k < c->nstate; k++) {
    HIPCHK(c, hipMalloc(&c->p[k], (size_t)c->nzone * rs));
    HIPCHK(c, hipMalloc(&c->ph[k], (size_t)c->nzone * rs));
    HIPCHK(c, hipMemset(c->p[k], 0, (size_t)c->nzone * rs));
    HIPCHK(c, hipMemset(c->ph[k], 0, (size_t)c->nzone * rs));
  }
  if (c->mono && !c->sph3) {
    HIPCHK(c, hipMalloc(&c->dgrav, sizeof(double) * (size_t)c->nzone));
    HIPCHK(c, hipMemset(c->dgrav, 0, sizeof(double) * (size_t)c->nzone));
  }
  if (c->mono == MDS_MONOPOLE_GR) {
    // per problem: the host-made shell geometry (first four arrays), the
    // rest zero; Gamma is set by the first call
    std::vector<size_t> goff(nprob + 1, 0);
    for (int p = 0; p < nprob; p++) goff[p + 1] = goff[p] + (size_t)MDS_GR_COUNT * (c->hprob[p].n[0] + 1);
    c->gr_doubles = goff[nprob];
    std::vector<double> h(c->gr_doubles, 0.0);
    for (int p = 0; p < nprob; p++)
      if (mds_gr_shell_geometry(probs[p].grid, h.data() + goff[p]) != MDS_OK)
        return set_err(c, MDS_EINVAL, "problem %d: GR monopole shell geometry", p);
    HIPCHK(c, hipMalloc(&c->dgr, sizeof(double) * c->gr_doubles));
    HIPCHK(c, hipMemcpy(c->dgr, h.data(), sizeof(double) * c->gr_doubles, hipMemcpyHostToDevice));
    HIPCHK(c, hipMalloc(&c->dgrst, sizeof(int) * 4 * nprob));
    HIPCHK(c, hipMemset(c->dgrst, 0, sizeof(int) * 4 * nprob));
    for (int p = 0; p < nprob; p++) {
      c->hprob[p].gr = c->dgr + goff[p];
      c->hprob[p].grst = c->dgrst + 4 * p;
    }
  }
  if (c->sph3) {
    const DevProb &h = c->hprob[0];
    Sph3Launch &L = c->s3;
    HIPCHK(c, hipStreamCreateWithFlags(&L.side, hipStreamNonBlocking));
    for (int k = 0; k < 5; k++) HIPCHK(c, hipEventCreateWithFlags(&L.ev[k], hipEventDisableTiming));
    L.fp32 = c->precision == MDS_FP32_BULK;
    L.tab = c->tab;
    L.mono = c->mono;
    L.upd = 3;
    const int nslot = c->tab ? 6 : 5;
    for (int d = 0; d < 3; d++) {
      L.nf[d] = (long long)(h.n[0] + (d == 0)) * (h.n[1] + (d == 1)) * (h.n[2] + (d == 2));
      const size_t fs = L.fp32 ? sizeof(float) : sizeof(double);
      // the update addresses one slot's faces with 32-bit byte offsets
      if (fs * (size_t)L.nf[d] >= ((size_t)1 << 32))
        return set_err(c, MDS_EINVAL, "3D spherical grid too large: %lld faces in direction %d (at most %zu)",
                       L.nf[d], d, (((size_t)1 << 32) - 1) / fs);
      HIPCHK(c, hipMalloc(&L.F[d], fs * nslot * (size_t)L.nf[d]));
      HIPCHK(c, hipMemset(L.F[d], 0, fs * nslot * (size_t)L.nf[d]));
    }
    if (c->tab) {
      HIPCHK(c, hipMalloc(&L.P, rs * (size_t)c->nzone));
      HIPCHK(c, hipMalloc(&L.G, rs * (size_t)c->nzone));
      HIPCHK(c, hipMalloc(&L.CS, rs * (size_t)c->nzone));
      HIPCHK(c, hipMalloc(&L.tg, sizeof(unsigned short) * (size_t)c->nzone));
      HIPCHK(c, hipMemset(L.tg, 0, sizeof(unsigned short) * (size_t)c->nzone));
    }
    if (c->mono) {
      HIPCHK(c, hipMalloc(&L.ms, sizeof(double) * h.n[0]));
      L.npart = (int)(((long long)h.n[1] * h.n[2] + 4 * MDS_SHELL_ROWS - 1) / (4 * MDS_SHELL_ROWS));
      // shell-mass parts, or the four GR shell sums' parts
      const size_t nq = c->mono == MDS_MONOPOLE_GR ? 4 : 1;
      HIPCHK(c, hipMalloc(&L.part, sizeof(double) * nq * (size_t)L.npart * h.n[0]));
      HIPCHK(c, hipMalloc(&L.grav, sizeof(double) * h.n[0]));
    }
    const mds_grid *g = probs[0].grid;
    if (g->dendritic) {
      L.dend = 1;
      int rc1 = build_dendritic_lists(c, g, L);
      if (rc1) return rc1;
    }
    if (probs[0].multipole_lmax > 0) {
      int rc1 = build_multipole(c, g, probs[0].multipole_lmax, L);
      if (rc1) return rc1;
    }
  }
  HIPCHK(c, hipMalloc(&c->dprob, sizeof(DevProb) * nprob));
  HIPCHK(c, hipMemcpy(c->dprob, c->hprob.data(), sizeof(DevProb) * nprob, hipMemcpyHostToDevice));
  HIPCHK(c, hipMalloc(&c->dclock, sizeof(DevClock) * nprob));
  HIPCHK(c, hipMemset(c->dclock, 0, sizeof(DevClock) * nprob));
  HIPCHK(c, hipMalloc(&c->dcount, 4 * sizeof(unsigned long long)));
  HIPCHK(c, hipMemset(c->dcount, 0, 4 * sizeof(unsigned long long)));
  HIPCHK(c, hipMalloc(&c->dzstart, sizeof(long long) * (nprob + 1)));
  HIPCHK(c, hipMemcpy(c->dzstart, c->zstart.data(), sizeof(long long) * (nprob + 1), hipMemcpyHostToDevice));
  if (c->ndim == 1) {
    // segment table, longest problems first so the tail of the launch is short
    std::vector<int> order(nprob);
    for (int p = 0; p < nprob; p++) order[p] = p;
    std::vector<int2> seg;
    std::sort(order.begin(), order.end(), [&](int a, int b) { return c->hprob[a].n[0] > c->hprob[b].n[0]; });
    for (int p : order)
      for (int s = 0; s < c->hprob[p].n[0]; s += MDS_SEG1D) seg.push_back(make_int2(p, s));
    c->nseg = (int)seg.size();
    HIPCHK(c, hipMalloc(&c->dseg, sizeof(int2) * seg.size()));
    HIPCHK(c, hipMemcpy(c->dseg, seg.data(), sizeof(int2) * seg.size(), hipMemcpyHostToDevice));
    seg.clear();
    for (int p : order)
      for (int s = 0; s < c->hprob[p].n[0]; s += MDS_SEG1D2) seg.push_back(make_int2(p, s));
    c->nseg2 = (int)seg.size();
    HIPCHK(c, hipMalloc(&c->dseg2, sizeof(int2) * seg.size()));
    HIPCHK(c, hipMemcpy(c->dseg2, seg.data(), sizeof(int2) * seg.size(), hipMemcpyHostToDevice));
    seg.clear();
    for (int p : order)
      for (int s = 0; s < c->hprob[p].n[0]; s += MDS_SEG1D2Z) seg.push_back(make_int2(p, s));
    c->nseg3 = (int)seg.size();
    HIPCHK(c, hipMalloc(&c->dseg3, sizeof(int2) * seg.size()));
    HIPCHK(c, hipMemcpy(c->dseg3, seg.data(), sizeof(int2) * seg.size(), hipMemcpyHostToDevice));
    // the two-stage kernel needs every ghost source zone inside the wave, and
    // no field that depends on the whole column between the stages
    for (const DevProb &h : c->hprob) c->nmax1d = std::max(c->nmax1d, h.n[0]);
    c->can_fuse1d = !c->mono && !c->has_slab && rp->hydro_interp_order == 3;
    for (int p = 0; p < nprob; p++)
      if (c->hprob[p].bc_lo[0] == MDS_BC_PERIODIC || c->hprob[p].bc_hi[0] == MDS_BC_PERIODIC) c->can_fuse1d = 0;
    c->fuse1d = c->can_fuse1d;
    // second clocks and running minima of folded steps (mds_clock.h)
    if (c->can_fuse1d) {
      const double big = 1.0e100;
      unsigned long long k;
      memcpy(&k, &big, sizeof(k));
      const std::vector<unsigned long long> mind((size_t)nprob * MDS_FOLD, k);
      HIPCHK(c, hipMalloc(&c->dclock2, sizeof(DevClock) * nprob));
      HIPCHK(c, hipMemset(c->dclock2, 0, sizeof(DevClock) * nprob));
      HIPCHK(c, hipMalloc(&c->dmind, sizeof(unsigned long long) * mind.size()));
      HIPCHK(c, hipMemcpy(c->dmind, mind.data(), sizeof(unsigned long long) * mind.size(), hipMemcpyHostToDevice));
    }
  } else {
    HIPCHK(c, hipMalloc(&c->dflags, (size_t)c->nzone));
    HIPCHK(c, hipMemset(c->dflags, 0, (size_t)c->nzone));
  }
  default_shapes(c);
  if (const char *e = getenv("MDS_TILE_ROWS2D")) c->chunk2d = atoi(e) > 0 ? atoi(e) : c->chunk2d;
  return MDS_OK;
}

extern "C" int mds_create(const mds_problem *probs, int nprob, const mds_run_params *rp, int precision,
                          mds_ctx **out)
{
  if (!out) return MDS_EINVAL;
  *out = nullptr;
  if (!probs || nprob < 1 || !rp) return MDS_EINVAL;
  if (precision != MDS_FP64 && precision != MDS_FP32_BULK) return MDS_EINVAL;
  mds_ctx *c = new (std::nothrow) mds_ctx();
  if (!c) return MDS_ENOMEM;
  c->precision = precision;
  int rc = create_impl(c, probs, nprob, rp);
  if (rc) {
    // keep the message for the caller: print it, since the context is released
    fprintf(stderr, "mds_create: %s\n", c->err);
    mds_destroy(c);
    return rc;
  }
  *out = c;
  return MDS_OK;
}

// The values of every PROB side of problem prob from eval(i, j, k, q):
// out(d, side) names the host buffer of side (d, side) (MDS_NG * MDS_SLAB_NV
// * T doubles, entry-major), or null to skip it.
template <class Eval, class Out>
static void prob_fill_host(mds_ctx *c, int prob, Eval eval, Out out)
{
  const DevProb &pb = c->hprob[prob];
  for (int d = 0; d < pb.ndim; d++)
    for (int side = 0; side < 2; side++) {
      const int code = side ? pb.bc_hi[d] : pb.bc_lo[d];
      if (code != MDS_BC_PROB) continue;
      double *h = out(d, side);
      if (!h) continue;
      const long long T = slab_T(pb, d);
      const int lo1 = d == 0 ? 1 : 0, lo2 = d == 2 ? 1 : 2;   // transverse directions in index order
      for (int g = 0; g < MDS_NG; g++) {
        const int c0 = side ? pb.n[d] + g : g - MDS_NG;
        for (long long t = 0; t < T; t++) {
          const int a = (int)(t % pb.n[lo1]), b = (int)(t / pb.n[lo1]);
          int idx[3];
          idx[d] = c0;
          idx[lo1] = a;
          idx[lo2] = b;
          if (!c->hdj.empty()) {
            // dendritic outer radius: the positions of the ghost shell's own level
            const int S1 = pb.n[1] + 2 * MDS_NG;
            const int dj = c->hdj[c0 + MDS_NG];
            if (idx[1] >= pb.n[1] / dj) continue;
            const int dk = c->hdk[(size_t)(c0 + MDS_NG) * S1 + idx[1] + MDS_NG];
            if (idx[2] >= pb.n[2] / dk) continue;
          }
          double q[8] = {0, 0, 0, 0, 0, 0, 0, 0};
          eval(pb.ndim > 0 ? idx[0] : 0, pb.ndim > 1 ? idx[1] : 0, pb.ndim > 2 ? idx[2] : 0, q);
          for (int v = 0; v < 6; v++) {
            if (v >= 2 + c->nv && v < 5) continue;   // velocity components the state does not carry
            if (v == 5 && !c->tab) continue;
            h[((size_t)g * MDS_SLAB_NV + v) * T + t] = q[v];
          }
        }
      }
    }
}

extern "C" int mds_set_prob_bounds(mds_ctx *c, int prob, mds_prob_bounds_fn fn, void *user)
{
  if (!c || prob < 0 || prob >= c->nprob || !fn) return MDS_EINVAL;
  const DevProb &pb = c->hprob[prob];
  HIPCHK(c, hipStreamSynchronize(c->st));
  std::vector<double> h[3][2];
  prob_fill_host(c, prob, [&](int i, int j, int k, double *q) { fn(i, j, k, q, user); },
                 [&](int d, int side) {
                   h[d][side].assign((size_t)MDS_NG * MDS_SLAB_NV * slab_T(pb, d), 0.0);
                   return h[d][side].data();
                 });
  for (int d = 0; d < 3; d++)
    for (int side = 0; side < 2; side++)
      if (!h[d][side].empty())
        HIPCHK(c, hipMemcpy(pb.gs[d][side], h[d][side].data(), h[d][side].size() * sizeof(double),
                            hipMemcpyHostToDevice));
  if (!c->tdep_fn.empty() && c->tdep_fn[prob]) { c->tdep_fn[prob] = nullptr; c->ntdep--; }
  c->prob_pending[prob] = 0;
  return MDS_OK;
}

extern "C" int mds_set_prob_bounds_t(mds_ctx *c, int prob, mds_prob_bounds_t_fn fn, void *user)
{
  if (!c || prob < 0 || prob >= c->nprob || !fn) return MDS_EINVAL;
  const DevProb &pb = c->hprob[prob];
  bool any = false;
  for (int d = 0; d < pb.ndim; d++) any = any || pb.bc_lo[d] == MDS_BC_PROB || pb.bc_hi[d] == MDS_BC_PROB;
  if (!any) return set_err(c, MDS_EINVAL, "problem %d has no PROB side", prob);
  HIPCHK(c, hipStreamSynchronize(c->st));
  if (c->tdep_fn.empty()) {
    c->tdep_fn.assign(c->nprob, nullptr);
    c->tdep_user.assign(c->nprob, nullptr);
    c->tdep_buf.assign((size_t)c->nprob * 12, nullptr);
  }
  for (int d = 0; d < pb.ndim; d++)
    for (int side = 0; side < 2; side++) {
      if ((side ? pb.bc_hi[d] : pb.bc_lo[d]) != MDS_BC_PROB) continue;
      for (int st = 0; st < 2; st++) {
        double *&b = c->tdep_buf[(size_t)prob * 12 + (d * 2 + side) * 2 + st];
        if (!b)
          HIPCHK(c, hipHostMalloc((void **)&b, sizeof(double) * MDS_NG * MDS_SLAB_NV * slab_T(pb, d),
                                  hipHostMallocDefault));
        memset(b, 0, sizeof(double) * MDS_NG * MDS_SLAB_NV * slab_T(pb, d));
      }
    }
  if (!c->tdep_fn[prob]) c->ntdep++;
  c->tdep_fn[prob] = fn;
  c->tdep_user[prob] = user;
  c->prob_pending[prob] = 0;
  return MDS_OK;
}

extern "C" int mds_upload_prims(mds_ctx *c, int prob, const double *prims, int nvars)
{
  if (!c || prob < 0 || prob >= c->nprob || !prims || nvars < 2 + c->nv) return MDS_EINVAL;
  if (c->tab && nvars < 6) return set_err(c, MDS_EINVAL, "a table EOS context needs 6 variables (Ye last)");
  long long nz = c->zstart[prob + 1] - c->zstart[prob];
  long long off = c->zstart[prob];
  HIPCHK(c, hipStreamSynchronize(c->st));
  for (int k = 0; k < c->nstate; k++) {
    if (k >= 2 + c->nv && k < 5) continue;
    const double *src = prims + (size_t)k * nz;
    if (c->precision == MDS_FP32_BULK) {
      std::vector<float> tmp(nz);
      for (long long q = 0; q < nz; q++) tmp[q] = (float)src[q];
      HIPCHK(c, hipMemcpy((float *)c->p[k] + off, tmp.data(), nz * sizeof(float), hipMemcpyHostToDevice));
    } else {
      HIPCHK(c, hipMemcpy((double *)c->p[k] + off, src, nz * sizeof(double), hipMemcpyHostToDevice));
    }
  }
  return MDS_OK;
}

// Most bytes in each half of the pinned staging of downloads.
#define MDS_PIN_BYTES (8LL << 20)

// the variables of `vars` of one problem's state (zones off .. off + nz), one
// after the other, to `out`
template <class R>
__global__ __launch_bounds__(256) void pack_kernel(StateArrays<R> s, long long off, long long nz, unsigned vars,
                                                   R *__restrict__ out)
{
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nz) return;
  for (int k = 0; k < 6; k++)
    if (vars >> k & 1) {
      *(out + q) = s.v[k][off + q];
      out += nz;
    }
}

// The staging of downloads, made by the first one: two halves of the largest
// problem's state, at most MDS_PIN_BYTES each.
static int pin_ready(mds_ctx *c)
{
  if (c->pin) return MDS_OK;
  long long most = 0;
  for (int p = 0; p < c->nprob; p++) most = std::max(most, c->zstart[p + 1] - c->zstart[p]);
  const long long half = std::min(MDS_PIN_BYTES, (long long)(most * c->nstate * rsize(c) + 255) / 256 * 256);
  for (auto &e : c->pin_ev)
    if (!e) HIPCHK(c, hipEventCreateWithFlags(&e, hipEventDisableTiming));
  void *m = nullptr;
  HIPCHK(c, hipHostMalloc(&m, 2 * (size_t)half, hipHostMallocDefault));
  c->pin = (char *)m;
  c->pin_half = half;
  return MDS_OK;
}

// The state of a problem, to the caller's (pageable) array.  A copy to
// pageable memory costs some 12 us whatever its size and one host thread
// widens and writes fresh memory at some 5 GB/s, so a state that fits the
// staging comes over with one kernel that writes its variables there, and a
// larger one in pieces, each of which the host's threads take out while the
// next is on its way.  The kernel takes the pieces over too: the copy engine is
// no faster, and its first use in a context costs 2 ms (the first 512^2 FP64
// state 4.3 ms, 1.9 without it, 0.5 from then on).  300 columns of 3000 zones
// with five variables: 16.8 ms before, 6.7 now; 1024 columns 37 and 21.6 ms,
// 256^3 in FP32 122 and 15.5 ms.
extern "C" int mds_download_prims(mds_ctx *c, int prob, double *prims, int nvars)
{
  if (!c || prob < 0 || prob >= c->nprob || !prims || nvars < 2) return MDS_EINVAL;
  const long long nz = c->zstart[prob + 1] - c->zstart[prob], off = c->zstart[prob];
  const int fp32 = c->precision == MDS_FP32_BULK;
  const size_t rs = rsize(c);
  // the variables the context holds; the others are zero
  unsigned vars = 0;
  int nhave = 0;
  for (int k = 0; k < nvars && k < c->nstate; k++)
    if (k < 2 + c->nv || k >= 5) {
      vars |= 1u << k;
      nhave++;
    }
  const int rc = pin_ready(c);
  if (rc) return rc;
  const auto fetch = [&](long long o, long long n, unsigned v, char *to) {
    const dim3 g((unsigned)((n + 255) / 256)), b(256);
    if (fp32) hipLaunchKernelGGL(pack_kernel<float>, g, b, 0, c->st, arrays<float>(c->p), o, n, v, (float *)to);
    else hipLaunchKernelGGL(pack_kernel<double>, g, b, 0, c->st, arrays<double>(c->p), o, n, v, (double *)to);
    return hipGetLastError();
  };
  const bool whole = nhave * nz * (long long)rs <= c->pin_half;
  if (whole) HIPCHK(c, fetch(off, nz, vars, c->pin));
  // while the state is on its way
  for (int k = 0; k < nvars; k++)
    if (k >= 6 || !(vars >> k & 1)) memset(prims + (size_t)k * nz, 0, (size_t)nz * sizeof(double));
  if (whole) {
    HIPCHK(c, hipStreamSynchronize(c->st));
    const char *s = c->pin;
    for (int k = 0; k < 6; k++)
      if (vars >> k & 1) {
        mds_stage_out(prims + (size_t)k * nz, s, fp32, nz);
        s += (size_t)nz * rs;
      }
    return MDS_OK;
  }
  const long long piece = c->pin_half / (long long)rs;
  double *dst = nullptr;                // the piece that is on its way
  long long m = 0;
  int h = 0;
  for (int k = 0; k < 6; k++) {
    if (!(vars >> k & 1)) continue;
    for (long long q = 0; q < nz; q += piece) {
      const long long mn = std::min(piece, nz - q);
      HIPCHK(c, fetch(off + q, mn, 1u << k, c->pin + h * c->pin_half));
      HIPCHK(c, hipEventRecord(c->pin_ev[h], c->st));
      if (dst) {
        HIPCHK(c, hipEventSynchronize(c->pin_ev[h ^ 1]));
        mds_stage_out(dst, c->pin + (h ^ 1) * c->pin_half, fp32, m);
      }
      dst = prims + (size_t)k * nz + q;
      m = mn;
      h ^= 1;
    }
  }
  HIPCHK(c, hipEventSynchronize(c->pin_ev[h ^ 1]));
  mds_stage_out(dst, c->pin + (h ^ 1) * c->pin_half, fp32, m);
  return MDS_OK;
}

extern "C" int mds_update_eos(mds_ctx *c)
{
  if (!c) return MDS_EINVAL;
  std::vector<DevClock> ck(c->nprob);
  for (int p = 0; p < c->nprob; p++) {
    memset(&ck[p], 0, sizeof(DevClock));
    ck[p].t = 0.0;
    ck[p].dt = 0.0;
    ck[p].dtold = 1.0e100;
    ck[p].tmax = c->tmax;
    ck[p].mindt = (unsigned long long)0x7FF0000000000000ull;   // +inf until the zone pass
    ck[p].istep = 0;
    ck[p].active = 1;
  }
  // estimate_dt's first call starts from min_dt = 1e100 (step.c:171-174)
  {
    double big = 1.0e100;
    unsigned long long k;
    memcpy(&k, &big, sizeof(k));
    for (int p = 0; p < c->nprob; p++) ck[p].mindt = k;
  }
  HIPCHK(c, hipMemcpyAsync(c->dclock, ck.data(), sizeof(DevClock) * c->nprob, hipMemcpyHostToDevice, c->st));
  HIPCHK(c, hipMemsetAsync(c->dcount, 0, 4 * sizeof(unsigned long long), c->st));
  dim3 block(256), grid((unsigned)((c->nzone + 255) / 256));
  if (c->precision == MDS_FP32_BULK) {
    hipLaunchKernelGGL(init_dt_kernel<float>, grid, block, 0, c->st, c->dprob, c->dclock, c->dzstart, c->nprob,
                       arrays<float>(c->p), c->tab, c->deos);
  } else {
    hipLaunchKernelGGL(init_dt_kernel<double>, grid, block, 0, c->st, c->dprob, c->dclock, c->dzstart,
                       c->nprob, arrays<double>(c->p), c->tab, c->deos);
  }
  HIPCHK(c, hipGetLastError());
  HIPCHK(c, hipStreamSynchronize(c->st));
  return MDS_OK;
}

// one RK stage of every problem: the fused sweep kernel
static int enqueue_stage(mds_ctx *c, int stage, int fp32)
{
  if (c->has_slab) {
    for (int p = 0; p < c->nprob; p++)
      if (c->prob_pending[p]) return set_err(c, MDS_EINVAL, "problem %d: PROB boundary values not set", p);
    // ghost layers of the PROB/EXTRAP sides from the stage's input state
    void *const *in = stage == 0 ? c->p : c->ph;
    HIPCHK(c, mds_launch_slab_fill(fp32, c->dprob, c->nprob, c->slab_items, in, &c->deos, c->tab, c->nv, c->st));
  }
  if (c->ndim == 1) {
    Sweep1DArgs a;
    a.zpl = 1;
    a.fold = -1;
    a.clock2 = nullptr;
    a.mind = nullptr;
    a.seg = c->dseg;
    a.nseg = c->nseg;
    a.prob = c->dprob;
    a.clock = c->dclock;
    a.counters = c->dcount;
    a.rp = c->rp;
    a.eos = c->deos;
    a.grav = c->dgrav;
    a.ncu = c->ncu;
    a.persist = c->grid1d;
    a.gen = c->has_slab || c->hprob[0].order != 3;
    if (fp32) {
      StateArrays<float> sp = arrays<float>(c->p), sh = arrays<float>(c->ph);
      // monopole field of the stage input state (gravity.c:145-251 at p_to_phys_src_start)
      if (c->mono)
        HIPCHK(c, mds_launch_monopole(1, c->mono, c->tab, c->nprob, c->nmax1d, c->dprob, c->dclock, &c->deos,
                                      stage == 0 ? &sp : &sh, c->dgrav, c->st));
      HIPCHK(c, mds_launch_sweep1d(1, c->nv, c->sph, c->tab, c->mono, &a, &sp, &sh, stage, c->st));
    } else {
      StateArrays<double> sp = arrays<double>(c->p), sh = arrays<double>(c->ph);
      if (c->mono)
        HIPCHK(c, mds_launch_monopole(0, c->mono, c->tab, c->nprob, c->nmax1d, c->dprob, c->dclock, &c->deos,
                                      stage == 0 ? &sp : &sh, c->dgrav, c->st));
      HIPCHK(c, mds_launch_sweep1d(0, c->nv, c->sph, c->tab, c->mono, &a, &sp, &sh, stage, c->st));
    }
  } else if (c->sph3) {
    c->s3.flags = c->dflags;
    if (fp32) {
      StateArrays<float> sp = arrays<float>(c->p), sh = arrays<float>(c->ph);
      HIPCHK(c, mds_launch_sph3d(&c->s3, &c->hprob[0], c->dclock, c->dcount, &c->deos, &sp, &sh, stage, c->st));
    } else {
      StateArrays<double> sp = arrays<double>(c->p), sh = arrays<double>(c->ph);
      HIPCHK(c, mds_launch_sph3d(&c->s3, &c->hprob[0], c->dclock, c->dcount, &c->deos, &sp, &sh, stage, c->st));
    }
  } else if (c->ndim == 3) {
    Sweep3DArgs a;
    const DevProb &h = c->hprob[0];
    a.prob = c->dprob;
    a.clock = c->dclock;
    a.counters = c->dcount;
    a.flags = c->dflags;
    a.nstrip = (h.n[0] + MDS_SEG1D - 1) / MDS_SEG1D;
    a.ntile = (h.n[1] + c->ty3d - 1) / c->ty3d;
    a.chunk = c->kc3d;
    a.nchunk = (h.n[2] + a.chunk - 1) / a.chunk;
    a.src = (h.g0[0] != 0.0 || h.g0[1] != 0.0 || h.g0[2] != 0.0);
    a.slab = c->has_slab || h.order != 3;     // the general instances: ghost layers, low orders
    if (fp32) {
      StateArrays<float> sp = arrays<float>(c->p), sh = arrays<float>(c->ph);
      HIPCHK(c, mds_launch_sweep3d(1, c->ty3d, c->halo3d, &a, &sp, &sh, stage, c->st));
    } else {
      StateArrays<double> sp = arrays<double>(c->p), sh = arrays<double>(c->ph);
      HIPCHK(c, mds_launch_sweep3d(0, c->ty3d, c->halo3d, &a, &sp, &sh, stage, c->st));
    }
  } else {
    Sweep2DArgs a;
    a.prob = c->dprob;
    a.clock = c->dclock;
    a.counters = c->dcount;
    a.flags = c->dflags;
    a.chunk = c->chunk2d;
    a.nstrip = (c->hprob[0].n[0] + MDS_SEG1D - 1) / MDS_SEG1D;
    a.nchunk = (c->hprob[0].n[1] + a.chunk - 1) / a.chunk;
    a.src = (c->hprob[0].g0[0] != 0.0 || c->hprob[0].g0[1] != 0.0 || c->hprob[0].g0[2] != 0.0);
    a.slab = c->has_slab || c->hprob[0].order != 3;     // the general instances: ghost layers, low orders
    if (fp32) {
      StateArrays<float> sp = arrays<float>(c->p), sh = arrays<float>(c->ph);
      HIPCHK(c, mds_launch_sweep2d(1, c->nv, &a, &sp, &sh, stage, c->st));
    } else {
      StateArrays<double> sp = arrays<double>(c->p), sh = arrays<double>(c->ph);
      HIPCHK(c, mds_launch_sweep2d(0, c->nv, &a, &sp, &sh, stage, c->st));
    }
  }
  return MDS_OK;
}

// both RK stages of every 1D problem in one launch: p -> ph (the caller swaps)
static int enqueue_fused1d(mds_ctx *c, int fold = -1)
{
  Sweep1DArgs a;
  a.fold = fold;
  a.clock2 = c->dclock2;
  a.mind = c->dmind;
  a.zpl = c->fuse1d == 2 ? 2 : 1;
  a.seg = a.zpl == 2 ? c->dseg3 : c->dseg2;
  a.nseg = a.zpl == 2 ? c->nseg3 : c->nseg2;
  a.prob = c->dprob;
  a.clock = c->dclock;
  a.counters = c->dcount;
  a.rp = c->rp;
  a.eos = c->deos;
  a.grav = nullptr;
  a.ncu = c->ncu;
  a.persist = c->grid1d;
  a.gen = 0;                  // two-stage instances are plain (order 3, no ghost layers)
  int fp32 = c->precision == MDS_FP32_BULK;
  if (fp32) {
    StateArrays<float> sp = arrays<float>(c->p), sh = arrays<float>(c->ph);
    HIPCHK(c, mds_launch_sweep1d(1, c->nv, c->sph, c->tab, 0, &a, &sp, &sh, -1, c->st));
  } else {
    StateArrays<double> sp = arrays<double>(c->p), sh = arrays<double>(c->ph);
    HIPCHK(c, mds_launch_sweep1d(0, c->nv, c->sph, c->tab, 0, &a, &sp, &sh, -1, c->st));
  }
  return MDS_OK;
}

// after a two-stage launch the new state is in ph: swap the buffer names
static void finish_step(mds_ctx *c)
{
  if (!c->fuse1d) return;
  for (int k = 0; k < 6; k++) std::swap(c->p[k], c->ph[k]);
  c->par ^= 1;
}

static void enqueue_dt(mds_ctx *c)
{
  hipLaunchKernelGGL(dt_policy_kernel, dim3((c->nprob + 127) / 128), dim3(128), 0, c->st, c->dclock, c->nprob,
                     c->rp);
}

// estimate_dt + dt policy, then step(): two RK stages (step.c:28-129);
// the kernels only (the caller runs finish_step once they are enqueued)
static int enqueue_step_kernels(mds_ctx *c)
{
  int fp32 = c->precision == MDS_FP32_BULK;
  enqueue_dt(c);
  HIPCHK(c, hipGetLastError());
  if (c->fuse1d) return enqueue_fused1d(c);
  for (int stage = 0; stage < 2; stage++) {
    int rc = enqueue_stage(c, stage, fp32);
    if (rc) return rc;
  }
  return MDS_OK;
}

static int enqueue_step(mds_ctx *c)
{
  int rc = enqueue_step_kernels(c);
  if (rc == MDS_OK) finish_step(c);
  return rc;
}

// Whether this context's two-stage steps run folded: a batch whose wavefronts
// the device holds at once (16 per compute unit) waits for its steps' launches,
// not for issue slots.  There the dt launch costs more than the policy in
// every wavefront (a tube of 3001 zones in FP32 16.0 us a step with it, 6.8
// folded and replayed; 820 wavefronts of FP64 columns 17.5 and 16.5 us); with
// several rounds of wavefronts the policy costs more (1024 columns 115.0 and
// 116.6 us, 300 rotating ones 49.1 and 50.1 us).
static bool folds(const mds_ctx *c)
{
  return c->fuse1d && (c->fuse1d == 2 ? c->nseg3 : c->nseg2) <= 16 * std::max(1, c->ncu);
}

// A group of MDS_FOLD two-stage column steps without a dt launch between them
// (mds_clock.h); the buffers' names end as they began.
static int enqueue_group(mds_ctx *c)
{
  for (int f = 0; f < MDS_FOLD; f++) {
    const int rc = enqueue_fused1d(c, f);
    if (rc) {
      if (f & 1) finish_step(c);          // the names of the last whole pair of steps
      return rc;
    }
    finish_step(c);
  }
  return MDS_OK;
}

// One step of a context with time-dependent PROB hooks: the dt policy on
// the device and a wait for it, the hooks on the host at the times the
// reference's fills see (t and t + dt, bc.c:717-721), and their values
// copied in on the stream before each stage's ghost-layer refill.
static int step_tdep(mds_ctx *c)
{
  const int fp32 = c->precision == MDS_FP32_BULK;
  std::vector<DevClock> ck0(c->nprob), ck1(c->nprob);
  HIPCHK(c, hipStreamSynchronize(c->st));
  HIPCHK(c, hipMemcpy(ck0.data(), c->dclock, sizeof(DevClock) * c->nprob, hipMemcpyDeviceToHost));
  enqueue_dt(c);
  HIPCHK(c, hipGetLastError());
  HIPCHK(c, hipMemcpyAsync(ck1.data(), c->dclock, sizeof(DevClock) * c->nprob, hipMemcpyDeviceToHost, c->st));
  HIPCHK(c, hipStreamSynchronize(c->st));
  auto buf = [&](int p, int d, int side, int st) { return c->tdep_buf[(size_t)p * 12 + (d * 2 + side) * 2 + st]; };
  for (int p = 0; p < c->nprob; p++) {
    if (!c->tdep_fn[p] || !ck1[p].active) continue;
    const double tt[2] = {ck0[p].t, ck0[p].t + ck1[p].dt};
    for (int st = 0; st < 2; st++)
      prob_fill_host(c, p, [&](int i, int j, int k, double *q) { c->tdep_fn[p](i, j, k, tt[st], q, c->tdep_user[p]); },
                     [&](int d, int side) { return buf(p, d, side, st); });
  }
  for (int stage = 0; stage < 2; stage++) {
    for (int p = 0; p < c->nprob; p++) {
      if (!c->tdep_fn[p] || !ck1[p].active) continue;
      const DevProb &pb = c->hprob[p];
      for (int d = 0; d < pb.ndim; d++)
        for (int side = 0; side < 2; side++)
          if ((side ? pb.bc_hi[d] : pb.bc_lo[d]) == MDS_BC_PROB)
            HIPCHK(c, hipMemcpyAsync(pb.gs[d][side], buf(p, d, side, stage),
                                     sizeof(double) * MDS_NG * MDS_SLAB_NV * slab_T(pb, d), hipMemcpyHostToDevice,
                                     c->st));
    }
    int rc = enqueue_stage(c, stage, fp32);
    if (rc) return rc;
  }
  finish_step(c);
  return MDS_OK;
}

#define MDS_GRAPH_GROUPS 4     // groups of folded steps in one graph

extern "C" int mds_run(mds_ctx *c, int nsteps)
{
  if (!c || nsteps < 0) return MDS_EINVAL;
  if (c->ntdep > 0) {
    for (int s = 0; s < nsteps; s++) {
      int rc = step_tdep(c);
      if (rc) return rc;
    }
    return MDS_OK;
  }
  int s = 0;
  for (; folds(c) && s + MDS_FOLD <= nsteps; s += MDS_FOLD) {
    int rc = enqueue_group(c);
    if (rc) return rc;
  }
  for (; s < nsteps; s++) {
    int rc = enqueue_step(c);
    if (rc) return rc;
  }
  return MDS_OK;
}

extern "C" int mds_run_graph(mds_ctx *c, int nsteps)
{
  if (!c || nsteps < 0) return MDS_EINVAL;
  if (c->ntdep > 0) return mds_run(c, nsteps);     // host hooks between the stages: no graph
  // launch graph k, captured first if it is new
  auto replay = [&](int k, auto enqueue) -> int {
    if (!c->gexec[k]) {
      HIPCHK(c, hipStreamBeginCapture(c->st, hipStreamCaptureModeThreadLocal));
      c->s3.serial = 1;
      int rc = enqueue();
      c->s3.serial = 0;
      hipGraph_t g = nullptr;
      hipError_t e = hipStreamEndCapture(c->st, &g);
      if (rc) { if (g) hipGraphDestroy(g); return rc; }
      if (e != hipSuccess) return set_err(c, MDS_EDEVICE, "graph capture failed: %s", hipGetErrorString(e));
      c->graph[k] = g;
      HIPCHK(c, hipGraphInstantiate(&c->gexec[k], c->graph[k], nullptr, nullptr, 0));
    }
    HIPCHK(c, hipGraphLaunch(c->gexec[k], c->st));
    return MDS_OK;
  };
  // one graph per buffer parity: the two-stage 1D step alternates p and ph.
  // A launch of a graph takes the host some 16 us whatever it holds, which
  // is a whole step of a small batch: folded steps replay MDS_GRAPH_GROUPS
  // groups at a time.
  const int par = c->fuse1d ? c->par : 0;
  int s = 0;
  for (; folds(c) && s + MDS_FOLD * MDS_GRAPH_GROUPS <= nsteps; s += MDS_FOLD * MDS_GRAPH_GROUPS) {
    int rc = replay(2 + par, [&]() -> int {
      for (int g = 0; g < MDS_GRAPH_GROUPS; g++) {
        const int r1 = enqueue_group(c);
        if (r1) return r1;
      }
      return MDS_OK;
    });
    if (rc) return rc;
  }
  for (; s < nsteps; s++) {
    int rc = replay(c->fuse1d ? c->par : 0, [&]() -> int { return enqueue_step_kernels(c); });
    if (rc) return rc;
    finish_step(c);
  }
  return MDS_OK;
}

extern "C" int mds_run_timed(mds_ctx *c, int nsteps, double ms[3])
{
  if (!c || nsteps < 1 || !ms) return MDS_EINVAL;
  if (c->ntdep > 0) return set_err(c, MDS_EINVAL, "time-dependent PROB hooks step with mds_run only");
  std::vector<hipEvent_t> ev(3 * (size_t)nsteps + 1, nullptr);
  int rc = MDS_OK;
  for (auto &e : ev) {
    if (hipEventCreate(&e) != hipSuccess) { rc = set_err(c, MDS_EDEVICE, "hipEventCreate failed"); break; }
  }
  if (rc == MDS_OK) {
    int fp32 = c->precision == MDS_FP32_BULK;
    hipError_t e = hipEventRecord(ev[0], c->st);
    for (int s = 0; s < nsteps && e == hipSuccess && rc == MDS_OK; s++) {
      enqueue_dt(c);
      if (c->fuse1d) {
        // one two-stage launch: ms[1] gets its duration, ms[2] stays ~0
        e = hipEventRecord(ev[3 * s + 1], c->st);
        if (e == hipSuccess) rc = enqueue_fused1d(c);
        if (e == hipSuccess && rc == MDS_OK) e = hipEventRecord(ev[3 * s + 2], c->st);
        if (e == hipSuccess && rc == MDS_OK) finish_step(c);
      } else {
        for (int stage = 0; stage < 2 && e == hipSuccess; stage++) {
          e = hipEventRecord(ev[3 * s + 1 + stage], c->st);
          if (e != hipSuccess) break;
          rc = enqueue_stage(c, stage, fp32);
          if (rc) break;
        }
      }
      if (e == hipSuccess && rc == MDS_OK) e = hipEventRecord(ev[3 * s + 3], c->st);
    }
    if (e == hipSuccess && rc == MDS_OK) e = hipEventSynchronize(ev[3 * (size_t)nsteps]);
    if (e != hipSuccess && rc == MDS_OK) rc = set_err(c, MDS_EDEVICE, "timed run: %s", hipGetErrorString(e));
    if (rc == MDS_OK) {
      float f = 0.0f;
      double tot[3] = {0.0, 0.0, 0.0};
      hipEventElapsedTime(&f, ev[0], ev[3 * (size_t)nsteps]);
      tot[0] = f;
      for (int s = 0; s < nsteps; s++) {
        hipEventElapsedTime(&f, ev[3 * s + 1], ev[3 * s + 2]); tot[1] += f;
        hipEventElapsedTime(&f, ev[3 * s + 2], ev[3 * s + 3]); tot[2] += f;
      }
      ms[0] = tot[0]; ms[1] = tot[1]; ms[2] = tot[2];
    }
  }
  for (auto &e : ev) if (e) hipEventDestroy(e);
  return rc;
}

__global__ void copy_probe_kernel(const float4 *__restrict__ src, float4 *__restrict__ dst, long long n)
{
  long long stride = (long long)gridDim.x * blockDim.x;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

extern "C" int mds_copy_probe(long long nbytes, int reps, double *ms)
{
  if (nbytes < 16 || reps < 1 || !ms) return MDS_EINVAL;
  long long n = nbytes / 16;
  float4 *a = nullptr, *b = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  hipError_t e = hipMalloc(&a, n * 16);
  if (e == hipSuccess) e = hipMalloc(&b, n * 16);
  if (e == hipSuccess) e = hipMemset(a, 0, n * 16);
  if (e == hipSuccess) e = hipEventCreate(&e0);
  if (e == hipSuccess) e = hipEventCreate(&e1);
  int dev = 0, ncu = 256;
  hipGetDevice(&dev);
  hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
  dim3 blk(256), grd((unsigned)std::min<long long>((n + 255) / 256, (long long)ncu * 32));
  if (e == hipSuccess) {
    hipLaunchKernelGGL(copy_probe_kernel, grd, blk, 0, 0, a, b, n);   // warm up
    e = hipEventRecord(e0, 0);
  }
  for (int r = 0; r < reps && e == hipSuccess; r++) hipLaunchKernelGGL(copy_probe_kernel, grd, blk, 0, 0, a, b, n);
  if (e == hipSuccess) e = hipEventRecord(e1, 0);
  if (e == hipSuccess) e = hipEventSynchronize(e1);
  float f = 0.0f;
  if (e == hipSuccess) e = hipEventElapsedTime(&f, e0, e1);
  if (e == hipSuccess) *ms = f / reps;
  if (e0) hipEventDestroy(e0);
  if (e1) hipEventDestroy(e1);
  hipFree(a);
  hipFree(b);
  return e == hipSuccess ? MDS_OK : MDS_EDEVICE;
}

// eight independent chains per lane: the VALU issue rate without memory.
// OP 0: fused multiply-add; 1: reciprocal (v_rcp_f32 / v_rcp_f64); 2: square
// root (v_sqrt_f32 / v_sqrt_f64).  The reciprocal and root chains stay
// bounded (x -> 1/x alternates, x -> sqrt(x) tends to 1).
__device__ __forceinline__ float probe_rcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ double probe_rcp(double x) { return __builtin_amdgcn_rcp(x); }
__device__ __forceinline__ float probe_sqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
__device__ __forceinline__ double probe_sqrt(double x) { return __builtin_amdgcn_sqrt(x); }

template <class T, int OP>
__global__ __launch_bounds__(256) void valu_probe_kernel(T *out, int iters, T a, T b)
{
  T x[8];
  for (int k = 0; k < 8; k++) x[k] = (T)(threadIdx.x * 1.0e-3 + k + 1);
  for (int i = 0; i < iters; i++) {
#pragma unroll
    for (int k = 0; k < 8; k++) {
      if constexpr (OP == 0) x[k] = fma(x[k], a, b);   // one v_fma per chain (the library builds with contraction off)
      else if constexpr (OP == 1) x[k] = probe_rcp(x[k]);
      else x[k] = probe_sqrt(x[k]);
    }
  }
  T s = 0;
  for (int k = 0; k < 8; k++) s += x[k];
  out[(long long)blockIdx.x * blockDim.x + threadIdx.x] = s;
}

template <class T, int OP>
static hipError_t valu_probe(int reps, double *rate)
{
  int dev = 0, ncu = 256;
  hipGetDevice(&dev);
  hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
  const int blocks = ncu * 16, iters = OP == 0 ? 4000 : 1000;
  T *d = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  hipError_t e = hipMalloc(&d, sizeof(T) * (size_t)blocks * 256);
  if (e == hipSuccess) e = hipEventCreate(&e0);
  if (e == hipSuccess) e = hipEventCreate(&e1);
  if (e == hipSuccess) hipLaunchKernelGGL((valu_probe_kernel<T, OP>), dim3(blocks), dim3(256), 0, 0, d, iters, (T)0.999, (T)1e-3);
  if (e == hipSuccess) e = hipEventRecord(e0, 0);
  for (int r = 0; r < reps && e == hipSuccess; r++)
    hipLaunchKernelGGL((valu_probe_kernel<T, OP>), dim3(blocks), dim3(256), 0, 0, d, iters, (T)0.999, (T)1e-3);
  if (e == hipSuccess) e = hipEventRecord(e1, 0);
  if (e == hipSuccess) e = hipEventSynchronize(e1);
  float f = 0.0f;
  if (e == hipSuccess) e = hipEventElapsedTime(&f, e0, e1);
  if (e == hipSuccess) *rate = (double)blocks * 4.0 * iters * 8.0 * reps / (f * 1.0e-3);
  if (e0) hipEventDestroy(e0);
  if (e1) hipEventDestroy(e1);
  if (d) hipFree(d);
  return e;
}

extern "C" int mds_valu_probe(int kind, int reps, double *wave_instr_per_s)
{
  if (reps < 1 || !wave_instr_per_s || kind < 0 || kind > 5) return MDS_EINVAL;
  hipError_t e = hipSuccess;
  switch (kind) {
    case 0: e = valu_probe<float, 0>(reps, wave_instr_per_s); break;
    case 1: e = valu_probe<double, 0>(reps, wave_instr_per_s); break;
    case 2: e = valu_probe<float, 1>(reps, wave_instr_per_s); break;
    case 3: e = valu_probe<double, 1>(reps, wave_instr_per_s); break;
    case 4: e = valu_probe<float, 2>(reps, wave_instr_per_s); break;
    default: e = valu_probe<double, 2>(reps, wave_instr_per_s); break;
  }
  return e == hipSuccess ? MDS_OK : MDS_EDEVICE;
}

// 3D Cartesian problems on the general sweep instances (one tile shape)
static bool gen3d(const mds_ctx *c)
{
  return c->ndim == 3 && !c->sph3 && (c->has_slab || c->hprob[0].order != 3);
}

extern "C" int mds_set_tile(mds_ctx *c, int param, int value)
{
  if (!c) return MDS_EINVAL;
  int *slot = nullptr;
  if (param == MDS_TILE_ROWS2D) {
    if (value < 1 || value > 4096) return set_err(c, MDS_EINVAL, "rows per wavefront out of range: %d", value);
    slot = &c->chunk2d;
  } else if (param == MDS_TILE_TY3D) {
    if (value != 4 && value != 8 && value != 12)
      return set_err(c, MDS_EINVAL, "3D tile rows must be 4, 8 or 12: %d", value);
    if (value != 4 && gen3d(c))
      return set_err(c, MDS_EINVAL, "3D problems with PROB/EXTRAP sides or hydro_interp_order < 3 run 4-row tiles");
    slot = &c->ty3d;
  } else if (param == MDS_TILE_KC3D) {
    if (value < 1 || value > 4096) return set_err(c, MDS_EINVAL, "planes per workgroup out of range: %d", value);
    slot = &c->kc3d;
  } else if (param == MDS_TILE_FUSE1D) {
    if (value < 0 || value > 2) return set_err(c, MDS_EINVAL, "two-stage 1D switch must be 0, 1 or 2: %d", value);
    if (value && !c->can_fuse1d)
      return set_err(c, MDS_EINVAL, "the two-stage 1D kernel needs 1D problems without periodic x boundaries");
    if (value == 2 && c->precision != MDS_FP32_BULK)
      return set_err(c, MDS_EINVAL, "two zones per lane is an FP32-bulk launch shape");
    slot = &c->fuse1d;
  } else if (param == MDS_TILE_HALO3D) {
    if (value != 0 && value != 1) return set_err(c, MDS_EINVAL, "3D halo mode must be 0 or 1: %d", value);
    if (value && gen3d(c))
      return set_err(c, MDS_EINVAL,
                     "3D problems with PROB/EXTRAP sides or hydro_interp_order < 3 run the halo-wavefront tile");
    slot = &c->halo3d;
  } else if (param == MDS_TILE_GRID1D) {
    if (value != 0 && value != 1) return set_err(c, MDS_EINVAL, "1D grid mode must be 0 or 1: %d", value);
    slot = &c->grid1d;
  } else if (param == MDS_TILE_UPD3S) {
    if (value < 0 || value > 3) return set_err(c, MDS_EINVAL, "spherical update shape must be 0 to 3: %d", value);
    slot = &c->s3.upd;
  } else {
    return set_err(c, MDS_EINVAL, "unknown tile parameter %d", param);
  }
  if (*slot != value) {
    *slot = value;
    drop_graphs(c);
  }
  return MDS_OK;
}

extern "C" int mds_get_tile(mds_ctx *c, int param, int *value)
{
  if (!c || !value) return MDS_EINVAL;
  if (param == MDS_TILE_ROWS2D) { *value = c->chunk2d; return MDS_OK; }
  if (param == MDS_TILE_TY3D) { *value = c->ty3d; return MDS_OK; }
  if (param == MDS_TILE_KC3D) { *value = c->kc3d; return MDS_OK; }
  if (param == MDS_TILE_FUSE1D) { *value = c->fuse1d; return MDS_OK; }
  if (param == MDS_TILE_GRID1D) { *value = c->grid1d; return MDS_OK; }
  if (param == MDS_TILE_HALO3D) { *value = c->halo3d; return MDS_OK; }
  if (param == MDS_TILE_UPD3S) { *value = c->s3.upd; return MDS_OK; }
  return set_err(c, MDS_EINVAL, "unknown tile parameter %d", param);
}

// save/restore of the evolving device state around autotuning trials
struct Snapshot {
  std::vector<void *> buf;
  void *clock = nullptr, *count = nullptr, *flags = nullptr;
  void *gr = nullptr, *grst = nullptr;     // GR monopole blocks (Gamma warm start) and state
};

static void snap_free(Snapshot &s)
{
  for (void *b : s.buf) hipFree(b);
  s.buf.clear();
  if (s.clock) hipFree(s.clock);
  if (s.count) hipFree(s.count);
  if (s.flags) hipFree(s.flags);
  if (s.gr) hipFree(s.gr);
  if (s.grst) hipFree(s.grst);
  s.clock = s.count = s.flags = s.gr = s.grst = nullptr;
}

static int snap_alloc(mds_ctx *c, Snapshot &s)
{
  size_t bytes = (size_t)c->nzone * rsize(c);
  for (int k = 0; k < 2 * c->nstate; k++) {
    void *b = nullptr;
    HIPCHK(c, hipMalloc(&b, bytes));
    s.buf.push_back(b);
  }
  HIPCHK(c, hipMalloc(&s.clock, sizeof(DevClock) * c->nprob));
  HIPCHK(c, hipMalloc(&s.count, 4 * sizeof(unsigned long long)));
  if (c->dflags) HIPCHK(c, hipMalloc(&s.flags, (size_t)c->nzone));
  if (c->dgr) {
    HIPCHK(c, hipMalloc(&s.gr, sizeof(double) * c->gr_doubles));
    HIPCHK(c, hipMalloc(&s.grst, sizeof(int) * 4 * c->nprob));
  }
  return MDS_OK;
}

// save = true: context -> snapshot; false: snapshot -> context
static int snap_copy(mds_ctx *c, Snapshot &s, bool save)
{
  size_t bytes = (size_t)c->nzone * rsize(c);
  for (int k = 0; k < c->nstate; k++) {
    void *dst = save ? s.buf[k] : c->p[k], *src = save ? c->p[k] : s.buf[k];
    HIPCHK(c, hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, c->st));
    dst = save ? s.buf[c->nstate + k] : c->ph[k];
    src = save ? c->ph[k] : s.buf[c->nstate + k];
    HIPCHK(c, hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, c->st));
  }
  HIPCHK(c, hipMemcpyAsync(save ? s.clock : (void *)c->dclock, save ? (void *)c->dclock : s.clock,
                           sizeof(DevClock) * c->nprob, hipMemcpyDeviceToDevice, c->st));
  HIPCHK(c, hipMemcpyAsync(save ? s.count : (void *)c->dcount, save ? (void *)c->dcount : s.count,
                           4 * sizeof(unsigned long long), hipMemcpyDeviceToDevice, c->st));
  if (c->dflags)
    HIPCHK(c, hipMemcpyAsync(save ? s.flags : (void *)c->dflags, save ? (void *)c->dflags : s.flags,
                             (size_t)c->nzone, hipMemcpyDeviceToDevice, c->st));
  if (c->dgr) {
    HIPCHK(c, hipMemcpyAsync(save ? s.gr : (void *)c->dgr, save ? (void *)c->dgr : s.gr,
                             sizeof(double) * c->gr_doubles, hipMemcpyDeviceToDevice, c->st));
    HIPCHK(c, hipMemcpyAsync(save ? s.grst : (void *)c->dgrst, save ? (void *)c->dgrst : s.grst,
                             sizeof(int) * 4 * c->nprob, hipMemcpyDeviceToDevice, c->st));
  }
  HIPCHK(c, hipStreamSynchronize(c->st));
  return MDS_OK;
}

extern "C" int mds_autotune(mds_ctx *c, int nsteps, double *best_ms)
{
  if (!c || nsteps < 1) return MDS_EINVAL;
  // fixed shapes: contexts whose time-dependent PROB hooks run on the host
  // every step
  if (c->ntdep > 0) { if (best_ms) *best_ms = 0.0; return MDS_OK; }
  // candidates: (a, b, c) = 1D (two-stage launch, persistent grid, -);
  // 2D (rows per wavefront, -, -); 3D (rows per workgroup, planes, halo mode);
  // 2D/3D spherical (update workgroup shape, -, -)
  struct Shape { int a, b, c; };
  std::vector<Shape> cand;
  if (c->sph3) {
    for (int v : {0, 1, 2, 3}) cand.push_back({v, 0, 0});
  } else if (c->ndim == 1) {
    for (int g : {0, 1}) {
      cand.push_back({0, g, 0});
      if (c->can_fuse1d) cand.push_back({1, g, 0});
      if (c->can_fuse1d && c->precision == MDS_FP32_BULK) cand.push_back({2, g, 0});
    }
  } else if (c->ndim == 2) {
    // the rows whose cost is near the least
    for (int v : rows2d)
      if (v <= c->hprob[0].n[1] && cost2d(c, v) <= 1.15 * cost2d(c, rows_for(c))) cand.push_back({v, 0, 0});
  } else {
    // problems with PROB/EXTRAP ghost layers have one tile shape (4 rows,
    // halo wavefronts); only the planes per workgroup vary
    for (int hs : {0, 1})
      for (int ty : {4, 8, 12}) {
        if (gen3d(c) && (ty != 4 || hs)) continue;
        const double least = cost3d(c, ty, planes_for(c, ty, hs), hs);
        for (int kc : planes3d)
          if (kc <= c->hprob[0].n[2] && cost3d(c, ty, kc, hs) <= 1.15 * least) cand.push_back({ty, kc, hs});
      }
  }
  auto apply = [&](const Shape &v) {
    if (c->sph3) c->s3.upd = v.a;
    else if (c->ndim == 1) { c->fuse1d = v.a; c->grid1d = v.b; }
    else if (c->ndim == 2) c->chunk2d = v.a;
    else { c->ty3d = v.a; c->kc3d = v.b; c->halo3d = v.c; }
  };
  Snapshot s;
  int rc = snap_alloc(c, s);
  if (rc == MDS_OK) rc = snap_copy(c, s, true);
  Shape best = c->sph3 ? Shape{c->s3.upd, 0, 0}
               : c->ndim == 1 ? Shape{c->fuse1d, c->grid1d, 0}
               : c->ndim == 2 ? Shape{c->chunk2d, 0, 0} : Shape{c->ty3d, c->kc3d, c->halo3d};
  double bms = 1e300;
  for (const Shape &v : cand) {
    if (rc) break;
    apply(v);
    double ms[3];
    rc = mds_run_timed(c, 1, ms);      // warm the shape
    // best of two timed runs from the same state, each of half a millisecond at
    // least: one run of a few steps is at the mercy of clock ramps and other
    // work on the device
    int n = nsteps;
    while (rc == MDS_OK && n * ms[0] < 0.5 && n < 64) n *= 2;
    double t = 1e300;
    for (int rep = 0; rep < 2 && rc == MDS_OK; rep++) {
      rc = snap_copy(c, s, false);
      if (rc == MDS_OK) rc = mds_run_timed(c, n, ms);
      if (rc == MDS_OK && ms[0] < t) t = ms[0];
    }
    if (rc == MDS_OK && t / n < bms) { bms = t / n; best = v; }
    if (rc == MDS_OK) rc = snap_copy(c, s, false);
  }
  snap_free(s);
  apply(best);
  drop_graphs(c);
  if (best_ms) *best_ms = bms;
  return rc;
}

extern "C" int mds_sync(mds_ctx *c)
{
  if (!c) return MDS_EINVAL;
  HIPCHK(c, hipStreamSynchronize(c->st));
  return MDS_OK;
}

extern "C" int mds_get_clock(mds_ctx *c, int prob, double *t, double *dt, int *istep)
{
  if (!c || prob < 0 || prob >= c->nprob) return MDS_EINVAL;
  DevClock ck;
  HIPCHK(c, hipStreamSynchronize(c->st));
  HIPCHK(c, hipMemcpy(&ck, c->dclock + prob, sizeof(ck), hipMemcpyDeviceToHost));
  if (t) *t = ck.t;
  if (dt) *dt = ck.dt;
  if (istep) *istep = ck.istep;
  if (ck.status) return set_err(c, MDS_EINVAL, "problem %d: dt dropped below dtmin", prob);
  return MDS_OK;
}

extern "C" int mds_get_health(mds_ctx *c, int prob, mds_health *out)
{
  if (!c || prob < 0 || prob >= c->nprob || !out) return MDS_EINVAL;
  DevClock ck;
  HIPCHK(c, hipStreamSynchronize(c->st));
  HIPCHK(c, hipMemcpy(&ck, c->dclock + prob, sizeof(ck), hipMemcpyDeviceToHost));
  out->t = ck.t;
  out->dt = ck.dt;
  out->istep = ck.istep;
  out->dt_below_min = ck.status;
  out->bad_state = (long long)ck.nbad;
  out->eos_off_table = (long long)ck.noff;
  // the running CFL minimum of the step being taken: a NaN limit never wins
  // the bitwise minimum, so a NaN state shows here only through bad_state
  return MDS_OK;
}

extern "C" int mds_get_gr_state(mds_ctx *c, int prob, double *gtov, double *mr, double *lapse_edge,
                                double *lapse, int *passes, int *nonconverged)
{
  if (!c || prob < 0 || prob >= c->nprob) return MDS_EINVAL;
  if (c->mono != MDS_MONOPOLE_GR) return set_err(c, MDS_EINVAL, "no GR monopole in this context");
  const DevProb &pb = c->hprob[prob];
  const size_t N = (size_t)pb.n[0] + 1;
  HIPCHK(c, hipStreamSynchronize(c->st));
  std::vector<double> h((size_t)MDS_GR_COUNT * N);
  int st[4];
  HIPCHK(c, hipMemcpy(h.data(), pb.gr, sizeof(double) * h.size(), hipMemcpyDeviceToHost));
  HIPCHK(c, hipMemcpy(st, pb.grst, sizeof(st), hipMemcpyDeviceToHost));
  if (gtov) memcpy(gtov, &h[MDS_GR_GTOV * N], sizeof(double) * N);
  if (mr) memcpy(mr, &h[MDS_GR_MR * N], sizeof(double) * N);
  if (lapse_edge) memcpy(lapse_edge, &h[MDS_GR_LAPSE_E * N], sizeof(double) * N);
  if (lapse) memcpy(lapse, &h[MDS_GR_LAPSE * N], sizeof(double) * (N - 1));
  if (passes) *passes = st[1];
  if (nonconverged) *nonconverged = st[2];
  return MDS_OK;
}

extern "C" int mds_counters(mds_ctx *c, long long out[2])
{
  if (!c || !out) return MDS_EINVAL;
  unsigned long long h[4];
  HIPCHK(c, hipStreamSynchronize(c->st));
  HIPCHK(c, hipMemcpy(h, c->dcount, sizeof(h), hipMemcpyDeviceToHost));
  out[0] = (long long)h[0];
  out[1] = (long long)h[1];
  return MDS_OK;
}

// Block partials of the totals of problem prob into dpart (device, 4 doubles
// per block) and back into h (host), on the context stream, synchronised.
hipError_t mds_totals_partials(mds_ctx *c, int prob, int nblk, double *dpart, double *h)
{
  const long long nz = c->zstart[prob + 1] - c->zstart[prob];
  if (c->precision == MDS_FP32_BULK)
    hipLaunchKernelGGL(totals_kernel<float>, dim3(nblk), dim3(256), 0, c->st, c->dprob, prob, nz, c->nv,
                       arrays<float>(c->p), dpart);
  else
    hipLaunchKernelGGL(totals_kernel<double>, dim3(nblk), dim3(256), 0, c->st, c->dprob, prob, nz, c->nv,
                       arrays<double>(c->p), dpart);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpyAsync(h, dpart, sizeof(double) * 4 * nblk, hipMemcpyDeviceToHost, c->st);
  if (e == hipSuccess) e = hipStreamSynchronize(c->st);
  return e;
}

// accessors for the other translation units of the library
int mds_ctx_device(const mds_ctx *c) { return c->dev; }
int mds_ctx_check_prob(mds_ctx *c, int prob)
{
  return (prob < 0 || prob >= c->nprob) ? set_err(c, MDS_EINVAL, "problem %d out of range", prob) : MDS_OK;
}
int mds_ctx_error(mds_ctx *c, int code, const char *msg) { return set_err(c, code, "%s", msg); }

// Neumaier sum of the block partials, in block order
void mds_totals_finish(const double *h, int nblk, double out[2])
{
  for (int k = 0; k < 2; k++) {
    double S = 0.0, C = 0.0;
    for (int b = 0; b < nblk; b++)
      for (int m = 0; m < 2; m++) {
        double v = h[4 * b + 2 * k + m];
        double t = S + v;
        if (fabs(S) >= fabs(v)) C += (S - t) + v; else C += (v - t) + S;
        S = t;
      }
    out[k] = S + C;
  }
}

extern "C" int mds_conserved_totals(mds_ctx *c, int prob, double out[2])
{
  if (!c || prob < 0 || prob >= c->nprob || !out) return MDS_EINVAL;
  long long nz = c->zstart[prob + 1] - c->zstart[prob];
  int nblk = 256;
  double *dpart = nullptr;
  HIPCHK(c, hipMalloc(&dpart, sizeof(double) * 4 * nblk));
  std::vector<double> h(4 * nblk);
  hipError_t e = mds_totals_partials(c, prob, nblk, dpart, h.data());
  hipFree(dpart);
  if (e != hipSuccess) return set_err(c, MDS_EDEVICE, "totals: %s", hipGetErrorString(e));
  mds_totals_finish(h.data(), nblk, out);
  return MDS_OK;
}

// ---------------------------------------------------------------------------
// pointwise parity entry points
// ---------------------------------------------------------------------------
__global__ void recon_points_x64(int n, const double *a, const double *mom, const double *x, double *al,
                                 double *ar)
{
  int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  ReconGeo64 g;
  g.am = mom[9 * c + 0]; g.bm = mom[9 * c + 1]; g.gm = mom[9 * c + 2];
  g.a0 = mom[9 * c + 3]; g.b0 = mom[9 * c + 4]; g.g0 = mom[9 * c + 5];
  g.ap = mom[9 * c + 6]; g.bp = mom[9 * c + 7]; g.gp = mom[9 * c + 8];
  g.xlo = x[2 * c];
  g.xhi = x[2 * c + 1];
  recon_geo_x64(g);
  g.y0 = drcp(g.g0);
  para_recon_x64(a[3 * c], a[3 * c + 1], a[3 * c + 2], g, al[c], ar[c]);
}

__global__ void recon_points_f32(int n, const double *a, const double *rc, double *al, double *ar)
{
  int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  ReconGeo32 g;
  const double *r = rc + (size_t)c * MDS_RC_COUNT;
  g.clm = (float)r[MDS_RC_CLM]; g.clp = (float)r[MDS_RC_CLP]; g.crm = (float)r[MDS_RC_CRM];
  g.crp = (float)r[MDS_RC_CRP]; g.mu1 = (float)r[MDS_RC_MU1]; g.kinv = (float)r[MDS_RC_KINV];
  g.inur = (float)r[MDS_RC_INUR]; g.imu2 = (float)r[MDS_RC_IMU2];
  float l, rr;
  para_recon_f32((float)a[3 * c], (float)a[3 * c + 1], (float)a[3 * c + 2], g, l, rr);
  al[c] = l;
  ar[c] = rr;
}

template <class R>
__global__ void riemann_points(int solver, int n, const double *pl, const double *pr, const double *fg, int dir,
                               double *flux, double *sig, int *shock)
{
  int f = blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= n) return;
  PState<R, 3> L, Rt;
  L.rho = (R)pl[7 * f + 0]; L.uu = (R)pl[7 * f + 1];
  L.v[0] = (R)pl[7 * f + 2]; L.v[1] = (R)pl[7 * f + 3]; L.v[2] = (R)pl[7 * f + 4];
  L.P = (R)pl[7 * f + 5]; L.G = (R)pl[7 * f + 6];
  Rt.rho = (R)pr[7 * f + 0]; Rt.uu = (R)pr[7 * f + 1];
  Rt.v[0] = (R)pr[7 * f + 2]; Rt.v[1] = (R)pr[7 * f + 3]; Rt.v[2] = (R)pr[7 * f + 4];
  Rt.P = (R)pr[7 * f + 5]; Rt.G = (R)pr[7 * f + 6];
  FaceGeo<R> g;
  g.area = (R)fg[5 * f + 0];
  g.scale = (R)fg[5 * f + 1];
  g.gcov[0] = (R)fg[5 * f + 2]; g.gcov[1] = (R)fg[5 * f + 3]; g.gcov[2] = (R)fg[5 * f + 4];
  int sh = 0;
  if constexpr (sizeof(R) == 8) {
    double F[5], s;
    if (solver == 0) sh = hllc_x64<3, false>(L, Rt, g, dir, F, s);
    else hlle_x64<3, false>(L, Rt, g, dir, F, s);
    for (int q = 0; q < 5; q++) flux[5 * f + q] = F[q];
    sig[f] = s;
  } else {
    float F[5] = {0, 0, 0, 0, 0}, s = 0.0f;
    FaceGeo<float> g1 = g;
    g1.area = 1.0f;
    if (g.area < 1.0e-16f) { for (int q = 0; q < 5; q++) F[q] = 0.0f; s = 1.0e-30f; }
    else if (solver == 0) sh = hllc_f32<3, false>(L, Rt, g1, dir, F, s);
    else hlle_f32<3, false>(L, Rt, g1, dir, F, s);
    for (int q = 0; q < 5; q++) flux[5 * f + q] = fg[5 * f + 0] * (double)F[q];
    sig[f] = s;
  }
  shock[f] = sh;
}

template <class T>
static hipError_t dcopy(T **d, const T *h, size_t n)
{
  hipError_t e = hipMalloc((void **)d, n * sizeof(T) + 8);
  if (e != hipSuccess) return e;
  if (h) e = hipMemcpy(*d, h, n * sizeof(T), hipMemcpyHostToDevice);
  return e;
}

extern "C" int mds_recon_points(int precision, int ncell, const double *a, const double *mom, const double *x,
                                const double *rcoef, double *al, double *ar)
{
  if (ncell <= 0 || !a || !al || !ar) return MDS_EINVAL;
  double *da = nullptr, *dm = nullptr, *dx = nullptr, *drc = nullptr, *dl = nullptr, *dr = nullptr;
  hipError_t e = dcopy(&da, a, 3 * (size_t)ncell);
  if (e == hipSuccess) e = dcopy(&dl, (const double *)nullptr, (size_t)ncell);
  if (e == hipSuccess) e = dcopy(&dr, (const double *)nullptr, (size_t)ncell);
  dim3 b(128), g((ncell + 127) / 128);
  if (e == hipSuccess) {
    if (precision == MDS_FP64) {
      if (!mom || !x) e = hipErrorInvalidValue;
      if (e == hipSuccess) e = dcopy(&dm, mom, 9 * (size_t)ncell);
      if (e == hipSuccess) e = dcopy(&dx, x, 2 * (size_t)ncell);
      if (e == hipSuccess) hipLaunchKernelGGL(recon_points_x64, g, b, 0, 0, ncell, da, dm, dx, dl, dr);
    } else {
      if (!rcoef) e = hipErrorInvalidValue;
      if (e == hipSuccess) e = dcopy(&drc, rcoef, (size_t)MDS_RC_COUNT * ncell);
      if (e == hipSuccess) hipLaunchKernelGGL(recon_points_f32, g, b, 0, 0, ncell, da, drc, dl, dr);
    }
  }
  if (e == hipSuccess) e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpy(al, dl, ncell * sizeof(double), hipMemcpyDeviceToHost);
  if (e == hipSuccess) e = hipMemcpy(ar, dr, ncell * sizeof(double), hipMemcpyDeviceToHost);
  hipFree(da); hipFree(dm); hipFree(dx); hipFree(drc); hipFree(dl); hipFree(dr);
  return e == hipSuccess ? MDS_OK : MDS_EDEVICE;
}

extern "C" int mds_riemann_points(int precision, int solver, int nface, const double *pl, const double *pr,
                                  const double *fg, int dir, double *flux, double *sig, int *isshock)
{
  if (nface <= 0 || !pl || !pr || !fg || !flux || !sig || !isshock || dir < 0 || dir > 2) return MDS_EINVAL;
  double *dpl = nullptr, *dpr = nullptr, *dfg = nullptr, *dfl = nullptr, *dsg = nullptr;
  int *dsh = nullptr;
  hipError_t e = dcopy(&dpl, pl, 7 * (size_t)nface);
  if (e == hipSuccess) e = dcopy(&dpr, pr, 7 * (size_t)nface);
  if (e == hipSuccess) e = dcopy(&dfg, fg, 5 * (size_t)nface);
  if (e == hipSuccess) e = dcopy(&dfl, (const double *)nullptr, 5 * (size_t)nface);
  if (e == hipSuccess) e = dcopy(&dsg, (const double *)nullptr, (size_t)nface);
  if (e == hipSuccess) e = dcopy(&dsh, (const int *)nullptr, (size_t)nface);
  dim3 b(128), g((nface + 127) / 128);
  if (e == hipSuccess) {
    if (precision == MDS_FP64)
      hipLaunchKernelGGL(riemann_points<double>, g, b, 0, 0, solver, nface, dpl, dpr, dfg, dir, dfl, dsg, dsh);
    else
      hipLaunchKernelGGL(riemann_points<float>, g, b, 0, 0, solver, nface, dpl, dpr, dfg, dir, dfl, dsg, dsh);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpy(flux, dfl, 5 * (size_t)nface * sizeof(double), hipMemcpyDeviceToHost);
  if (e == hipSuccess) e = hipMemcpy(sig, dsg, (size_t)nface * sizeof(double), hipMemcpyDeviceToHost);
  if (e == hipSuccess) e = hipMemcpy(isshock, dsh, (size_t)nface * sizeof(int), hipMemcpyDeviceToHost);
  hipFree(dpl); hipFree(dpr); hipFree(dfg); hipFree(dfl); hipFree(dsg); hipFree(dsh);
  return e == hipSuccess ? MDS_OK : MDS_EDEVICE;
}

// ---------------------------------------------------------------------------
// allocation-free pointwise Riemann solve
// ---------------------------------------------------------------------------
// The staging of mds_riemann_points (its inputs and outputs on the device)
// lives in this file-scope array instead of per-call hipMalloc: per face,
// 7 + 7 + 5 doubles in (pl, pr, fg), 5 + 1 doubles out (flux, sig), and one
// int (isshock) in the tail.  Every GPU holds its own copy, at its own
// address, until the process ends.  In host code the name `scratch` is a
// host-side stand-in: only the address from hipGetSymbolAddress (kept per
// device in noalloc_ptr) may reach a kernel or a copy.
namespace {
constexpr int NOALLOC_DOUBLES_PER_FACE = 7 + 7 + 5 + 5 + 1;
constexpr size_t NOALLOC_BYTES =
    (size_t)MDS_NOALLOC_MAX_FACES * (NOALLOC_DOUBLES_PER_FACE * sizeof(double) + sizeof(int));
}  // namespace

static __device__ __align__(256) double scratch[NOALLOC_BYTES / sizeof(double)];

namespace {
constexpr int NOALLOC_MAX_DEVICES = 64;
double *noalloc_ptr[NOALLOC_MAX_DEVICES];
std::atomic<int> noalloc_lock{0};

// The device address of `scratch` on the current device, resolved once per
// device (with that device current) and kept.
hipError_t noalloc_scratch(double **out)
{
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= NOALLOC_MAX_DEVICES) return hipErrorInvalidDevice;
  while (noalloc_lock.exchange(1, std::memory_order_acquire)) {
  }
  if (!noalloc_ptr[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e == hipSuccess) noalloc_ptr[dev] = (double *)p;
  }
  *out = noalloc_ptr[dev];
  noalloc_lock.store(0, std::memory_order_release);
  return (e == hipSuccess && !*out) ? hipErrorInvalidSymbol : e;
}
}  // namespace

extern "C" int mds_riemann_points_noalloc(int precision, int solver, int nface, const double *pl, const double *pr,
                                          const double *fg, int dir, double *flux, double *sig, int *isshock)
{
  if (nface <= 0 || !pl || !pr || !fg || !flux || !sig || !isshock || dir < 0 || dir > 2) return MDS_EINVAL;
  if (nface > MDS_NOALLOC_MAX_FACES) return MDS_ERANGE;
  double *base = nullptr;
  hipError_t e = noalloc_scratch(&base);
  if (e != hipSuccess) return MDS_EDEVICE;
  const size_t n = (size_t)nface;
  // regions sized for nface faces, packed from the start of the array;
  // every output element is written by the kernel, so nothing needs clearing
  double *dpl = base, *dpr = dpl + 7 * n, *dfg = dpr + 7 * n, *dfl = dfg + 5 * n, *dsg = dfl + 5 * n;
  int *dsh = (int *)(dsg + n);
  e = hipMemcpy(dpl, pl, 7 * n * sizeof(double), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(dpr, pr, 7 * n * sizeof(double), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(dfg, fg, 5 * n * sizeof(double), hipMemcpyHostToDevice);
  dim3 b(128), g((nface + 127) / 128);
  if (e == hipSuccess) {
    if (precision == MDS_FP64)
      hipLaunchKernelGGL(riemann_points<double>, g, b, 0, 0, solver, nface, dpl, dpr, dfg, dir, dfl, dsg, dsh);
    else
      hipLaunchKernelGGL(riemann_points<float>, g, b, 0, 0, solver, nface, dpl, dpr, dfg, dir, dfl, dsg, dsh);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpy(flux, dfl, 5 * n * sizeof(double), hipMemcpyDeviceToHost);
  if (e == hipSuccess) e = hipMemcpy(sig, dsg, n * sizeof(double), hipMemcpyDeviceToHost);
  if (e == hipSuccess) e = hipMemcpy(isshock, dsh, n * sizeof(int), hipMemcpyDeviceToHost);
  return e == hipSuccess ? MDS_OK : MDS_EDEVICE;
}
