// Vector-Jacobian product of the interior residual on gfx950.
//
// Given a cotangent w(nshg,4) (same layout as res), computes
//   ybar  = w^T d res / d y      (nshg,4), y = (u1,u2,u3,p)
//   acbar = w^T d res / d ac     (nshg,4), ac = (a1,a2,a3, unused), optional
//   mubar = w^T d res / d mu     (scalar)
// for res the interior ElmGMR residual that crimson_form_interior returns
// (flux pass, e3 with itau = 0 and iconvflow = 2, scatter; before bc3Res).
// The derivative is the exact one of the formulation as written (no lazy
// tangent): tauM and tauC through u (e3stab.f90:108-133), tauBar and ubar
// through the strong residual L (e3stab.f90:356-374), and the reconstructed
// flux q through qpbc's lumped projection of mu (grad u + grad u^T)
// (e3q.f90:100-145, qpbc.f90:67-71).  The acceleration enters the momentum
// residual's rNa and the strong residual L (e3res.f90:775-789), both with
// factor rho.
//
// Reverse mode written by hand and deterministic (no atomics):
//   vjp_e3_elem    element: recompute each quadrature point forward, then
//                  back-propagate the element's residual cotangent; writes
//                  ybar (and acbar) for its four nodes, the cotangent of its
//                  divergence of q, and its workgroup's mubar part
//   vjp_q_node     node: qbar from its elements' divergence cotangents, times
//                  1/rmass (the adjoint of q = qres / rmass)
//   vjp_node       node: ybar gathered over the incidences in element order,
//                  with the adjoint of the lumped projection (the elements'
//                  flux cotangents sum_a m_a qbar_a / rmass_a, back to u)
//   mu_final       the workgroups' mubar parts summed in a fixed order

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "form_common.hpp"

namespace {

// Element records.  kVRecY: per node a its ybar at 4 a; kVRecYA: per node its
// ybar and acbar at 8 a (the eighth unused).  kVRecD: the cotangent of
// the element's divergence of q.
constexpr int kVRecY = 16, kVRecYA = 32, kVRecD = 4;
// Packed x and qbar of a node, 10 doubles (x, qbar, one unused).
constexpr int kXQ = 10;
constexpr int kVjpLanes = 8;   // lanes per node
constexpr int kVjpUnroll = 3;  // records in flight per lane (three on a Kuhn mesh's 24 incidences)
constexpr int kVjpCap = 20;    // neighbours staged per row by vjp_q_node
constexpr int kVjpCap2 = 16;   // by vjp_node: 40 KB a workgroup, four workgroups in a CU's LDS (three with 20: 15 us more)

// The forward sums are e3_elem's; what does not vary over the element is
// kept out of the loop over the quadrature points here as well.  With V = -W sum_a
// w_a g_a^T the cotangent of the flux sum (constant), per point: rLb = tauM V u
// + V^T lg - ..., the cotangents of u and a through the point's value (uq, aq,
// overwriting the nodal u and a), and gub^T += aqb u^T + (lgrb - tauM rnab) L^T.
// The rule's weights (one at the point's own node, another at the rest) give
// sum_q N_a(q) f_q = w_other(a) sum f + w_diff(a) f_a.  The records are staged in
// LDS and stored as one block per workgroup, coalesced.  Bound by latency at two
// waves a SIMD, as e3_elem.  1.7 M elements: 470 us with every point's terms written
// out and 448-byte records stored per thread, 186 so.
// What a point does not need is parked in LDS (a thread's own slots, bank-conflict
// free): a and w of the nodes (a's place takes its cotangent) and g.  Kept in
// registers they spilled 250 bytes a lane.
constexpr int kVThreads = 128;
constexpr int kVPark = 33, VP_A = 0, VP_W = 12, VP_G = 24;
// The value is computed by here (the compiler would put the sums of one point off
// to the next ones, and hold their terms).
__device__ inline void settle(double &x) { asm volatile("" : "+v"(x)); }
template <bool AC>
__global__ void __launch_bounds__(kVThreads) __attribute__((amdgpu_waves_per_eu(2)))
vjp_e3_elem(int nel, const int *__restrict__ ien, const double *__restrict__ node, const double *__restrict__ w,
            int nshg, FormConst c0, Ens en, double *__restrict__ vrec, double *__restrict__ vdq,
            double *__restrict__ part) {
  constexpr int kR = AC ? kVRecYA : kVRecY, kPad = kR + 1, kA = kR / 4;
  __shared__ double sh_rec[kVThreads * kVPark];  // parked values, then the records
  static_assert(kPad <= kVPark && kVPark % 2 == 1, "");
  __shared__ double sh_mu[kVThreads / 64];
  const int blk = xcd_block(64u);
  const int e0 = blk * kVThreads, e = e0 + threadIdx.x;
  const int ee = e < nel ? e : nel - 1;  // tail threads evaluate a valid element; nothing of theirs is stored
  const double mu = ens_mu(en, ee, c0.mu);
  const FormConst &c = c0;
  const size_t N = nshg;
  double *pk = sh_rec + threadIdx.x * kVPark;
  double ul[4][3], V[3][3], SUb[3];
  double W, gg[6], gu[3][3], gpd[3], as[3], ws[3];
  {
    double xl[4][3], al[4][3], wl[4][3], pl[4], ql[4][6], w3[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const int nd = ien[a * (size_t)nel + ee];
      double nl[kNRec];
      load_record(node + (size_t)nd * kNRec, nl);
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        xl[a][i] = nl[N_X + i];
        ul[a][i] = nl[N_U + i];
        al[a][i] = nl[N_A + i];
        wl[a][i] = w[nd + N * i];
      }
      w3[a] = w[nd + N * 3];
      pl[a] = nl[N_P];
#pragma unroll
      for (int k = 0; k < 6; ++k) ql[a][k] = nl[N_Q + k];
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      as[i] = w_other(0) * (al[0][i] + al[1][i] + al[2][i]) + w_other(3) * al[3][i];
#pragma unroll
      for (int a = 0; a < 4; ++a) pk[VP_A + 3 * a + i] = al[a][i];
    }
    __builtin_amdgcn_sched_barrier(0);
    double dx[3][3], g4[4][3];
    p1_metric(xl, dx, W, g4);
    gijd_tet(dx, gg);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 3; ++j)
      gpd[j] = g4[0][j] * pl[0] + g4[1][j] * pl[1] + g4[2][j] * pl[2] + g4[3][j] * pl[3];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int i = 0; i < 3; ++i)
        gpd[i] -= g4[a][0] * ql[a][qsym(i)] + g4[a][1] * ql[a][qsym(i + 3)] + g4[a][2] * ql[a][qsym(i + 6)];
    __builtin_amdgcn_sched_barrier(0);
    // cotangents of the element sums: rl_a,i = -W (RNa_ai + g_a . RGN_i:),
    // rl_a,4 = W g_a . SU
#pragma unroll
    for (int i = 0; i < 3; ++i) {
#pragma unroll
      for (int j = 0; j < 3; ++j)
        V[i][j] = -W * (wl[0][i] * g4[0][j] + wl[1][i] * g4[1][j] + wl[2][i] * g4[2][j] + wl[3][i] * g4[3][j]);
      SUb[i] = W * (w3[0] * g4[0][i] + w3[1] * g4[1][i] + w3[2] * g4[2][i] + w3[3] * g4[3][i]);
      ws[i] = w_other(0) * (wl[0][i] + wl[1][i] + wl[2][i]) + w_other(3) * wl[3][i];
#pragma unroll
      for (int a = 0; a < 4; ++a) pk[VP_W + 3 * a + i] = wl[a][i];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        gu[j][i] = g4[0][j] * ul[0][i] + g4[1][j] * ul[1][i] + g4[2][j] * ul[2][i] + g4[3][j] * ul[3][i];
        pk[VP_G + 3 * i + j] = g4[i][j];
      }
  }
  wave_lds_sync();  // (keeps the compiler from holding the parked values)
  const double rho = c.rho, rhoinv = 1.0 / rho, rnu = mu * rhoinv;
  const double dts = c.Dtgl * c.dtsfct;
  const double GG = gg[0] * gg[0] + gg[1] * gg[1] + gg[2] * gg[2] +
                    2.0 * (gg[3] * gg[3] + gg[4] * gg[4] + gg[5] * gg[5]);
  const double tau0 = (2.0 * dts) * (2.0 * dts) + 36.0 * (rnu * rnu) * GG;
  const double tc = rho * 0.125 / (gg[0] + gg[1] + gg[2]) * (c.taucfct / c.dtsfct);  // tauC = tc fact
  const double divu = gu[0][0] + gu[1][1] + gu[2][2];
  const double trV = V[0][0] + V[1][1] + V[2][2];
  double us[3], gpb[3], gub[3][3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    us[i] = w_other(0) * (ul[0][i] + ul[1][i] + ul[2][i]) + w_other(3) * ul[3][i];
    gpb[i] = 0.0;
#pragma unroll
    for (int j = 0; j < 3; ++j) gub[j][i] = 0.0;
  }
  double sf = 0.0, Sbs = 0.0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    // forward, as in e3_elem
    double u[3], aq[3], L[3], Gu[3], GL[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      u[i] = us[i] + w_diff(q) * ul[q][i];
      aq[i] = as[i] + w_diff(q) * pk[VP_A + 3 * q + i];
    }
#pragma unroll
    for (int i = 0; i < 3; ++i)
      L[i] = (aq[i] + u[0] * gu[0][i] + u[1] * gu[1][i] + u[2] * gu[2][i]) * rho + gpd[i];
    Gu[0] = gg[0] * u[0] + gg[3] * u[1] + gg[5] * u[2];
    Gu[1] = gg[3] * u[0] + gg[1] * u[1] + gg[4] * u[2];
    Gu[2] = gg[5] * u[0] + gg[4] * u[1] + gg[2] * u[2];
    GL[0] = gg[0] * L[0] + gg[3] * L[1] + gg[5] * L[2];
    GL[1] = gg[3] * L[0] + gg[1] * L[1] + gg[4] * L[2];
    GL[2] = gg[5] * L[0] + gg[4] * L[1] + gg[2] * L[2];
    const double s2 = tau0 + (u[0] * Gu[0] + u[1] * Gu[1] + u[2] * Gu[2]);
    const double tauM = rsqrt(s2);
    sf += s2 * tauM;
    const double sL = L[0] * GL[0] + L[1] * GL[1] + L[2] * GL[2];
    const double isq = (sL != 0.0) ? rsqrt(sL) : 0.0;
    const double tauB = tauM * isq;
    // backward.  rna_i = (aq_i + ub . grad u_i) rho; ub = u - tauM L / rho;
    // v_ij = mu (gu_ij + gu_ji) + tauM L_i u_j + tauB lgr_i L_j + delta_ij (-p +
    // tauC div u), lgr_i = L . grad u_i
    double rnab[3], ubb[3], lgrb[3], rLb[3];
    double tMb = 0.0, tBb = 0.0;
#pragma unroll
    for (int i = 0; i < 3; ++i) rnab[i] = -W * (ws[i] + w_diff(q) * pk[VP_W + 3 * q + i]);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      ubb[i] = SUb[i] + rho * (gu[i][0] * rnab[0] + gu[i][1] * rnab[1] + gu[i][2] * rnab[2]);
      const double vu = V[i][0] * u[0] + V[i][1] * u[1] + V[i][2] * u[2];
      const double vl = V[i][0] * L[0] + V[i][1] * L[1] + V[i][2] * L[2];
      const double lgr = L[0] * gu[0][i] + L[1] * gu[1][i] + L[2] * gu[2][i];
      tMb += L[i] * (vu - ubb[i] * rhoinv);
      rLb[i] = tauM * (vu - ubb[i] * rhoinv);
      tBb += vl * lgr;
      lgrb[i] = tauB * vl;
      aq[i] = tauB * lgr;  // lg_i
    }
    // tauB = tauM (L G L)^(-1/2)
    tMb += tBb * isq;
    const double sLb = -tBb * tauB * (isq * isq);
    // tauM = 1 / fact, tauC = tc fact, fact = sqrt(tau0 + uGu)
    const double Sb = 0.5 * tauM * (trV * divu * tc - tMb * tauM * tauM);
    Sbs += Sb;
#pragma unroll
    for (int k = 0; k < 3; ++k)
      rLb[k] += (V[0][k] * aq[0] + V[1][k] * aq[1] + V[2][k] * aq[2]) +
                (gu[k][0] * lgrb[0] + gu[k][1] * lgrb[1] + gu[k][2] * lgrb[2]) + sLb * GL[k];
    // L_i = (a_i + u . grad u_i) rho + dp/dx_i - (div q)_i
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const double uq = ubb[j] + tauM * (V[0][j] * L[0] + V[1][j] * L[1] + V[2][j] * L[2]) + 2.0 * Sb * Gu[j] +
                        rho * (gu[j][0] * rLb[0] + gu[j][1] * rLb[1] + gu[j][2] * rLb[2]);
      gpb[j] += rLb[j];
      pk[VP_W + 3 * q + j] = uq;
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const double ab = rho * (rnab[i] + rLb[i]);  // the acceleration's cotangent: rna and L, each times rho
      const double lb = lgrb[i] - tauM * rnab[i];
#pragma unroll
      for (int j = 0; j < 3; ++j) gub[j][i] += ab * u[j] + lb * L[j];
      if (AC) pk[VP_A + 3 * q + i] = ab;
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) {
#pragma unroll
      for (int j = 0; j < 3; ++j) settle(gub[j][i]);
      settle(gpb[i]);
    }
    settle(sf);
    settle(Sbs);
    wave_lds_sync();
  }
  double mub = Sbs * (72.0 * rnu * rhoinv * GG), vg = 0.0;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      gub[i][j] += 4.0 * mu * (V[i][j] + V[j][i]);
      vg += V[i][j] * (gu[i][j] + gu[j][i]);
    }
    gub[i][i] += trV * (tc * sf);
  }
  mub += 4.0 * vg;
  double g[3][3], al[4][3], uqs[3], aqs[3], gs[3] = {0, 0, 0};
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      al[a][i] = AC ? pk[VP_A + 3 * a + i] : 0.0;
      ul[a][i] = pk[VP_W + 3 * a + i];
      if (a < 3) g[a][i] = pk[VP_G + 3 * a + i];
    }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    uqs[i] = (ul[0][i] + ul[1][i]) + (ul[2][i] + ul[3][i]);
    aqs[i] = (al[0][i] + al[1][i]) + (al[2][i] + al[3][i]);
  }
  __syncthreads();  // the parked values are read: the records take their place
  double *r = sh_rec + threadIdx.x * kPad;
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    double ga[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      ga[j] = a < 3 ? g[a < 3 ? a : 0][j] : -gs[j];
      gs[j] += ga[j];
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      r[kA * a + i] = w_other(a) * uqs[i] + w_diff(a) * ul[a][i] +
                      (ga[0] * gub[0][i] + ga[1] * gub[1][i] + ga[2] * gub[2][i]);
      if (AC) r[kA * a + 4 + i] = w_other(a) * aqs[i] + w_diff(a) * al[a][i];
    }
    r[kA * a + 3] = -trV * sum_n(a) + (ga[0] * gpb[0] + ga[1] * gpb[1] + ga[2] * gpb[2]);
    if (AC) r[kA * a + 7] = 0.0;
  }
  if (e < nel) {
    double2 *d = reinterpret_cast<double2 *>(vdq + (size_t)e * kVRecD);
    d[0] = make_double2(-gpb[0], -gpb[1]);
    d[1] = make_double2(-gpb[2], 0.0);
  }
  const double ms = block_sum<kVThreads>(e < nel ? mub : 0.0, sh_mu);  // (its barrier also orders the records)
  if (threadIdx.x == 0) part[blk] = ms;
  const int cnt = min(kVThreads, nel - e0);
  constexpr int kH = kR / 2;
  double2 *dst = reinterpret_cast<double2 *>(vrec + (size_t)e0 * kR);
  for (int i = threadIdx.x; i < cnt * kH; i += kVThreads) {
    const double *src = sh_rec + (i / kH) * kPad + 2 * (i % kH);
    dst[i] = make_double2(src[0], src[1]);
  }
}

// g of the element's own node from the four nodes' x (o: the other three in
// local order), and W = WdetJ, whose sign takes the own node's local number n.
__device__ inline double own_gradient(const double (&xa)[3], const double (&x0)[3], const double (&x1)[3],
                                      const double (&x2)[3], int n, double (&g)[3]) {
  double e[3], e0[3], e1[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    e[i] = xa[i] - x2[i];
    e0[i] = x0[i] - x2[i];
    e1[i] = x1[i] - x2[i];
  }
  const double c[3] = {e0[1] * e1[2] - e0[2] * e1[1], e0[2] * e1[0] - e0[0] * e1[2], e0[0] * e1[1] - e0[1] * e1[0]};
  const double det = e[0] * c[0] + e[1] * c[1] + e[2] * c[2], inv = 1.0 / det;
#pragma unroll
  for (int i = 0; i < 3; ++i) g[i] = c[i] * inv;
  return (n & 1 ? -0.125 * kQwt : 0.125 * kQwt) * det;
}

// qbar at the nodes: g_a (x) the element's divergence cotangent, symmetrised,
// summed over the node's incidences (fixed lanes and shuffle tree), times
// 1/rmass; written with the node's x as its packed record.  The gradient is rebuilt
// from the row's coordinates (staged in LDS) rather than read: an element then
// passes 32 bytes on instead of 192.  306 k nodes: 167 us from the records, 65 so.
template <class IL>
__global__ void __launch_bounds__(256) vjp_q_node(int nshg, const int *__restrict__ rowptr,
                                                  const int *__restrict__ diagk, const int *__restrict__ col,
                                                  const int *__restrict__ inc_ptr, const int *__restrict__ inc,
                                                  const IL *__restrict__ iloc, const double *__restrict__ xu,
                                                  const double *__restrict__ vdq, const double *__restrict__ invm,
                                                  double *__restrict__ xq) {
  __shared__ double xs_all[256 / kVjpLanes][kVjpCap * 4];
  const unsigned gid = xcd_block() * blockDim.x + threadIdx.x;
  const int i = (int)(gid / kVjpLanes), lane = (int)(gid % kVjpLanes);
  const bool live = i < nshg;
  const int ii = live ? i : nshg - 1;
  const int k0 = rowptr[ii], ns = rowptr[ii + 1] - k0, d = diagk[ii] - k0;
  const int p0 = inc_ptr[ii], p1 = live ? inc_ptr[ii + 1] : p0;
  double *xs = xs_all[threadIdx.x / kVjpLanes];
  auto get = [&](int s, double (&x)[3]) {
    const double *r = xs + 4 * min(s, kVjpCap - 1);
#pragma unroll
    for (int j = 0; j < 3; ++j) x[j] = r[j];
    if (s >= kVjpCap) {
      const double *m = xu + (size_t)col[k0 + s] * kXU;
#pragma unroll
      for (int j = 0; j < 3; ++j) x[j] = m[j];
    }
  };
  double s[6] = {0, 0, 0, 0, 0, 0}, xa[3];
  bool staged = false;
  int p = p0 + lane;
  do {
    IL il[kVjpUnroll];
    double2 r[kVjpUnroll][2];
#pragma unroll
    for (int u = 0; u < kVjpUnroll; ++u) {
      const int pu = max(min(p + kVjpLanes * u, p1 - 1), 0);
      il[u] = iloc[pu];
      const double2 *q = reinterpret_cast<const double2 *>(vdq + (size_t)(inc[pu] >> 2) * kVRecD);
      r[u][0] = q[0];
      r[u][1] = q[1];
    }
    if (!staged) {
      stage_row<kVjpLanes, kVjpCap, 2, kXU>(lane, k0, ns, col, xu, xs);
      wave_lds_sync();
      get(d, xa);
      staged = true;
    }
#pragma unroll
    for (int u = 0; u < kVjpUnroll; ++u)
      if (p + kVjpLanes * u < p1) {
        int o[3];
        IncLoc<IL>::others(il[u], o);
        double x0[3], x1[3], x2[3], g[3];
        get(o[0], x0);
        get(o[1], x1);
        get(o[2], x2);
        own_gradient(xa, x0, x1, x2, 0, g);
        const double d0 = r[u][0].x, d1 = r[u][0].y, d2 = r[u][1].x;
        s[0] += g[0] * d0;
        s[1] += g[1] * d0 + g[0] * d1;
        s[2] += g[2] * d0 + g[0] * d2;
        s[3] += g[1] * d1;
        s[4] += g[2] * d1 + g[1] * d2;
        s[5] += g[2] * d2;
      }
    p += kVjpLanes * kVjpUnroll;
  } while (p < p1);
#pragma unroll
  for (int off = 1; off < kVjpLanes; off <<= 1)
#pragma unroll
    for (int k = 0; k < 6; ++k) s[k] += __shfl_xor(s[k], off, kVjpLanes);
  if (!live || lane >= kXQ / 2) return;
  const double m = invm[i];
  double2 v;
  switch (lane) {
    case 0: v = make_double2(xa[0], xa[1]); break;
    case 1: v = make_double2(xa[2], m * s[0]); break;
    case 2: v = make_double2(m * s[1], m * s[2]); break;
    case 3: v = make_double2(m * s[3], m * s[4]); break;
    default: v = make_double2(m * s[5], 0.0); break;
  }
  reinterpret_cast<double2 *>(xq + (size_t)i * kXQ)[lane] = v;
}

// ybar (and, with AC, acbar) at the nodes, (nshg,4) column-major like res;
// acbar's fourth column is zero.  Sums the node's element records and, from the
// row's staged x and qbar, the adjoint of the lumped projection: the element's
// viscous flux qdi = mu (grad u + grad u^T) (elem_flux's slots
// 11,12,13,22,23,33) enters q at its nodes with weight m_a / rmass, so with Q =
// sum_a m_a qbar_a as a symmetric form (Q_ij twice on the diagonal) ybar_a gets
// mu t, t = Q g_a, and mubar gets sum_a u_a . t.  306 k nodes: 289 us and 147 us for
// an element pass that wrote 128-byte records for it, 159 so (122 are the records).
template <class IL, bool AC>
__global__ void __launch_bounds__(256) vjp_node(int nshg, const int *__restrict__ rowptr,
                                                const int *__restrict__ diagk, const int *__restrict__ col,
                                                const int *__restrict__ inc_ptr, const int *__restrict__ inc,
                                                const IL *__restrict__ iloc, const double *__restrict__ xu,
                                                const double *__restrict__ xq, const double *__restrict__ vrec,
                                                double mu0, Ens en, double *__restrict__ ybar,
                                                double *__restrict__ acbar, double *__restrict__ part) {
  constexpr int kR = AC ? 8 : 4;  // doubles of a node's record
  constexpr int kP = 4;           // lanes per record (without AC two pairs read the same, so that both sum in one order)
  __shared__ double xs_all[256 / kVjpLanes][kVjpCap2 * kXQ];
  const unsigned blk = xcd_block();
  const unsigned gid = blk * blockDim.x + threadIdx.x;
  const int i = (int)(gid / kVjpLanes), lane = (int)(gid % kVjpLanes);
  const bool live = i < nshg;
  const int ii = live ? i : nshg - 1;
  const int k0 = rowptr[ii], ns = rowptr[ii + 1] - k0, d = diagk[ii] - k0;
  const int p0 = inc_ptr[ii], p1 = live ? inc_ptr[ii + 1] : p0;
  double *xs = xs_all[threadIdx.x / kVjpLanes];
  const double *ur = xu + (size_t)ii * kXU;
  const double ua[3] = {ur[3], ur[4], ur[5]};
  auto get = [&](int s, double (&x)[9]) {
    const double *r = xs + kXQ * min(s, kVjpCap2 - 1);
#pragma unroll
    for (int j = 0; j < 9; ++j) x[j] = r[j];
    if (s >= kVjpCap2) {
      const double *m = xq + (size_t)col[k0 + s] * kXQ;
#pragma unroll
      for (int j = 0; j < 9; ++j) x[j] = m[j];
    }
  };
  // the element records: kP lanes per incidence, 16 bytes each, so that a
  // load takes whole records (a lane per record took a line's tag for 16 bytes)
  constexpr int kG = kVjpLanes / kP;  // incidences per load
  double2 rs = make_double2(0.0, 0.0);
  double t3[3] = {0, 0, 0}, xa[9], mub = 0.0;
  bool staged = false;
  int p = p0;
  stage_row<kVjpLanes, kVjpCap2, kXQ / 2, kXQ>(lane, k0, ns, col, xq, xs);
  do {
    IL il[kVjpUnroll];
    int ea[kVjpUnroll];
#pragma unroll
    for (int u = 0; u < kVjpUnroll; ++u) {
      const int pu = max(min(p + lane + kVjpLanes * u, p1 - 1), 0);
      il[u] = iloc[pu];
      ea[u] = inc[pu];
    }
    double2 r[kVjpUnroll * kP];
#pragma unroll
    for (int v = 0; v < kVjpUnroll * kP; ++v) {
      const int t = v * kG + lane / kP;  // of the 8 kVjpUnroll incidences
      const int ev = __shfl(ea[v / kP], t % kVjpLanes, kVjpLanes);
      r[v] = reinterpret_cast<const double2 *>(vrec + (size_t)ev * kR)[lane % (kR / 2)];
    }
#pragma unroll
    for (int v = 0; v < kVjpUnroll * kP; ++v)
      if (p + v * kG + lane / kP < p1) {
        rs.x += r[v].x;
        rs.y += r[v].y;
      }
    settle(rs.x);
    settle(rs.y);
    if (!staged) {
      wave_lds_sync();
      get(d, xa);
      staged = true;
    }
#pragma unroll
    for (int u = 0; u < kVjpUnroll; ++u)
      if (p + lane + kVjpLanes * u < p1) {
        int o[3];
        IncLoc<IL>::others(il[u], o);
        const int n = IncLoc<IL>::a(il[u]);
        double b0[9], b1[9], b2[9], g[3];
        get(o[0], b0);
        get(o[1], b1);
        get(o[2], b2);
        const double x0[3] = {b0[0], b0[1], b0[2]}, x1[3] = {b1[0], b1[1], b1[2]}, x2[3] = {b2[0], b2[1], b2[2]},
                     xo[3] = {xa[0], xa[1], xa[2]};
        const double W = own_gradient(xo, x0, x1, x2, n, g);
        // m_a: local node 3 has a weight of its own (flux_weight)
        const double m0 = flux_weight(W, 0), m3 = flux_weight(W, 3);
        const double ma = n == 3 ? m3 : m0, m2 = n == 3 ? m0 : m3;
        double Q[6];
#pragma unroll
        for (int k = 0; k < 6; ++k) Q[k] = ma * xa[3 + k] + m0 * (b0[3 + k] + b1[3 + k]) + m2 * b2[3 + k];
        const double t[3] = {2.0 * Q[0] * g[0] + Q[1] * g[1] + Q[2] * g[2],
                             Q[1] * g[0] + 2.0 * Q[3] * g[1] + Q[4] * g[2],
                             Q[2] * g[0] + Q[4] * g[1] + 2.0 * Q[5] * g[2]};
        const double mu = ens_mu(en, ea[u] >> 2, mu0);
        mub += ua[0] * t[0] + ua[1] * t[1] + ua[2] * t[2];
#pragma unroll
        for (int k = 0; k < 3; ++k) t3[k] += mu * t[k];
      }
    p += kVjpLanes * kVjpUnroll;
  } while (p < p1);
#pragma unroll
  for (int off = kP; off < kVjpLanes; off <<= 1) {
    rs.x += __shfl_xor(rs.x, off, kVjpLanes);
    rs.y += __shfl_xor(rs.y, off, kVjpLanes);
  }
#pragma unroll
  for (int off = 1; off < kVjpLanes; off <<= 1)
#pragma unroll
    for (int k = 0; k < 3; ++k) t3[k] += __shfl_xor(t3[k], off, kVjpLanes);
  // lane k < kP holds components 2 k, 2 k + 1: ybar 0..3, acbar 4..6
  const size_t N = nshg;
  if (live && lane < kR / 2) {
    double *o = (lane < 2 ? ybar : acbar) + i + N * (2 * (lane % 2));
    o[0] = lane == 0 ? rs.x + t3[0] : lane == 1 ? rs.x + t3[2] : rs.x;
    o[N] = lane == 0 ? rs.y + t3[1] : lane == 3 ? 0.0 : rs.y;
  }
  __syncthreads();  // the staged neighbours are read: their LDS takes the parts
  const double ms = block_sum<256>(mub, *reinterpret_cast<double(*)[256 / 64]>(&xs_all[0][0]));
  if (threadIdx.x == 0) part[blk] = ms;
}

// mubar: the workgroups' parts in a fixed order, one workgroup.
constexpr int kMuThreads = 1024;
__global__ void __launch_bounds__(kMuThreads) mu_final(int n, const double *__restrict__ part,
                                                       double *__restrict__ out) {
  __shared__ double sh[kMuThreads / 64];
  double s = 0.0;
#pragma unroll 8
  for (int k = threadIdx.x; k < n; k += kMuThreads) s += part[k];
  s = block_sum<kMuThreads>(s, sh);
  if (threadIdx.x == 0) *out = s;
}

template <class IL>
void vjp_nodes(crimson_form *f, double *d_ybar, double *d_acbar, const crimson::VjpWork &w, double *part) {
  hipStream_t s = f->stream;
  const unsigned gn = crimson::grid_for((size_t)f->nshg * kVjpLanes, 256);
  const IL *il = reinterpret_cast<const IL *>(f->d_iloc.p);
  vjp_q_node<IL><<<gn, 256, 0, s>>>(f->nshg, f->near_ptr(), f->near_diag(), f->d_col.p, f->d_inc_ptr.p, f->d_inc.p, il,
                                    f->d_xu.p, w.vrec2, w.invm, w.qbar);
  if (d_acbar)
    vjp_node<IL, true><<<gn, 256, 0, s>>>(f->nshg, f->near_ptr(), f->near_diag(), f->d_col.p, f->d_inc_ptr.p,
                                          f->d_inc.p, il, f->d_xu.p, w.qbar, w.vrec, f->prm.mu, f->ens(), d_ybar,
                                          d_acbar, part);
  else
    vjp_node<IL, false><<<gn, 256, 0, s>>>(f->nshg, f->near_ptr(), f->near_diag(), f->d_col.p, f->d_inc_ptr.p,
                                           f->d_inc.p, il, f->d_xu.p, w.qbar, w.vrec, f->prm.mu, f->ens(), d_ybar,
                                           nullptr, part);
}

}  // namespace

namespace crimson {
void vjp_work_sizes(const crimson_form *f, size_t n[6]) {
  const size_t ne = (size_t)std::max(f->nel, 1), nn = (size_t)f->nshg;
  n[0] = ne * kVRecYA;
  n[1] = ne * kVRecD;
  n[2] = nn * kXQ;
  n[3] = nn;
  n[4] = (ne + kVThreads - 1) / kVThreads + (nn * kVjpLanes + 255) / 256 +
         (size_t)form_boundary_vjp_parts(f) + 1;
  n[5] = form_boundary_vjp_doubles(f);
}

int vjp_run(crimson_form *f, const double *d_y, const double *d_ac, const double *d_x, const double *d_w,
            double *d_ybar, double *d_acbar, double *mubar, const VjpWork &w) {
  if (f->wall) {
    crimson::set_error("crimson_form_vjp_dev: the deformable wall's rows have no adjoint here");
    return CRIMSON_EUNSUPPORTED;
  }
  hipStream_t s = f->stream;
  const FormConst c = make_const(f->prm);
  CR_TRY(crimson::form_flux_pass(f, d_y, d_ac, d_x, nullptr, w.invm));
  const unsigned ge = crimson::grid_for(f->nel, kVThreads);
  const int nm1 = (int)(ge + crimson::grid_for((size_t)f->nshg * kVjpLanes, 256));
  const int nmu = nm1 + form_boundary_vjp_parts(f);
  if (f->nel > 0) {
    if (d_acbar)
      vjp_e3_elem<true><<<ge, kVThreads, 0, s>>>(f->nel, f->d_ien.p, f->d_node.p, d_w, f->nshg, c, f->ens(), w.vrec,
                                                 w.vrec2, w.mupart);
    else
      vjp_e3_elem<false><<<ge, kVThreads, 0, s>>>(f->nel, f->d_ien.p, f->d_node.p, d_w, f->nshg, c, f->ens(), w.vrec,
                                                  w.vrec2, w.mupart);
  }
  if (f->wide)
    vjp_nodes<unsigned long long>(f, d_ybar, d_acbar, w, w.mupart + ge);
  else
    vjp_nodes<unsigned>(f, d_ybar, d_acbar, w, w.mupart + ge);
  CR_TRY(crimson::form_boundary_vjp(f, d_w, d_ybar, w.mupart + nm1, w.bvrec));  // the boundary rows (crimson_form_set_boundary)
  mu_final<<<1, kMuThreads, 0, s>>>(nmu, w.mupart, w.mupart + nmu);
  CR_HIP(hipGetLastError());
  double mb = 0.0;
  CR_HIP(hipMemcpyAsync(&mb, w.mupart + nmu, sizeof(double), hipMemcpyDeviceToHost, s));
  CR_HIP(hipStreamSynchronize(s));
  if (mubar) *mubar = mb;
  return CRIMSON_OK;
}

}  // namespace crimson

namespace {
int vjp_entry(crimson_form *f, const double *d_y, const double *d_ac, const double *d_x, const double *d_w,
              double *d_ybar, double *d_acbar, double *mubar) {
  if (!f || !d_y || !d_ac || !d_x || !d_w || !d_ybar) {
    crimson::set_error("crimson_form_vjp_dev: null argument");
    return CRIMSON_EARG;
  }
  size_t n[6];
  crimson::vjp_work_sizes(f, n);
  CR_TRY(f->d_vrec.alloc(n[0]));
  CR_TRY(f->d_vrec2.alloc(n[1]));
  CR_TRY(f->d_qbar.alloc(n[2]));
  CR_TRY(f->d_invm.alloc(n[3]));
  CR_TRY(f->d_mupart.alloc(n[4]));
  const crimson::VjpWork w{f->d_vrec.p, f->d_vrec2.p, f->d_qbar.p, f->d_invm.p, f->d_mupart.p, nullptr};
  return crimson::vjp_run(f, d_y, d_ac, d_x, d_w, d_ybar, d_acbar, mubar, w);
}
}  // namespace

extern "C" int crimson_form_vjp_dev(crimson_form *f, const double *d_y, const double *d_ac, const double *d_x,
                                    const double *d_w, double *d_ybar, double *mubar) {
  return vjp_entry(f, d_y, d_ac, d_x, d_w, d_ybar, nullptr, mubar);
}

extern "C" int crimson_form_vjp_ac_dev(crimson_form *f, const double *d_y, const double *d_ac, const double *d_x,
                                       const double *d_w, double *d_ybar, double *d_acbar, double *mubar) {
  if (!d_acbar) {
    crimson::set_error("crimson_form_vjp_ac_dev: null acbar");
    return CRIMSON_EARG;
  }
  return vjp_entry(f, d_y, d_ac, d_x, d_w, d_ybar, d_acbar, mubar);
}
