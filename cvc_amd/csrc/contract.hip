// Conserved-vector-current contraction Pi_{mu nu}(x), contact term, Ward
// identity, Pi(q) and the whole-source pipeline.
//
// The reference (cvc_exact2_xspace.c:577-861) sweeps the volume 4608 times
// per source.  Written with 12x12 propagator matrices S(x) (rows: sink
// spin-colour, columns: source spin-colour k = 3*spin + colour) the same sum is
//
//   conn_{mu nu}(x) = -1/4 sum_{k,l} { G1_{kl} [ Sd_nu(x)_l^+  Gm_mu U~_mu(x)   Su_4(x+mu)_k
//                                              + Sd_nu(x+mu)_l^+ Gp_mu U~_mu(x)^+ Su_4(x)_k ]
//                                    + G2_{kl} [ Sd_4(x)_l^+   Gm_mu U~_mu(x)   Su_nu(x+mu)_k
//                                              + Sd_4(x+mu)_l^+ Gp_mu U~_mu(x)^+ Su_nu(x)_k ] }
//
// with sink vertices Gm_mu = gamma5 (gamma_mu - 1), Gp_mu = gamma5 (gamma_mu + 1),
// source vertices G1 = (gamma_nu gamma5 - gamma5) (x) Us_nu and
// G2 = (gamma_nu gamma5 + gamma5) (x) Us_nu^+ (spin (x) colour, Us_nu = U~_nu(y)),
// Su_s / Sd_s the up / down propagators from y + s^ (s = 4: y).  Here the
// reference's gperm / gperm_sign / isimag tables (:336-383) are the non-zero
// entries of gamma_nu gamma5 and gamma5, and the conj(Us[ib][ia]) of part 2 is
// (Us^+)[ia][ib].
//
// GPU schedule: both kinds of vertex have rank 2 in spin.  gamma_mu couples the
// spins in two pairs (a, b = GCOL[mu][a]), a = 0, 1, with units e_a and conj(e_a),
// so (gamma -+ 1) is -+(1, -+conj(e_a)) (x) (1, -+e_a) on a pair.  With the source
// vertex split like this, the 12 x 12 sum over (k, l) is one over 6 products of
// combined columns, indexed by (pair, colour), for either part:
//   part 1:  D = sum_ib conj(Us[ia][ib]) (Sd_nu(a,ib) + conj(e) Sd_nu(b,ib)),  U = Su_4(a,ia) - conj(e) Su_4(b,ia)
//   part 2:  D = sum_ib Us[ib][ia] (Sd_4(a,ib) - conj(e) Sd_4(b,ib)),          U = Su_nu(a,ia) + conj(e) Su_nu(b,ia)
//   k_cols:  D and U of the 12 combined columns of each nu for a few time slices
//   k_conn:  one thread per (x, nu, column): the sink vertex split the same way,
//            conn_{mu nu}(x) = -1/4 sum_cols sign (<D_a + e D_b, U_mu (x+mu)...>), see there
// (one combined column instead of two column pairs: half the bytes and a third
// of the arithmetic of contracting 24 columns of Psi with 24 of Su).
// FP64 throughout.
#include <stdio.h>
#include <string.h>
#include <math.h>
#include <algorithm>
#include <vector>

#include "contract_common.h"

namespace cvchip {

int invert_her_fields(cvchip_ctx *c, Field &x, const Field &b, double sp, int niter_max, int prec,
                      double delta, unsigned flags, cvchip_stats *stats);

// Psi fields for one nu.  up/dn: 60-column sets (12*s + k); psi: 24-column set.
// A block of 240 threads handles 10 sites: the 24 down-propagator columns the
// block needs (12 from y + nu, 12 from y, all 12 components) are staged in LDS
// with coalesced loads, each read once; then one thread per (x, part, k)
// (k fastest): part 0 is Psi1 from the columns of y + nu, part 1 Psi2 from y.
constexpr int kPsiSites = 10;
__global__ void __launch_bounds__(240) k_psi(double2 *__restrict__ psi, const double2 *__restrict__ dn,
                                             SrcLinks L, int nu, uint32_t V) {
  __shared__ double2 sd[kPsiSites][12][24];
  const uint32_t x0 = blockIdx.x * (uint32_t)kPsiSites;
  const uint32_t VN = V * 60u, VP = V * 24u;
  for (uint32_t e = threadIdx.x; e < (uint32_t)kPsiSites * 12u * 24u; e += blockDim.x) {
    const uint32_t col = e % 24u, rem = e / 24u, c = rem % 12u, xs = rem / 12u;
    const uint32_t x = x0 + xs;
    if (x < V) sd[xs][c][col] = dn[(size_t)c * VN + (size_t)x * 60u + (col < 12u ? 12u * (uint32_t)nu + col : 36u + col)];
  }
  __syncthreads();
  const uint32_t xs = threadIdx.x / 24u, x = x0 + xs;
  if (x >= V) return;
  const int j24 = (int)(threadIdx.x % 24u), part = j24 / 12, k = j24 % 12;
  const int ir = k / 3, ia = k % 3;
  // (gamma_nu gamma5)_{ir, j}: j = GCOL[nu][ir], value = GVAL[nu][ir] * g5sign(j)
  const int j = GCOL[nu][ir];
  double2 e = unit_val(GVAL[nu][ir]);
  if (g5sign(j) < 0) { e.x = -e.x; e.y = -e.y; }
  const double s5 = (double)g5sign(ir);
  const double2 *Us = L.u[nu];
  double2 p[12];
#pragma unroll
  for (int c = 0; c < 12; c++) p[c] = make_double2(0, 0);
  for (int ib = 0; ib < 3; ib++) {
    double2 wa, wb;
    if (part == 0) {
      // conj(G1_{k,l}) with G1 = (e d_{l,j} - s5 d_{l,ir}) Us[ia][ib]
      const double2 u1 = Us[3 * ia + ib];
      wa = cmulc(u1, cmulc(e, make_double2(1, 0)));      // conj(e * u1)
      wb = make_double2(-s5 * u1.x, s5 * u1.y);          // conj(-s5 * u1)
    } else {
      // G2 = (e d_{l,j} + s5 d_{l,ir}) conj(Us[ib][ia]); conj(G2) = conj(e) Us[ib][ia], s5 Us[ib][ia]
      const double2 u2 = Us[3 * ib + ia];
      wa = cmulc(e, u2);
      wb = make_double2(s5 * u2.x, s5 * u2.y);
    }
    const int la = 12 * part + 3 * j + ib, lb = 12 * part + 3 * ir + ib;
#pragma unroll
    for (int c = 0; c < 12; c++) p[c] = cfma(cfma(p[c], wa, sd[xs][c][la]), wb, sd[xs][c][lb]);
#pragma unroll
    for (int c = 0; c < 12; c++) pin(p[c]);
  }
#pragma unroll
  for (int c = 0; c < 12; c++) psi[(size_t)c * VP + (size_t)x * 24u + j24] = p[c];
}

// Combined columns of one slab: [2 (D, U)][4 nu][12 comps][sites of ns slices][12 columns].
struct Slab {
  double2 *p;
  uint32_t slice, ns;
  __host__ __device__ __forceinline__ size_t plane() const { return (size_t)ns * slice * 12u; }
  __host__ __device__ __forceinline__ size_t at(int which, int nu, int comp) const {
    return ((size_t)(which * 4 + nu) * 12 + comp) * plane();
  }
};

// The combined columns of kColSites sites of one slice (blockIdx.x), one
// component (blockIdx.y): the sites' 60 + 60 columns of that component are
// contiguous; they are staged in LDS and read from memory once.  Slice tau of the
// sweep (blockIdx.z past tau0) is time slice tau mod T, in slot tau mod ns.
// Bound by memory: 120 columns read, 96
// written, 41.5 KB a site; 365 us for the 32000 sites of a slab at 40x20^3, 3.6 TB/s beside the copies of conn.
constexpr int kColSites = 16;
__global__ void __launch_bounds__(256) k_cols(Slab B, const double2 *__restrict__ up, const double2 *__restrict__ dn,
                                              SrcLinks L, uint32_t V, uint32_t T, uint32_t tau0) {
  __shared__ double2 su[kColSites * 60], sd[kColSites * 60], us[4][9], ce[4][2];
  const uint32_t tau = tau0 + blockIdx.z, x0 = blockIdx.x * (uint32_t)kColSites;
  const uint32_t nx = min((uint32_t)kColSites, B.slice - x0);
  const int comp = (int)blockIdx.y;
  const size_t base = ((size_t)comp * V + (size_t)(tau % T) * B.slice + x0) * 60u;
  for (uint32_t e = threadIdx.x; e < nx * 60u; e += 256u) {
    su[e] = up[base + e];
    sd[e] = dn[base + e];
  }
  if (threadIdx.x < 36) us[threadIdx.x / 9][threadIdx.x % 9] = L.u[threadIdx.x / 9][threadIdx.x % 9];
  if (threadIdx.x < 8) {
    const double2 e = unit_val(GVAL[threadIdx.x / 2][threadIdx.x % 2]);
    ce[threadIdx.x / 2][threadIdx.x % 2] = make_double2(e.x, -e.y);
  }
  __syncthreads();
  // 8 (which, nu) groups of 16 sites x 12 columns; a group is three whole waves
#pragma unroll 1
  for (uint32_t o = threadIdx.x; o < 8u * kColSites * 12u; o += 256u) {
    const uint32_t g = o / (kColSites * 12u), rem = o - g * (kColSites * 12u);
    const uint32_t xs = rem / 12u, col = rem - xs * 12u;
    if (xs >= nx) continue;
    const int which = (int)(g >> 2), nu = (int)(g & 3u);
    const int part = (int)(col / 6u), a = (int)(col % 6u) / 3, ia = (int)(col % 3u), b = GCOL[nu][a];
    const double2 ec = ce[nu][a];
    double2 r = make_double2(0, 0);
    if (which == 0) {
      // part 1: columns of y + nu, + conj(e); part 2: columns of y, - conj(e)
      const double2 *q = sd + xs * 60u + (part == 0 ? 12 * nu : 48);
      const double2 e = part == 0 ? ec : make_double2(-ec.x, -ec.y);
#pragma unroll
      for (int ib = 0; ib < 3; ib++) {
        const double2 v = cfma(q[3 * a + ib], e, q[3 * b + ib]);
        r = part == 0 ? cfmac(r, us[nu][3 * ia + ib], v) : cfma(r, us[nu][3 * ib + ia], v);
      }
    } else {
      // part 1: columns of y, - conj(e); part 2: columns of y + nu, + conj(e)
      const double2 *q = su + xs * 60u + (part == 0 ? 48 : 12 * nu);
      const double2 e = part == 0 ? make_double2(-ec.x, -ec.y) : ec;
      r = cfma(q[3 * a + ia], e, q[3 * b + ia]);
    }
    B.p[B.at(which, nu, comp) + ((size_t)(tau % B.ns) * B.slice + x0 + xs) * 12u + col] = r;
  }
}

// sum over the thread's column of both sink terms of one mu: with
// gamma5 (gamma_mu - 1) and gamma5 (gamma_mu + 1) split on the pairs (a, b),
//   -<D_a + e D_b, U_mu(x) (U_a - e U_b)(x+mu)> + <U_mu(x) (D_a - e D_b)(x+mu), U_a + e U_b>
// (D, U at x the thread's own, at x + mu loaded from dn, un).
template <int MU>
__device__ __forceinline__ void conn_mu(double2 &acc, const double2 d[12], const double2 u[12],
                                        const double2 *__restrict__ dn, const double2 *__restrict__ un, size_t plane,
                                        const double2 *__restrict__ link) {
#pragma unroll
  for (int a = 0; a < 2; a++) {
    const int b = GCOL[MU][a], ua = GVAL[MU][a];
    double2 w[3], q[3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const double2 da = dn[(size_t)(3 * a + c) * plane], db = dn[(size_t)(3 * b + c) * plane];
      const double2 va = un[(size_t)(3 * a + c) * plane], vb = un[(size_t)(3 * b + c) * plane];
      q[c] = csub(da, times_unit(ua, db));
      w[c] = csub(va, times_unit(ua, vb));
    }
#pragma unroll
    for (int i = 0; i < 3; i++) {
      double2 uw = make_double2(0, 0), uq = make_double2(0, 0);
#pragma unroll
      for (int j = 0; j < 3; j++) {
        const double2 l = link[3 * i + j];
        uw = cfma(uw, l, w[j]);
        uq = cfma(uq, l, q[j]);
      }
      const double2 qo = cadd(d[3 * a + i], times_unit(ua, d[3 * b + i]));
      const double2 wo = cadd(u[3 * a + i], times_unit(ua, u[3 * b + i]));
      acc = cfmac(acc, make_double2(-qo.x, -qo.y), uw);
      acc = cfmac(acc, uq, wo);
    }
    pin(acc);
  }
}

// One thread per (site, column), blocks of 240 = kConnSites sites x 12, nu =
// blockIdx.y, slice tau0 + blockIdx.z.  XCD j takes the j-th eighth of the
// slice, so that the y and x neighbours are in its L2: the thread keeps its own D and U for the four mu
// and reads the neighbours' at x + mu; the block's links (boundary phase applied)
// are staged in LDS.  The 12 columns of a (x, mu) are summed in LDS in a fixed
// order.  Two waves per SIMD (224 VGPRs; at three the compiler spills and it
// takes half as long again), bound by the latency of a mu's 24 neighbour loads: 288
// us for 32000 sites at 40x20^3 (340 us with the workgroups dealt to the XCDs in
// turn).
constexpr int kConnSites = 20;
__global__ void __launch_bounds__(240) k_conn(double2 *__restrict__ conn, Slab B, const double2 *__restrict__ U,
                                              ConnParams P, uint32_t tau0) {
  __shared__ double2 link[kConnSites][4][9];
  __shared__ double2 red[4][240];
  const uint32_t tau = tau0 + blockIdx.z, nu = blockIdx.y;
  const uint32_t x0 =   // within the slice; past its end in the last blocks
      ((blockIdx.x % kXcds) * (gridDim.x / kXcds) + blockIdx.x / kXcds) * (uint32_t)kConnSites;
  for (uint32_t e = threadIdx.x; e < 36u * kConnSites; e += 240u) {
    const uint32_t k = e / kConnSites, xs = e - k * kConnSites, mu = k / 9u;
    if (x0 + xs < B.slice)
      link[xs][mu][k - 9u * mu] =
          cmul(U[(size_t)k * P.V + (size_t)tau * B.slice + x0 + xs], make_double2(P.ph_re[mu], P.ph_im[mu]));
  }
  const uint32_t xs = threadIdx.x / 12u, col = threadIdx.x - 12u * xs, x = x0 + xs;
  const bool act = x < B.slice;
  const size_t plane = B.plane();
  const double2 *D = B.p + B.at(0, (int)nu, 0), *Up = B.p + B.at(1, (int)nu, 0);
  double2 acc[4] = {make_double2(0, 0), make_double2(0, 0), make_double2(0, 0), make_double2(0, 0)};
  double2 d[12], u[12];
  const uint32_t slot = tau % B.ns, slotp = (tau + 1u) % B.ns;
  if (act) {
    const size_t i = ((size_t)slot * B.slice + x) * 12u + col;
#pragma unroll
    for (int c = 0; c < 12; c++) d[c] = D[(size_t)c * plane + i];
#pragma unroll
    for (int c = 0; c < 12; c++) u[c] = Up[(size_t)c * plane + i];
  }
  __syncthreads();
  if (act) {
    const uint32_t cx = x / P.sX, rem = x - cx * P.sX;
    const uint32_t cy = rem / (uint32_t)P.LZ, cz = rem - cy * (uint32_t)P.LZ;
    const uint32_t LX = (uint32_t)P.LX, LY = (uint32_t)P.LY, LZ = (uint32_t)P.LZ;
    // z first: the z neighbour's columns were read moments ago by the next site's threads
    const uint32_t xz = cz == LZ - 1 ? x - (LZ - 1) : x + 1, xy = cy == LY - 1 ? x - (LY - 1) * LZ : x + LZ;
    const uint32_t xx = cx == LX - 1 ? x - (LX - 1) * P.sX : x + P.sX;
    const size_t iz = ((size_t)slot * B.slice + xz) * 12u + col, iy = ((size_t)slot * B.slice + xy) * 12u + col;
    const size_t ix = ((size_t)slot * B.slice + xx) * 12u + col, it = ((size_t)slotp * B.slice + x) * 12u + col;
    conn_mu<3>(acc[3], d, u, D + iz, Up + iz, plane, link[xs][3]);
    conn_mu<2>(acc[2], d, u, D + iy, Up + iy, plane, link[xs][2]);
    conn_mu<1>(acc[1], d, u, D + ix, Up + ix, plane, link[xs][1]);
    conn_mu<0>(acc[0], d, u, D + it, Up + it, plane, link[xs][0]);
  }
#pragma unroll
  for (int mu = 0; mu < 4; mu++) red[mu][threadIdx.x] = acc[mu];
  __syncthreads();
  if (col < 4u && act) {
    const uint32_t mu = col, t0 = threadIdx.x - col;
    double2 s = make_double2(0, 0);   // part 1 enters with -1
    for (uint32_t k = 0; k < 6; k++) { s.x -= red[mu][t0 + k].x; s.y -= red[mu][t0 + k].y; }
    for (uint32_t k = 6; k < 12; k++) { s.x += red[mu][t0 + k].x; s.y += red[mu][t0 + k].y; }
    conn[((size_t)tau * B.slice + x) * 16u + 4u * mu + nu] = make_double2(-0.25 * s.x, -0.25 * s.y);
  }
}

// contact term pieces: thread (nu, ir, ia) -> part-1 and part-2 values
__global__ void k_contact(double2 *__restrict__ out, const double2 *__restrict__ up, SrcLinks L,
                          uint32_t ys, const uint32_t ysp[4], uint32_t V) {
  const int t = threadIdx.x;
  if (t >= 48) return;
  const int nu = t / 12, k = t % 12;
  const uint32_t VN = V * 60u;
  double2 phi[12], w[12];
  const double2 *Us = L.u[nu];
  // part 1: (gamma_nu - 1) Us phi(y + nu), phi = up from y (s = 4), column k, row k
  for (int c = 0; c < 12; c++) phi[c] = up[(size_t)c * VN + (size_t)ysp[nu] * 60u + 48 + k];
  su3_mul(w, Us, phi, false);
  const int a = k / 3, cc = k % 3;
  {
    const int b = GCOL[nu][a];
    double2 g = cmul(unit_val(GVAL[nu][a]), w[3 * b + cc]);
    out[2 * t] = make_double2(-0.5 * (g.x - w[k].x), -0.5 * (g.y - w[k].y));
  }
  // part 2: (gamma_nu + 1) Us^+ phi(y), phi = up from y + nu (s = nu)
  for (int c = 0; c < 12; c++) phi[c] = up[(size_t)c * VN + (size_t)ys * 60u + 12 * nu + k];
  su3_mul(w, Us, phi, true);
  {
    const int b = GCOL[nu][a];
    double2 g = cmul(unit_val(GVAL[nu][a]), w[3 * b + cc]);
    out[2 * t + 1] = make_double2(0.5 * (g.x + w[k].x), 0.5 * (g.y + w[k].y));
  }
}

__global__ void k_src_links(SrcLinks *out, const double2 *__restrict__ U, uint32_t V, uint32_t y,
                            ConnParams P) {
  const int t = threadIdx.x;
  if (t >= 36) return;
  const int nu = t / 9, q = t % 9;
  out->u[nu][q] = cmul(U[(size_t)(nu * 9 + q) * V + y], make_double2(P.ph_re[nu], P.ph_im[nu]));
}

// Source links Us_nu = U_nu(y) * phase_nu on the host (for kernels taking them by value).
int source_links(cvchip_ctx *c, const int src[4], SrcLinks *out) {
  SrcLinks *dL = nullptr;
  CVC_HIP(hipMalloc(&dL, sizeof(SrcLinks)));
  const uint32_t y = site_of(c, src[0], src[1], src[2], src[3]);
  hipLaunchKernelGGL(k_src_links, dim3(1), dim3(64), 0, c->stream, dL, (const double2 *)c->gauge64,
                     (uint32_t)c->lat.V, y, conn_params(c));
  hipError_t e = hipMemcpyAsync(out, dL, sizeof(SrcLinks), hipMemcpyDeviceToHost, c->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
  (void)hipFree(dL);
  if (e != hipSuccess) return hip_fail(e, "source links", __FILE__, __LINE__);
  return 0;
}

// Psi1 / Psi2 of one nu (24-column set psi) from the down propagators
int launch_psi(cvchip_ctx *c, double2 *psi, const Field &dn, const SrcLinks &L, int nu) {
  const uint32_t V = (uint32_t)c->lat.V;
  hipLaunchKernelGGL(k_psi, dim3((V + kPsiSites - 1) / kPsiSites), dim3(240), 0, c->stream, psi,
                     (const double2 *)dn.data, L, nu, V);
  CVC_HIP(hipGetLastError());
  return 0;
}

// Sites of a slab: enough blocks for several rounds of the chip, and pieces of conn
// (8 MB) that the host copies while the next slabs are computed.  The whole
// contraction with 8000 / 16000 / 32000 / 64000 sites at least: 32x16^3 3.08 / 2.74 /
// 2.76 / 2.98 ms, 40x20^3 8.04 / 6.34 / 6.10 / 6.16, 96x12^3 3.62 / 3.36 / 3.19 / 4.54,
// 20x30x18x22 5.03 / 4.78 / 4.64 / 6.68, 48x24^3 12.9 / 12.5 / 13.0 / 18.4 (13.9 ms at
// 40x20^3 with 24-column Psi fields per nu and one copy at the end).
constexpr uint32_t kSlabSites = 32000;

// conn (host [V][16][2]) and contact from device up / dn sets of 60 columns
int contract_fields(cvchip_ctx *c, double *conn, double contact[8], const Field &up, const Field &dn,
                    const int src[4]) {
  if (!c->gauge_set) {
    set_error("gauge field not set (call cvchip_set_gauge first)");
    return CVCHIP_ERR_STATE;
  }
  if (up.nrhs != 60 || dn.nrhs != 60 || up.prec != CVCHIP_PREC_F64 || dn.prec != CVCHIP_PREC_F64) {
    set_error("contraction needs FP64 up and down sets of 60 propagator columns");
    return CVCHIP_ERR_ARG;
  }
  const uint32_t V = (uint32_t)c->lat.V;
  const ConnParams P = conn_params(c);
  const uint32_t y = site_of(c, src[0], src[1], src[2], src[3]);
  uint32_t ysp[4] = {site_of(c, src[0] + 1, src[1], src[2], src[3]), site_of(c, src[0], src[1] + 1, src[2], src[3]),
                     site_of(c, src[0], src[1], src[2] + 1, src[3]), site_of(c, src[0], src[1], src[2], src[3] + 1)};
  SrcLinks *dL = nullptr, hL;
  double2 *dconn = nullptr, *dct = nullptr;
  uint32_t *dysp = nullptr;
  int rc = 0;
  auto fail = [&](hipError_t e, const char *w) { return hip_fail(e, w, __FILE__, __LINE__); };
  // Slabs of nt time slices: the combined columns of a slab and of the slice after it
  // (18 KB a site, 737 MB at 40x20^3: they go through HBM, not the 256 MB MALL) are
  // formed, contracted, and overwritten by the next slab's.
  const uint32_t T = (uint32_t)c->lat.T, slice = V / T;
  const uint32_t nt = std::min(T, (kSlabSites + slice - 1) / slice);
  Slab B{nullptr, slice, nt == T ? T : nt + 1};
  const size_t conn_bytes = sizeof(double2) * 16 * (size_t)V, slab_bytes = sizeof(double2) * 96 * B.plane();
  hipError_t e = hipMalloc(&dL, sizeof(SrcLinks));
  if (e == hipSuccess) e = hipMalloc(&dct, sizeof(double2) * 96);
  if (e == hipSuccess) e = hipMalloc(&dysp, sizeof(uint32_t) * 4);
  if (e != hipSuccess) rc = fail(e, "contraction buffers");
  if (!rc) rc = pool_get(c, (void **)&dconn, conn_bytes);   // the large buffers come from the context's pool
  if (!rc) rc = pool_get(c, (void **)&B.p, slab_bytes);
  if (!rc) {
    hipLaunchKernelGGL(k_src_links, dim3(1), dim3(64), 0, c->stream, dL, (const double2 *)c->gauge64, V, y, P);
    e = hipMemcpyAsync(&hL, dL, sizeof(SrcLinks), hipMemcpyDeviceToHost, c->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(dysp, ysp, sizeof(ysp), hipMemcpyHostToDevice, c->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    if (e != hipSuccess) rc = fail(e, "source links");
  }
  HostStream out(c);
  const bool pieces = conn_bytes >= HostStream::kMinTotal;
  uint32_t have = 0;   // slices whose combined columns have been formed
  for (uint32_t t0 = 0; t0 < T && !rc; t0 += nt) {
    const uint32_t n = std::min(nt, T - t0);
    const uint32_t need = nt == T ? T : t0 + n + 1;   // slice T of the sweep is slice 0 again
    hipLaunchKernelGGL(k_cols, dim3((slice + kColSites - 1) / kColSites, 12, need - have), dim3(256), 0, c->stream, B,
                       (const double2 *)up.data, (const double2 *)dn.data, hL, V, T, have);
    have = need;
    const uint32_t nb = (slice + kConnSites - 1) / kConnSites;
    hipLaunchKernelGGL(k_conn, dim3((nb + kXcds - 1) / kXcds * kXcds, 4, n), dim3(240), 0, c->stream, dconn, B,
                       (const double2 *)c->gauge64, P, t0);
    e = hipGetLastError();
    if (e != hipSuccess) rc = fail(e, "contraction kernels");
    // conn leaves for the host slab by slab, behind the kernels of the next slabs
    const size_t off = (size_t)t0 * slice * 16;
    if (!rc && pieces) rc = out.push(conn + 2 * off, dconn + off, sizeof(double2) * 16 * n * slice);
  }
  if (!rc) {
    hipLaunchKernelGGL(k_contact, dim3(1), dim3(64), 0, c->stream, dct, (const double2 *)up.data, hL, y,
                       (const uint32_t *)dysp, V);
    double2 hct[96];
    rc = pieces ? out.finish() : copy_to_host(c, conn, dconn, conn_bytes);
    if (!rc) {
      e = hipMemcpyAsync(hct, dct, sizeof(hct), hipMemcpyDeviceToHost, c->stream);
      if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
      if (e != hipSuccess) rc = fail(e, "contraction results");
    }
    if (!rc) {
      // accumulate in the reference's order: part 1 over (ir, ia), then part 2
      for (int nu = 0; nu < 4; nu++) {
        double re = 0., im = 0.;
        for (int k = 0; k < 12; k++) { re += hct[2 * (12 * nu + k)].x; im += hct[2 * (12 * nu + k)].y; }
        for (int k = 0; k < 12; k++) { re += hct[2 * (12 * nu + k) + 1].x; im += hct[2 * (12 * nu + k) + 1].y; }
        contact[2 * nu] = re;
        contact[2 * nu + 1] = im;
      }
    }
  }
  (void)out.finish();   // (a failed call: nothing in flight from the buffers that go back)
  if (dL) (void)hipFree(dL);
  pool_put(c, dconn, conn_bytes);
  pool_put(c, B.p, slab_bytes);
  if (dct) (void)hipFree(dct);
  if (dysp) (void)hipFree(dysp);
  return rc;
}

// ------------------------------------------------------------ Ward identity
__global__ void k_wi(double2 *__restrict__ wi, const double2 *__restrict__ conn, ConnParams P) {
  const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= P.V) return;
  uint32_t rem = x;
  const uint32_t ct = rem / P.sT; rem -= ct * P.sT;
  const uint32_t cx = rem / P.sX; rem -= cx * P.sX;
  const uint32_t cy = rem / (uint32_t)P.LZ;
  const uint32_t cz = rem - cy * (uint32_t)P.LZ;
  const uint32_t xm[4] = {ct == 0 ? x + (P.T - 1) * P.sT : x - P.sT, cx == 0 ? x + (P.LX - 1) * P.sX : x - P.sX,
                          cy == 0 ? x + (P.LY - 1) * P.LZ : x - P.LZ, cz == 0 ? x + (P.LZ - 1) : x - 1};
  for (int nu = 0; nu < 4; nu++) {
    double re = 0., im = 0.;
    for (int mu = 0; mu < 4; mu++) {
      re += conn[(size_t)x * 16 + 4 * mu + nu].x;
      im += conn[(size_t)x * 16 + 4 * mu + nu].y;
    }
    for (int mu = 0; mu < 4; mu++) {
      re -= conn[(size_t)xm[mu] * 16 + 4 * mu + nu].x;
      im -= conn[(size_t)xm[mu] * 16 + 4 * mu + nu].y;
    }
    wi[(size_t)x * 4 + nu] = make_double2(re, im);
  }
}

// ------------------------------------------------------------------ Pi(q)
// One pass of a length-L DFT along a direction of stride `stride` (in sites):
// out[.. n ..] = sum_x w[(n x) mod L] in[.. x ..],  w[k] = exp(-2 pi i k / L).
// 16 components per site, one thread per (site, component).
__global__ void k_dft_dir(double2 *__restrict__ out, const double2 *__restrict__ in,
                          const double2 *__restrict__ w, uint32_t V, int L, uint32_t stride) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= V * 16u) return;
  const uint32_t site = i / 16u, comp = i % 16u;
  const uint32_t n = (site / stride) % (uint32_t)L;
  const uint32_t base = site - n * stride;
  double2 acc = make_double2(0, 0);
  uint32_t k = 0;
  for (int x = 0; x < L; x++) {
    acc = cfma(acc, w[k], in[(size_t)(base + x * stride) * 16u + comp]);
    k += n;
    if (k >= (uint32_t)L) k -= L;
  }
  out[i] = acc;
}

// Pi_{mu nu}(q) = exp(i q.y) exp(-i (q_mu - q_nu)/2) F_{mu nu}(q) - delta_{mu nu} contact_nu,
// F = DFT of conn; tables per direction d: ey[d][n] = exp(2 pi i n y_d / L_d),
// eh[d][n] = exp(-i pi n / L_d).
struct PiqParams {
  uint32_t V, sX, sT;
  int LZ, L[4];
  double2 contact[4];
};
__global__ void k_piq_phase(double2 *__restrict__ piq, const double2 *__restrict__ ey,
                            const double2 *__restrict__ eh, PiqParams P) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= P.V * 16u) return;
  const uint32_t site = i / 16u, comp = i % 16u;
  const int mu = comp / 4, nu = comp % 4;
  uint32_t rem = site;
  uint32_t n[4];
  n[0] = rem / P.sT; rem -= n[0] * P.sT;
  n[1] = rem / P.sX; rem -= n[1] * P.sX;
  n[2] = rem / (uint32_t)P.LZ;
  n[3] = rem - n[2] * (uint32_t)P.LZ;
  double2 f = make_double2(1, 0);
  for (int d = 0; d < 4; d++) f = cmul(f, ey[64 * d + n[d]]);
  f = cmul(f, eh[64 * mu + n[mu]]);
  f = cmulc(eh[64 * nu + n[nu]], f);
  double2 v = cmul(f, piq[i]);
  if (mu == nu) { v.x -= P.contact[nu].x; v.y -= P.contact[nu].y; }
  piq[i] = v;
}

int pi_q_device(cvchip_ctx *c, double2 *dpiq, double2 *tmp, const double contact[8], const int src[4]) {
  const Lattice &Lt = c->lat;
  const uint32_t V = (uint32_t)Lt.V;
  const int Ls[4] = {Lt.T, Lt.LX, Lt.LY, Lt.LZ};
  for (int d = 0; d < 4; d++)
    if (Ls[d] > 64) {
      set_error("Pi(q) supports extents up to 64 (got %d)", Ls[d]);
      return CVCHIP_ERR_ARG;
    }
  const uint32_t strides[4] = {(uint32_t)(Lt.LX * Lt.LY * Lt.LZ), (uint32_t)(Lt.LY * Lt.LZ), (uint32_t)Lt.LZ, 1u};
  double2 hw[4][64], hy[4][64], hh[4][64];
  for (int d = 0; d < 4; d++)
    for (int k = 0; k < 64; k++) {
      const double a = 2.0 * M_PI * (double)(k % Ls[d]) / (double)Ls[d];
      hw[d][k] = make_double2(cos(a), -sin(a));
      const double ay = 2.0 * M_PI * (double)(((int64_t)k * src[d]) % Ls[d]) / (double)Ls[d];
      hy[d][k] = make_double2(cos(ay), sin(ay));
      const double ah = M_PI * (double)k / (double)Ls[d];
      hh[d][k] = make_double2(cos(ah), -sin(ah));
    }
  double2 *tabs = nullptr;
  CVC_HIP(hipMalloc(&tabs, sizeof(double2) * 3 * 256));
  hipError_t e = hipMemcpyAsync(tabs, hw, sizeof(hw), hipMemcpyHostToDevice, c->stream);
  if (e == hipSuccess) e = hipMemcpyAsync(tabs + 256, hy, sizeof(hy), hipMemcpyHostToDevice, c->stream);
  if (e == hipSuccess) e = hipMemcpyAsync(tabs + 512, hh, sizeof(hh), hipMemcpyHostToDevice, c->stream);
  const dim3 g((V * 16u + 255) / 256), b(256);
  double2 *a = dpiq, *o = tmp;
  for (int d = 0; d < 4 && e == hipSuccess; d++) {
    hipLaunchKernelGGL(k_dft_dir, g, b, 0, c->stream, o, (const double2 *)a, (const double2 *)(tabs + 64 * d), V,
                       Ls[d], strides[d]);
    double2 *t = a; a = o; o = t;
  }
  // after 4 passes the result is back in dpiq
  PiqParams P;
  P.V = V;
  P.sX = strides[1];
  P.sT = strides[0];
  P.LZ = Lt.LZ;
  for (int d = 0; d < 4; d++) P.L[d] = Ls[d];
  for (int nu = 0; nu < 4; nu++) P.contact[nu] = make_double2(contact[2 * nu], contact[2 * nu + 1]);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_piq_phase, g, b, 0, c->stream, dpiq, (const double2 *)(tabs + 256),
                       (const double2 *)(tabs + 512), P);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
  (void)hipFree(tabs);
  if (e != hipSuccess) return hip_fail(e, "Pi(q)", __FILE__, __LINE__);
  return 0;
}

}  // namespace cvchip

using namespace cvchip;

extern "C" int cvchip_field_cvc_contract(cvchip_ctx *c, double *conn, double contact[8],
                                         const cvchip_field *up, const cvchip_field *dn, const int src[4]) {
  return cvchip::guarded("cvchip_field_cvc_contract", [&]() -> int {
    if (!c || !conn || !contact || !up || !dn || !src) {
      set_error("NULL argument to cvchip_field_cvc_contract");
      return CVCHIP_ERR_NULL;
    }
    return contract_fields(c, conn, contact, up->f, dn->f, src);
  });
}

extern "C" int cvchip_cvc_contract(cvchip_ctx *c, double *conn, double contact[8], const double *const *props,
                                   const int src[4]) {
  return cvchip::guarded("cvchip_cvc_contract", [&]() -> int {
    if (!c || !conn || !contact || !props || !src) {
      set_error("NULL argument to cvchip_cvc_contract");
      return CVCHIP_ERR_NULL;
    }
    for (int k = 0; k < 120; k++)
      if (!props[k]) {
        set_error("propagator %d is NULL", k);
        return CVCHIP_ERR_NULL;
      }
    TmpField up, dn;
    int rc = field_alloc(c, up, 60, CVCHIP_PREC_F64);
    if (!rc) rc = field_alloc(c, dn, 60, CVCHIP_PREC_F64);
    for (int k = 0; k < 120 && !rc; k++) rc = upload_aos(c, k < 60 ? up : dn, props[k], k % 60, 1);
    if (!rc) rc = contract_fields(c, conn, contact, up, dn, src);
    return rc;
  });
}

extern "C" int cvchip_wi(cvchip_ctx *c, double *wi, const double *conn) {
  return cvchip::guarded("cvchip_wi", [&]() -> int {
    if (!c || !wi || !conn) {
      set_error("NULL argument to cvchip_wi");
      return CVCHIP_ERR_NULL;
    }
    const size_t V = (size_t)c->lat.V;
    double2 *dc = nullptr, *dw = nullptr;
    CVC_HIP(hipMalloc(&dc, sizeof(double2) * 16 * V));
    hipError_t e = hipMalloc(&dw, sizeof(double2) * 4 * V);
    int rc = e == hipSuccess ? 0 : hip_fail(e, "Ward identity buffers", __FILE__, __LINE__);
    if (!rc) rc = copy_to_device(c, dc, conn, sizeof(double2) * 16 * V);
    if (!rc) {
      hipLaunchKernelGGL(k_wi, dim3((unsigned)((V + 255) / 256)), dim3(256), 0, c->stream, dw, (const double2 *)dc,
                         conn_params(c));
      e = hipGetLastError();
      if (e != hipSuccess) rc = hip_fail(e, "Ward identity", __FILE__, __LINE__);
    }
    if (!rc) rc = copy_to_host(c, wi, dw, sizeof(double2) * 4 * V);
    (void)hipStreamSynchronize(c->stream);   // nothing in flight before the buffers go
    (void)hipFree(dc);
    if (dw) (void)hipFree(dw);
    return rc;
  });
}

extern "C" int cvchip_pi_q(cvchip_ctx *c, double *piq, const double *conn, const double contact[8],
                           const int src[4]) {
  return cvchip::guarded("cvchip_pi_q", [&]() -> int {
    if (!c || !piq || !conn || !contact || !src) {
      set_error("NULL argument to cvchip_pi_q");
      return CVCHIP_ERR_NULL;
    }
    const size_t V = (size_t)c->lat.V;
    double2 *a = nullptr, *t = nullptr;
    CVC_HIP(hipMalloc(&a, sizeof(double2) * 16 * V));
    hipError_t e = hipMalloc(&t, sizeof(double2) * 16 * V);
    int rc = e == hipSuccess ? 0 : hip_fail(e, "Pi(q) buffers", __FILE__, __LINE__);
    if (!rc) rc = copy_to_device(c, a, conn, sizeof(double2) * 16 * V);
    if (!rc) rc = pi_q_device(c, a, t, contact, src);
    if (!rc) rc = copy_to_host(c, piq, a, sizeof(double2) * 16 * V);
    (void)hipStreamSynchronize(c->stream);   // nothing in flight before the buffers go
    (void)hipFree(a);
    if (t) (void)hipFree(t);
    return rc;
  });
}

namespace cvchip {

// Up to kBatchSites sites one solve takes the five 12-column sources together:
// 12 columns leave the chip idle there (a launch is then mostly latency) and
// the FP64 updates of the mixed solvers are shared by 60 columns.  One source
// point, five solves of 12 against one of 60 per flavour (even/odd, FP16 /
// FP32 / FP64 inside): 8^4 48 / 55 / 69 -> 15 / 18 / 28 ms, 16x8^3 55 / 63 / 85
// -> 22 / 27 / 55 ms, 16^3x8 90 / 112 / 202 -> 60 / 93 / 202 ms, 32x16^3 256 /
// 356 / 824 -> 238 / 351 / 729 ms.  Beyond, five times the workspaces (23 GB
// at 32x16^3) buy nothing more; without room for them the sources go one by one.
constexpr int64_t kBatchSites = 1 << 17;

int solve_five_sources(cvchip_ctx *c, Field &out, double mu, const std::function<int(Field &, int, int)> &source,
                       double sp, int niter_max, int prec, double delta, cvchip_stats *tot) {
  // solves the 12 ns columns of b into x
  auto solve = [&](Field &x, const Field &b, int ns) -> int {
    CVC_HIP(hipMemsetAsync(x.data, 0, x.bytes, c->stream));
    cvchip_stats st;
    memset(&st, 0, sizeof(st));
    struct Mass {   // the context's own mass again on every path
      cvchip_ctx *c;
      double mu0;
      ~Mass() { c->mu = mu0; }
    };
    int rc;
    {
      const Mass restore{c, c->mu};
      c->mu = mu;
      rc = invert_her_fields(c, x, b, sp, niter_max, prec, delta, 0, &st);
    }
    if (rc < 0 && rc != CVCHIP_ERR_NOCONV) return rc;
    // the sources before the first that did not converge count, as if solved in turn
    int good = 0;
    for (; good < ns; good++) {
      const auto it = c->col_iters.begin() + 12 * good;
      if (*std::min_element(it, it + 12) < 0) break;
      if (tot) tot->iterations += *std::max_element(it, it + 12);   // of the slowest of 12 columns
    }
    if (tot && good) {
      tot->converged += 12 * good;
      tot->reliable_updates += st.reliable_updates;
      tot->dslash_calls += st.dslash_calls;
      tot->seconds += st.seconds;
      if (good == ns && st.true_res2_max > tot->true_res2_max) tot->true_res2_max = st.true_res2_max;
    }
    return rc < 0 ? rc : 0;
  };
  int rc = CVCHIP_ERR_OOM;
  bool held = false;   // out holds the sources (its own columns may have been what source() reads)
  if (c->lat.V <= kBatchSites) {
    TmpField all;
    if (!field_alloc(c, all, 60, CVCHIP_PREC_F64)) {
      CVC_TRY(source(all, 0, 5));
      rc = solve(out, all, 5);
      if (rc == CVCHIP_ERR_OOM) {
        CVC_HIP(hipMemcpyAsync(out.data, all.data, all.bytes, hipMemcpyDeviceToDevice, c->stream));
        held = true;
      }
    }
  }
  if (rc != CVCHIP_ERR_OOM) return rc;
  // one by one, without the room for more than twelve columns
  TmpField b, x;
  CVC_TRY(field_alloc(c, b, 12, CVCHIP_PREC_F64));
  CVC_TRY(field_alloc(c, x, 12, CVCHIP_PREC_F64));
  for (int s = 0; s < 5; s++) {
    CVC_TRY(held ? copy_columns(c, b, 0, out, 12 * s, 12) : source(b, s, 1));
    CVC_TRY(solve(x, b, 1));
    CVC_TRY(copy_columns(c, out, 12 * s, x, 0, 12));
  }
  return 0;
}

// 5 x 12 up (mu) and 5 x 12 down (-mu) propagators from point sources at y + s^
// (s = 0..3) and y (s = 4) into the 60-column sets up / dn (column 12 s + k),
// with the gamma5-hermitian BiCGStab; statistics summed into tot.
int solve_source_props(cvchip_ctx *c, const int src[4], double sp, int niter_max, int prec, double delta,
                       Field &up, Field &dn, cvchip_stats *tot) {
  uint32_t sites[5];
  for (int s = 0; s < 5; s++)
    sites[s] = site_of(c, src[0] + (s == 0), src[1] + (s == 1), src[2] + (s == 2), src[3] + (s == 3));
  auto points = [&](Field &b, int s0, int ns) { return point_sources_at(c, b, ns, sites + s0); };
  CVC_TRY(solve_five_sources(c, up, c->mu, points, sp, niter_max, prec, delta, tot));
  return solve_five_sources(c, dn, -c->mu, points, sp, niter_max, prec, delta, tot);   // down flavour: mu -> -mu (record 1)
}

}  // namespace cvchip

// The whole path for one source point: 60 up and 60 down solves, then the
// contraction.
extern "C" int cvchip_cvc_source(cvchip_ctx *c, double *conn, double contact[8], const int src[4], double sp,
                                 int niter_max, int prec, double delta, cvchip_stats *stats) {
  return cvchip::guarded("cvchip_cvc_source", [&]() -> int {
    if (!c || !conn || !contact || !src) {
      set_error("NULL argument to cvchip_cvc_source");
      return CVCHIP_ERR_NULL;
    }
    TmpField up, dn;
    int rc = field_alloc(c, up, 60, CVCHIP_PREC_F64);
    if (!rc) rc = field_alloc(c, dn, 60, CVCHIP_PREC_F64);
    cvchip_stats tot;
    memset(&tot, 0, sizeof(tot));
    if (!rc) rc = solve_source_props(c, src, sp, niter_max, prec, delta, up, dn, &tot);
    if (!rc) rc = contract_fields(c, conn, contact, up, dn, src);
    if (stats) *stats = tot;
    return rc;
  });
}

// The propagators of cvchip_cvc_source, downloaded into the reference layout.
extern "C" int cvchip_cvc_propagators(cvchip_ctx *c, double *const *props, const int src[4], double sp, int niter_max,
                                      int prec, double delta, cvchip_stats *stats) {
  return cvchip::guarded("cvchip_cvc_propagators", [&]() -> int {
    if (!c || !props || !src) {
      set_error("NULL argument to cvchip_cvc_propagators");
      return CVCHIP_ERR_NULL;
    }
    for (int k = 0; k < 120; k++)
      if (!props[k]) {
        set_error("propagator %d is NULL", k);
        return CVCHIP_ERR_NULL;
      }
    TmpField up, dn;
    int rc = field_alloc(c, up, 60, CVCHIP_PREC_F64);
    if (!rc) rc = field_alloc(c, dn, 60, CVCHIP_PREC_F64);
    cvchip_stats tot;
    memset(&tot, 0, sizeof(tot));
    if (!rc) rc = solve_source_props(c, src, sp, niter_max, prec, delta, up, dn, &tot);
    for (int k = 0; k < 120 && !rc; k++) rc = download_aos(c, k < 60 ? up : dn, props[k], k % 60, 1);
    if (stats) *stats = tot;
    return rc;
  });
}
