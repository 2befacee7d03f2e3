// Twisted-mass Wilson operator on gfx950:
//   xi = D(mutm) phi = 1/(2 kappa) phi + i mutm gamma5 phi
//        - 1/2 sum_mu [ (1 - gamma_mu) U~_mu(x) phi(x+mu) + (1 + gamma_mu) U~_mu(x-mu)^dagger phi(x-mu) ]
// with U~_mu = U_mu * exp(i pi bc_mu / L_mu) (reference Q_phi.c:25-36, 38-188;
// phases cvc_geometry.c:452-459).
//
// One thread per (site, rhs); the rhs index is the fastest-moving index of the
// field layout, so the 64 lanes of a wave read 64 consecutive complex numbers
// of each colour-spin plane and lanes of the same site share link loads.
// Each hop projects the neighbour spinor to two spin components with
// (1 -+ gamma_mu) (rank 2 in the chiral basis), multiplies the half spinor by
// the link, and rebuilds the lower spin components from the upper ones.
// Periodic wrap and the boundary phase are resolved in the kernel: there is no
// halo.  Optional epilogues fuse the solver's per-rhs dot products.
#include <math.h>

#include <algorithm>

#include <type_traits>

#include "spinor_io.h"

namespace cvchip {

// n / d for a divisor fixed for the launch and n < 2^31: a shift for d = 2^l
// (m = 0, a branch uniform across the grid); else, with l = ceil(log2 d) and
// m = ceil(2^(31 + l) / d), m d exceeds 2^(31 + l) by less than 2^l, so the
// quotient of n m by 2^(31 + l) is exact: one high product and a shift, on the
// scalar unit where n is uniform (a 32-bit division is about 20 instructions).
struct FDiv {
  uint32_t m;
  int sh;
};
static FDiv make_fdiv(uint32_t d) {
  int l = 0;
  while (((uint64_t)1 << l) < d) l++;
  if (((uint64_t)1 << l) == d) return FDiv{0u, l};
  const uint64_t p = (uint64_t)1 << (31 + l);
  return FDiv{(uint32_t)((p + d - 1) / d), l - 1};
}
__device__ __forceinline__ uint32_t fdiv(uint32_t n, FDiv f) { return f.m ? __umulhi(n, f.m) >> f.sh : n >> f.sh; }

template <typename R>
struct DParams {
  uint32_t V, VN, sX, sT;
  int N, T, LX, LY, LZ;
  // coordinates of a traversal index, and the quotients of the block index
  FDiv fLZt, fLY, fLX, fT, fbpc, fbpcol, fbpp, fbpr, fncx, fslice, fncy, fncz;
  // 1/N and 1/S for the small quotients of thread and staging indices
  float invN, invS;
  // traversal (mode 1): the lattice is cut into chunks of csz consecutive
  // sites (one eighth of a time slice when possible), bpc blocks per chunk;
  // the 8 XCDs take the 8 chunks of a time slice side by side, so the whole
  // GPU advances through the slices together.  Mode 0: the same chunks with
  // no XCD interleave.  Mode 2: XCD j owns the time slices t = j mod 8 and
  // walks each slice in runs of yb consecutive y rows (yb*LZ consecutive
  // sites), x within y block: the x and y neighbours of a run were touched a
  // few runs earlier and are still in the XCD's L2, and the t neighbours are
  // the slices the adjacent XCDs are working on at the same time.
  // Mode 4: columns of bx x-planes x yb y-rows (all z) swept in t, slice by
  // slice.  The (column, slice) pairs, slices fastest, are cut into eight runs
  // of npx, one per XCD: the sites in flight on an XCD form a compact 4D region
  // and its t neighbours are one cross-section away, whether or not the columns
  // divide by eight.
  // Mode 5: columns of bx x-planes x yb y-rows x zb z-sites (powers of two)
  // swept along the whole t extent, one column at a time per XCD, with the
  // column's sites ordered z, y, x within a time slice: the t neighbour of a
  // site lies one cross-section (bx yb zb sites, a few blocks) ahead in the
  // sweep, inside the XCD's L2 window even for 12 rhs in FP64.
  uint32_t csz, bpc;
  int mode;
  uint32_t yb, runlen, bpr, nrun;
  uint32_t bx, ncx, bpp, npx, npair, bpcol;   // mode 4: bpp blocks per pair, npair pairs
  uint32_t zb, ncy, ncz, lzb, lyz, lA, colsz, sTt, sXt;
  // Mode 6 (k_dslash_march): mS columns per workgroup marched through mM
  // slices; patches of mXP x mYP x LZ columns (mNPX along x), mCP chunks of mS
  // columns per patch, mNR = T / mM slice ranges; mXcd: patch p on XCD p mod 8.
  uint32_t mS, mM, mXP, mYP, mCP, mNR, mNPX;
  int mXcd;
  int nt;       // streaming output stores
  int nt_own;   // even/odd: streaming loads of the own spinors
  // Even/odd operator (EO kernels): the traversal runs over the half lattice
  // (T, LX, LY, LZ/2); half-site h of parity par is the lexicographic site
  // with z = 2 (h mod LZ/2) + ((par + t + x + y) mod 2), i.e. lex = 2h or 2h+1.
  // The epilogue forms, with A = 1/(2 kappa) + i mutm gamma5 on the output
  // parity and hop the hopping sum:
  //   dmode 0: A own + hopc hop     1: A^-1 (hopc hop)
  //   dmode 2: own + hopc hop       3: A^-1 (own + hopc hop)
  uint32_t LZt;   // z extent of the traversal (LZ, or LZ/2 for EO)
  int par, dmode;
  R hopc, dinv;   // dinv = 1 / ((1/(2 kappa))^2 + mutm^2)
  R k2, mutm;
  cplx<R> ph[4];
  // converged right-hand sides of a running solve (done[r * dstride] != 0):
  // their lanes compute and store nothing
  const int *done;
  int dstride;
};

// floor(n / d) for n < 2^21 from inv, the float nearest 1/d (or within two
// roundings of it): (n + 1/2) / d stays at least 1/(2d) away from an integer,
// and the float product errs by less than (n + 1/2) 2^-22 / d
__device__ __forceinline__ uint32_t sdiv(uint32_t n, float inv) { return (uint32_t)(((float)n + 0.5f) * inv); }

// Spin projection of a neighbour spinor: h[a] = psi_a -+ g_a psi_{GCOL[a]}
// for the upper spins a = 0, 1 ((1 -+ gamma_mu) has rank 2 in the chiral
// basis).  get(c) returns component c = 3*spin + colour; FP64 loads each
// component where it is used, so no more than the half spinor and one pair of
// spin rows are live at a time.
template <int MU, bool FWD, typename C, typename Get>
__device__ __forceinline__ void project(C h[2][3], Get get) {
  constexpr int p0 = GCOL[MU][0], p1 = GCOL[MU][1];
  constexpr int g0 = FWD ? uneg(GVAL[MU][0]) : GVAL[MU][0];
  constexpr int g1 = FWD ? uneg(GVAL[MU][1]) : GVAL[MU][1];
#pragma unroll
  for (int c = 0; c < 3; c++) h[0][c] = cadd(get(c), cunit<g0>(get(3 * p0 + c)));
#pragma unroll
  for (int c = 0; c < 3; c++) h[1][c] = cadd(get(3 + c), cunit<g1>(get(3 * p1 + c)));
}

// FP16 storage: the projection of the stored halves, each output real one
// mixed-precision FMA of half operands (exact sums of two halves, rounded once
// to FP32; `one` is 1.0f, opaque to the compiler, which otherwise converts both
// halves and adds).  The site's scale multiplies the link product where it is
// added to the accumulator.
__device__ __forceinline__ float half_lo(uint32_t w) {
  return (float)__builtin_bit_cast(_Float16, (unsigned short)(w & 0xffffu));
}
__device__ __forceinline__ float half_hi(uint32_t w) {
  return (float)__builtin_bit_cast(_Float16, (unsigned short)(w >> 16));
}
template <int U>
__device__ __forceinline__ float2 half_pair(uint32_t A, uint32_t B, float one) {
  if constexpr (U == 0) return make_float2(__builtin_fmaf(half_lo(B), one, half_lo(A)), __builtin_fmaf(half_hi(B), one, half_hi(A)));
  else if constexpr (U == 1) return make_float2(__builtin_fmaf(half_lo(B), -one, half_lo(A)), __builtin_fmaf(half_hi(B), -one, half_hi(A)));
  else if constexpr (U == 2) return make_float2(__builtin_fmaf(half_hi(B), -one, half_lo(A)), __builtin_fmaf(half_lo(B), one, half_hi(A)));
  else return make_float2(__builtin_fmaf(half_hi(B), one, half_lo(A)), __builtin_fmaf(half_lo(B), -one, half_hi(A)));
}
template <int MU, bool FWD>
__device__ __forceinline__ void project_half(float2 h[2][3], const uint32_t w[12], float one) {
  constexpr int p0 = GCOL[MU][0], p1 = GCOL[MU][1];
  constexpr int g0 = FWD ? uneg(GVAL[MU][0]) : GVAL[MU][0];
  constexpr int g1 = FWD ? uneg(GVAL[MU][1]) : GVAL[MU][1];
#pragma unroll
  for (int c = 0; c < 3; c++) h[0][c] = half_pair<g0>(w[c], w[3 * p0 + c], one);
#pragma unroll
  for (int c = 0; c < 3; c++) h[1][c] = half_pair<g1>(w[3 + c], w[3 * p1 + c], one);
}

// acc += (1 - gamma_MU) U ph psi (FWD) or (1 + gamma_MU) U^dagger conj(ph) psi
// (!FWD), from the projected h: one colour row of the link at a time,
// w_a = row . h_a, then the upper spins take w_a and the lower spins
// -+g_b w_{GCOL[b]}.  base[k * stride] is the stored link entry k (9 entries,
// or the first two rows, the third rebuilt as conj(row0 x row1)).
// third row of an SU(3) link from its first two: conj(row0 x row1)
template <typename C>
__device__ __forceinline__ void rebuild_row3(C u[9]) {
  const C a = csub(cmul(u[1], u[5]), cmul(u[2], u[4]));
  const C b = csub(cmul(u[2], u[3]), cmul(u[0], u[5]));
  const C d = csub(cmul(u[0], u[4]), cmul(u[1], u[3]));
  u[6] = mk<decltype(a.x)>(a.x, -a.y);
  u[7] = mk<decltype(a.x)>(b.x, -b.y);
  u[8] = mk<decltype(a.x)>(d.x, -d.y);
}

// a + u n b for the unit code U of cunit (SCALED), or a + u b
template <int U, bool SCALED, typename C, typename R>
__device__ __forceinline__ C add_unit(C a, C b, R n) {
  if constexpr (!SCALED) return cadd(a, cunit<U>(b));
  else if constexpr (U == 0) return mk<R>(fmar(n, b.x, a.x), fmar(n, b.y, a.y));
  else if constexpr (U == 1) return mk<R>(fmar(-n, b.x, a.x), fmar(-n, b.y, a.y));
  else if constexpr (U == 2) return mk<R>(fmar(-n, b.y, a.x), fmar(n, b.x, a.y));
  else return mk<R>(fmar(n, b.y, a.x), fmar(-n, b.x, a.y));
}

// PHASE false: the entries at base already carry the boundary phase; SCALED:
// the spinor's scale n multiplies the product (FP16 storage)
template <typename R, int RECON, int MU, bool FWD, bool PHASE = true, bool SCALED = false>
__device__ __forceinline__ void link_apply(cplx<R> acc[12], const cplx<R> h[2][3],
                                           const cplx<R> *__restrict__ base, uint32_t stride, cplx<R> ph, R n = 1) {
  using C = cplx<R>;
  constexpr int q2 = GCOL[MU][2], q3 = GCOL[MU][3];
  constexpr int l2 = FWD ? uneg(GVAL[MU][2]) : GVAL[MU][2];
  constexpr int l3 = FWD ? uneg(GVAL[MU][3]) : GVAL[MU][3];
  C u[9];
  if constexpr (RECON == 12) {
#pragma unroll
    for (int k = 0; k < 6; k++) u[k] = base[(size_t)k * stride];
    rebuild_row3(u);
  }
#pragma unroll
  for (int i = 0; i < 3; i++) {
    C w0 = mk<R>(0, 0), w1 = mk<R>(0, 0);
#pragma unroll
    for (int j = 0; j < 3; j++) {
      const int k = FWD ? 3 * i + j : 3 * j + i;
      const C e = RECON == 18 ? base[(size_t)k * stride] : u[k];
      if constexpr (FWD) {
        w0 = cfma(w0, e, h[0][j]);
        w1 = cfma(w1, e, h[1][j]);
      } else {
        w0 = cfmac(w0, e, h[0][j]);
        w1 = cfmac(w1, e, h[1][j]);
      }
    }
    if constexpr (!PHASE) {
    } else if constexpr (FWD) {
      w0 = cmul(ph, w0);
      w1 = cmul(ph, w1);
    } else {
      w0 = cmulc(ph, w0);
      w1 = cmulc(ph, w1);
    }
    acc[i] = add_unit<0, SCALED>(acc[i], w0, n);
    acc[3 + i] = add_unit<0, SCALED>(acc[3 + i], w1, n);
    acc[6 + i] = add_unit<l2, SCALED>(acc[6 + i], q2 == 0 ? w0 : w1, n);
    acc[9 + i] = add_unit<l3, SCALED>(acc[9 + i], q3 == 0 ? w0 : w1, n);
  }
}

// Links of a block staged in LDS: [8 hops][KL entries][LDS_SITES], hop 2*mu is
// U_mu(x - mu) (backward), 2*mu + 1 is U_mu(x) (forward).
constexpr int LDS_SITES = 32;

// A neighbour spinor as it is stored: loaded whole, projected later, so that
// the loads of the next hop can be in flight during the products of this one.
template <typename IO> struct Raw;
template <> struct Raw<IOPlain<double>> {
  double2 v[12];
  __device__ __forceinline__ void load(const IOPlain<double> &in, uint32_t idx) { in.load(v, idx); }
  __device__ __forceinline__ void load_nt(const IOPlain<double> &in, uint32_t idx) { in.load_nt(v, idx); }
  __device__ __forceinline__ void full(double2 o[12]) const {
#pragma unroll
    for (int c = 0; c < 12; c++) o[c] = v[c];
  }
  template <int MU, bool FWD> __device__ __forceinline__ double project(double2 h[2][3], double) const {
    cvchip::project<MU, FWD>(h, [&](int c) { return v[c]; });
    return 1.;
  }
};
template <> struct Raw<IOPlain<float>> {
  float2 v[12];
  __device__ __forceinline__ void load(const IOPlain<float> &in, uint32_t idx) { in.load(v, idx); }
  __device__ __forceinline__ void load_nt(const IOPlain<float> &in, uint32_t idx) { in.load_nt(v, idx); }
  __device__ __forceinline__ void full(float2 o[12]) const {
#pragma unroll
    for (int c = 0; c < 12; c++) o[c] = v[c];
  }
  template <int MU, bool FWD> __device__ __forceinline__ float project(float2 h[2][3], float) const {
    cvchip::project<MU, FWD>(h, [&](int c) { return v[c]; });
    return 1.f;
  }
};
template <> struct Raw<IOHalf> {
  uint32_t w[12];
  float n;
  __device__ __forceinline__ void load(const IOHalf &in, uint32_t idx) {
    const uint4 *q = reinterpret_cast<const uint4 *>(in.p);
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const uint4 v = q[(size_t)k * in.VN + idx];
      w[4 * k] = v.x;
      w[4 * k + 1] = v.y;
      w[4 * k + 2] = v.z;
      w[4 * k + 3] = v.w;
    }
    n = in.nrm[idx];
  }
  __device__ __forceinline__ void load_nt(const IOHalf &in, uint32_t idx) {
    typedef unsigned u4v __attribute__((ext_vector_type(4)));
    const u4v *q = reinterpret_cast<const u4v *>(in.p);
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const u4v v = __builtin_nontemporal_load(q + (size_t)k * in.VN + idx);
      w[4 * k] = v.x;
      w[4 * k + 1] = v.y;
      w[4 * k + 2] = v.z;
      w[4 * k + 3] = v.w;
    }
    n = __builtin_nontemporal_load(in.nrm + idx);
  }
  __device__ __forceinline__ void full(float2 o[12]) const {
#pragma unroll
    for (int c = 0; c < 12; c++) o[c] = make_float2(half_lo(w[c]) * n, half_hi(w[c]) * n);
  }
  template <int MU, bool FWD> __device__ __forceinline__ float project(float2 h[2][3], float one) const {
    project_half<MU, FWD>(h, w, one);
    return n;
  }
};
template <typename IO> struct IsHalf { static constexpr bool value = false; };
template <> struct IsHalf<IOHalf> { static constexpr bool value = true; };

// Projected neighbour spinors, returning the scale that their link product
// takes.  With LDSS the block's own sites and the two sites before and after
// them are staged in LDS (scales applied), so the z neighbours (adjacent sites)
// and the own spinor come from LDS instead of the texture path.
template <typename IO, bool LDSS>
struct NbLoader {
  using R = typename IO::real;
  using C = cplx<R>;
  const IO &in;
  const C *Sp;
  uint32_t N, r, s0, S;
  R one;
  // the staged slot of site, or -1
  __device__ __forceinline__ int slot(uint32_t site, bool from_lds) const {
    if constexpr (LDSS) {
      if (from_lds) {
        const int64_t d = (int64_t)site - (int64_t)s0 + 1;
        if (d >= 0 && d <= (int64_t)S + 1) return (int)d;
      }
    }
    return -1;
  }
  template <int MU, bool FWD>
  __device__ __forceinline__ R proj(C h[2][3], uint32_t site, bool from_lds) const {
    const int d = slot(site, from_lds);
    if (d >= 0) {
      const C *q = Sp + (uint32_t)d * 12 * N + r;
      project<MU, FWD>(h, [&](int c) { return q[c * N]; });
      return (R)1;
    }
    const uint32_t idx = site * N + r;
    if constexpr (IO::K == 1) {   // each component loaded where it is used
      project<MU, FWD>(h, [&](int c) { return in.load_c(c, idx); });
      return (R)1;
    } else {
      Raw<IO> raw;
      raw.load(in, idx);
      return raw.template project<MU, FWD>(h, one);
    }
  }
  __device__ __forceinline__ void full(C v[12], uint32_t site, bool from_lds) const {
    const int d = slot(site, from_lds);
    if (d >= 0) {
#pragma unroll
      for (int c = 0; c < 12; c++) v[c] = Sp[((uint32_t)d * 12 + c) * N + r];
      return;
    }
    in.load(v, site * N + r);
  }
};

// Bounds a hop: an empty asm that reads and writes the accumulator (and the
// projected half spinor) and clobbers memory, so that its arithmetic is done
// before and the loads that follow cannot move above it (the compiler otherwise
// issues the loads of all eight hops first, keeps every loaded value live and
// runs one wave per SIMD).
template <typename C>
__device__ __forceinline__ void pin_regs(C *v, int n) {
#pragma unroll
  for (int k = 0; k < n; k++) asm volatile("" : "+v"(v[k].x), "+v"(v[k].y) : : "memory");
}

// A thread's output site: traversal coordinates (zt counts half-sites on the
// even/odd lattice), traversal index v, lexicographic site s, and there the
// offset s - 2 v of an even/odd half-site.
struct SitePos {
  uint32_t t, x, y, zt, v, s, off;
};

// Hop h = 2 mu (backward) or 2 mu + 1 (forward): traversal index of the
// neighbour.  A t, x or y neighbour on the even/odd lattice has the same zt
// (its parity and the coordinate change together); the z neighbours of offset
// off are zt - 1 + off and zt + off.
template <int H, bool EO, typename R>
__device__ __forceinline__ uint32_t neighbour(const SitePos &q, const DParams<R> &P) {
  constexpr int MU = H >> 1;
  constexpr bool FWD = (H & 1) != 0;
  const uint32_t crd = MU == 0 ? q.t : MU == 1 ? q.x : MU == 2 ? q.y : q.zt;
  const uint32_t L = (uint32_t)(MU == 0 ? P.T : MU == 1 ? P.LX : MU == 2 ? P.LY : (int)P.LZt);
  const uint32_t str = MU == 0 ? P.sTt : MU == 1 ? P.sXt : MU == 2 ? P.LZt : 1u;
  const uint32_t nb = FWD ? (crd == L - 1 ? q.v - (L - 1) * str : q.v + str)
                          : (crd == 0 ? q.v + (L - 1) * str : q.v - str);
  if constexpr (EO && MU == 3) return (q.off != 0) == FWD ? nb : q.v;
  return nb;
}

// the site whose link the hop takes: s (forward), s - mu (backward)
template <bool EO, typename R>
__device__ __forceinline__ uint32_t link_site(const SitePos &q, const DParams<R> &P, int mu, bool fwd) {
  if (fwd) return q.s;
  const uint32_t crd = mu == 0 ? q.t : mu == 1 ? q.x : mu == 2 ? q.y : (EO ? 2u * q.zt + q.off : q.zt);
  const uint32_t L = (uint32_t)(mu == 0 ? P.T : mu == 1 ? P.LX : mu == 2 ? P.LY : P.LZ);
  const uint32_t str = mu == 0 ? P.sT : mu == 1 ? P.sX : mu == 2 ? (uint32_t)P.LZ : 1u;
  return crd == 0 ? q.s + (L - 1) * str : q.s - str;
}

// one hop from the projected spinor h of scale n; links from LDS (Ul, slot sl) or memory
template <typename IO, int RECON, int H, bool LDSL, bool EO>
__device__ __forceinline__ void hop_links(cplx<typename IO::real> acc[12], const cplx<typename IO::real> h[2][3],
                                          typename IO::real n, const cplx<typename IO::real> *__restrict__ U,
                                          const cplx<typename IO::real> *__restrict__ Ul,
                                          const DParams<typename IO::real> &P, const SitePos &q, uint32_t sl) {
  using R = typename IO::real;
  constexpr int MU = H >> 1;
  constexpr bool FWD = (H & 1) != 0;
  constexpr int KL = RECON == 18 ? 9 : 6;
  // staged whole with the phase applied (see k_dslash): read as full links, no phase multiply
  constexpr bool FOLD = LDSL && RECON == 12 && sizeof(R) == 4;
  constexpr int KS = FOLD ? 9 : KL;
  constexpr int RL = FOLD ? 18 : RECON;
  constexpr bool SC = IsHalf<IO>::value;
  if constexpr (LDSL) link_apply<R, RL, MU, FWD, !FOLD, SC>(acc, h, Ul + H * KS * LDS_SITES + sl, LDS_SITES, P.ph[MU], n);
  else link_apply<R, RECON, MU, FWD, true, SC>(acc, h, U + (size_t)MU * KL * P.V + link_site<EO>(q, P, MU, FWD), P.V,
                                               P.ph[MU], n);
}

// Hop H of the multi-rhs operator with its neighbour in raw, and the loads of
// hop H + 1 (after the last, the own spinor's) in flight during the products of
// this one: each wave has up to two neighbours' loads outstanding.  What bounds
// the kernel: a wave's 108 (FP64) 1 KB loads mostly miss the 32 KB L1, and about
// 40 % of them the XCD's L2; the FP64 kernel needs 182 VGPRs with the second
// spinor in flight, so two waves per SIMD instead of four, which read 15.6
// instead of 19.4 GB from beyond L2 at 64x32^3 with 12 rhs.  Together with the
// batched link staging, the columns and the scalar index arithmetic, 12 rhs
// (before -> now): FP64 64x32^3 3.90 -> 3.51 ms, 40x20^3 649 -> 510 us, 32x16^3
// 246 -> 200 us; even/odd at 40x20^3 FP64 375 -> 265 us, FP32 188 -> 150 us,
// FP16 108 -> 85 us.
template <typename IO, int RECON, int H, bool EO>
__device__ __forceinline__ void hop_pipelined(cplx<typename IO::real> acc[12], Raw<IO> &raw, const IO &in,
                                              const IO &own, typename IO::real one, const cplx<typename IO::real> *__restrict__ Ul,
                                              const DParams<typename IO::real> &P, const SitePos &q, uint32_t r,
                                              uint32_t sl) {
  using R = typename IO::real;
  cplx<R> h[2][3];
  Raw<IO> next;
  if constexpr (H < 7) next.load(in, neighbour<H + 1, EO>(q, P) * (uint32_t)P.N + r);
  else if constexpr (!EO) next.load(in, q.v * (uint32_t)P.N + r);
  else if (P.dmode != 1) {
    if (P.nt_own) next.load_nt(own, q.v * (uint32_t)P.N + r);
    else next.load(own, q.v * (uint32_t)P.N + r);
  }
  asm volatile("" : : : "memory");
  const R n = raw.template project<(H >> 1), (H & 1) != 0>(h, one);
  hop_links<IO, RECON, H, true, EO>(acc, h, n, nullptr, Ul, P, q, sl);
  pin_regs(acc, 12);
  raw = next;
}

// the same without LDS links or with staged spinors: load, project, multiply.
// Links from memory (N < 8): the compiler issues the loads of all hops that nothing
// bounds at once.  One rhs gains by that (FEW: FP32 of one rhs unbounded, FP64 of
// one and two bounded once, after four hops); more rhs re-read less and gain by a
// second wave instead: FP32 bounded after three hops (48x24^3, 2 / 4 / 6 rhs: 136 /
// 232 / 346 us against 142 / 243 / 363 us unbounded; one rhs 72 against 66 us), FP64
// after three and six (48x24^3, 1 / 2 / 4 / 7 rhs: 185 / 265 / 444 / 752 us, after four
// hops at one wave 166 / 262 / 473 / 892 us, unbounded 169 / 265 / 481 / 880 us).  These
// are the whole-lattice kernels, none of which spills; the bounds were not measured on
// the even/odd ones, which do: FP32 127-156 registers with one rhs (616 B of
// scratch) and 3-32 with more, FP16 50-103, FP64 21-76 from three rhs (up to 10
// below).
template <typename IO, int RECON, int H, bool LDSL, bool LDSS, bool EO, bool FEW>
__device__ __forceinline__ void hop_plain(cplx<typename IO::real> acc[12], const NbLoader<IO, LDSS> &ld,
                                          const cplx<typename IO::real> *__restrict__ U,
                                          const cplx<typename IO::real> *__restrict__ Ul,
                                          const DParams<typename IO::real> &P, const SitePos &q, uint32_t sl) {
  using R = typename IO::real;
  cplx<R> h[2][3];
  const R n = ld.template proj<(H >> 1), (H & 1) != 0>(h, neighbour<H, EO>(q, P), (H >> 1) == 3);
  if constexpr (LDSL) pin_regs(&h[0][0], 6);
  hop_links<IO, RECON, H, LDSL, EO>(acc, h, n, U, Ul, P, q, sl);
  constexpr bool bound = IO::K == 1 ? (FEW ? H == 3 : H == 2 || H == 5) : IO::K == 2 && !FEW && H == 2;
  if constexpr (LDSL || bound) pin_regs(acc, 12);
}

// Minimum resident waves per SIMD the register allocation must allow (the
// compiler otherwise hoists every neighbour load and ends at one wave).  Links from
// memory (few rhs) in FP32 and FP16: two, at three the whole-lattice FP32 kernel
// spills (48x24^3, one / six rhs: 96 / 472 us against 66 / 346 us).
#ifndef CVC_DSLASH_WAVES64
#define CVC_DSLASH_WAVES64 1
#endif
#ifndef CVC_DSLASH_WAVES32
#define CVC_DSLASH_WAVES32 3
#endif
template <typename R, bool LDSL, bool FEW> struct DslashWaves {
  static constexpr int value = sizeof(R) == 8 ? (LDSL || FEW ? CVC_DSLASH_WAVES64 : 2) : LDSL ? CVC_DSLASH_WAVES32 : 2;
};

// A thread's terms of the fused dot products (DotMode): o the output, q the own
// spinor, w the shadow residual; products in FP64: squares of a small-scale rhs
// underflow FP32
template <int DM, typename C>
__device__ __forceinline__ void add_dots(double *dv, const C o[12], const C q[12], const C w[12]) {
  double a = 0, b = 0, n = 0, ra = 0, rb = 0;
#pragma unroll
  for (int c = 0; c < 12; c++) {
    const double ox = o[c].x, oy = o[c].y;
    if constexpr (DM == DOT_TS || DM == DOT_TSR) {
      const double qx = q[c].x, qy = q[c].y;
      a += ox * qx + oy * qy;
      b += ox * qy - oy * qx;
    }
    if constexpr (DM != DOT_R2) n += ox * ox + oy * oy;
    if constexpr (dot_shadow(DM)) {
      const double wx = w[c].x, wy = w[c].y;
      ra += wx * ox + wy * oy;
      rb += wx * oy - wy * ox;
    }
  }
  int k = 0;
  if constexpr (DM == DOT_TS || DM == DOT_TSR) { dv[k++] += a; dv[k++] += b; }
  if constexpr (DM == DOT_TS || DM == DOT_TSR || DM == DOT_NN || DM == DOT_NNR) dv[k++] += n;
  if constexpr (dot_shadow(DM)) { dv[k++] += ra; dv[k++] += rb; }
}

// LDSL: the block's sites share their links through LDS (N >= 8, at most
// LDS_SITES sites per block): every link entry crosses the texture path once
// per block instead of once per rhs lane.
// IOR: the storage of r2, the shadow residual of the <r2, out> epilogue (the
// FP32 mixed solver keeps it in FP16 with a per-site scale)
// FEW: one or two rhs (see hop_plain)
template <typename IOI, typename IOO, int RECON, bool G5OUT, int DM, bool LDSL, bool LDSS, bool EO, typename IOR = IOI,
          bool FEW = false>
__global__ void __launch_bounds__(256, (DslashWaves<typename IOI::real, LDSL, FEW>::value))
k_dslash(IOO out, IOI in, IOI own_f, const cplx<typename IOI::real> *__restrict__ U,
         DParams<typename IOI::real> P, IOR r2, double *__restrict__ part) {
  using R = typename IOI::real;
  using C = cplx<R>;
  constexpr int KL = RECON == 18 ? 9 : 6;
  static_assert(!(EO && LDSS), "the even/odd operator stages no spinors");
  const uint32_t S = blockDim.x / (uint32_t)P.N;
  // The block's range of slots, from the block index by scalar quotients.
  // Rows (modes 2, 4): slots j0 .. of a run of yb rows at (t0, x0, y0).
  // Chunks (modes 0, 1): consecutive traversal indices j0 .. jend.  Mode 5: slots
  // j0 .. of a column at (x0, y0, zt0).
  const uint32_t bx8 = blockIdx.x / kXcds, b8 = blockIdx.x % kXcds;
  uint32_t t0 = 0, x0 = 0, y0 = 0, z0 = 0, j0, jend;
  if (P.mode == 4) {
    const uint32_t k = fdiv(bx8, P.fbpp), rem = bx8 - k * P.bpp;
    const uint32_t xin = fdiv(rem, P.fbpr), blk = rem - xin * P.bpr;
    const uint32_t pair = b8 * P.npx + k;
    const uint32_t col = fdiv(pair, P.fT), cy = fdiv(col, P.fncx);
    t0 = pair - col * (uint32_t)P.T;
    x0 = (col - cy * P.ncx) * P.bx + xin;
    y0 = cy * P.yb;
    j0 = blk * S;
    jend = pair < P.npair ? P.runlen : 0u;   // the last XCD's run may be shorter
  } else if (P.mode == 2) {
    const uint32_t tl = fdiv(bx8, P.fslice), rem = bx8 - tl * (P.nrun * P.bpr);
    const uint32_t run = fdiv(rem, P.fbpr), blk = rem - run * P.bpr;
    const uint32_t ybl = fdiv(run, P.fLX);
    t0 = tl * kXcds + b8;
    x0 = run - ybl * (uint32_t)P.LX;
    y0 = ybl * P.yb;
    j0 = blk * S;
    jend = P.runlen;
  } else if (P.mode == 5) {
    const uint32_t cl = fdiv(bx8, P.fbpcol), col = cl * kXcds + b8;
    const uint32_t q = fdiv(col, P.fncz), cx = fdiv(q, P.fncy);
    z0 = (col - q * P.ncz) * P.zb;
    y0 = (q - cx * P.ncy) * P.yb;
    x0 = cx * P.bx;
    j0 = (bx8 - cl * P.bpcol) * S;
    jend = P.colsz;
  } else {
    uint32_t chunk, blk;
    if (P.mode == 1) {
      const uint32_t k = fdiv(bx8, P.fbpc);
      chunk = k * kXcds + b8;
      blk = bx8 - k * P.bpc;
    } else {
      chunk = fdiv(blockIdx.x, P.fbpc);
      blk = blockIdx.x - chunk * P.bpc;
    }
    j0 = chunk * P.csz + blk * S;
    jend = (chunk + 1) * P.csz;
  }
  const uint32_t vrow = ((t0 * (uint32_t)P.LX + x0) * (uint32_t)P.LY + y0) * P.LZt;   // rows: traversal index of slot 0
  // position of block slot sl; false past the end of the block's range
  auto slot_pos = [&](uint32_t sl, SitePos &q) -> bool {
    const uint32_t j = j0 + sl;
    if (j >= jend) return false;
    if (P.mode == 2 || P.mode == 4) {
      const uint32_t dy = fdiv(j, P.fLZt);
      q.t = t0;
      q.x = x0;
      q.y = y0 + dy;
      q.zt = j - dy * P.LZt;
      q.v = vrow + j;
    } else if (P.mode == 5) {
      const uint32_t rem = j & ((1u << P.lA) - 1u);
      q.t = j >> P.lA;
      q.x = x0 + (rem >> P.lyz);
      q.y = y0 + ((rem >> P.lzb) & (P.yb - 1u));
      q.zt = z0 + (rem & (P.zb - 1u));
      q.v = ((q.t * (uint32_t)P.LX + q.x) * (uint32_t)P.LY + q.y) * P.LZt + q.zt;
    } else {
      uint32_t k = fdiv(j, P.fLZt);
      q.zt = j - k * P.LZt;
      const uint32_t k2 = fdiv(k, P.fLY);
      q.y = k - k2 * (uint32_t)P.LY;
      q.t = fdiv(k2, P.fLX);
      q.x = k2 - q.t * (uint32_t)P.LX;
      q.v = j;
    }
    q.off = EO ? ((uint32_t)P.par + q.t + q.x + q.y) & 1u : 0u;
    q.s = EO ? 2u * q.v + q.off : q.v;
    return true;
  };
  const uint32_t sl = sdiv(threadIdx.x, P.invN);
  const uint32_t r = threadIdx.x - sl * (uint32_t)P.N;
  SitePos q;
  const bool active = slot_pos(sl, q) && !(P.done && P.done[(size_t)r * P.dstride]);
  double dv[dot_rows(DM) > 0 ? dot_rows(DM) : 1] = {};
  // FP32 / FP16 with 2-row links: the staged links are whole (third row rebuilt)
  // and carry the boundary phase, both done once per site here instead of once
  // per rhs lane in every hop (the multi-rhs kernels in these precisions are
  // bound by their arithmetic)
  constexpr bool FOLD = LDSL && RECON == 12 && sizeof(R) == 4;
  constexpr int KS = FOLD ? 9 : KL;
  __shared__ C Ul[LDSL ? 8 * KS * LDS_SITES : 1];
  // the first neighbour's loads are in flight while the links are staged
  constexpr bool PIPE = LDSL && !LDSS;
  Raw<IOI> raw;
  if constexpr (PIPE) {
    if (active) raw.load(in, neighbour<0, EO>(q, P) * (uint32_t)P.N + r);
    asm volatile("" : : : "memory");
  }
  if constexpr (FOLD) {
    for (uint32_t e = threadIdx.x; e < 8u * S; e += blockDim.x) {
      const uint32_t hopi = sdiv(e, P.invS), sle = e - hopi * S;
      SitePos qe;
      if (!slot_pos(sle, qe)) continue;
      const int mu = (int)(hopi >> 1);
      const uint32_t ls = link_site<EO>(qe, P, mu, (hopi & 1u) != 0);
      C u[9];
#pragma unroll
      for (int k = 0; k < 6; k++) u[k] = U[((size_t)mu * 6 + k) * P.V + ls];
      rebuild_row3(u);
#pragma unroll
      for (int k = 0; k < 9; k++) Ul[(hopi * 9 + k) * LDS_SITES + sle] = cmul(u[k], P.ph[mu]);
    }
    __syncthreads();
  } else if constexpr (LDSL) {
    // all entries of a link in flight together: one memory latency per block
    for (uint32_t e = threadIdx.x; e < 8u * S; e += blockDim.x) {
      const uint32_t hopi = sdiv(e, P.invS), sle = e - hopi * S;
      SitePos qe;
      if (!slot_pos(sle, qe)) continue;
      const int mu = (int)(hopi >> 1);
      const uint32_t ls = link_site<EO>(qe, P, mu, (hopi & 1u) != 0);
      C u[KL];
#pragma unroll
      for (int k = 0; k < KL; k++) u[k] = U[((size_t)mu * KL + k) * P.V + ls];
#pragma unroll
      for (int k = 0; k < KL; k++) Ul[(hopi * KL + k) * LDS_SITES + sle] = u[k];
    }
    __syncthreads();
  }
  extern __shared__ unsigned char dyn_lds[];
  C *Sp = reinterpret_cast<C *>(dyn_lds);
  uint32_t s0 = 0;   // first traversal index of the block's (contiguous) range
  if constexpr (LDSS) {
    s0 = P.mode == 2 || P.mode == 4 ? vrow + j0 : j0;
    // stage sites s0-1 .. s0+S (all rhs); (s0 - 1 + k) mod V, every index is a valid site
    const uint32_t nst = (S + 2) * (uint32_t)P.N;
    for (uint32_t u = threadIdx.x; u < nst; u += blockDim.x) {
      const uint32_t k = u / (uint32_t)P.N, rr = u - k * (uint32_t)P.N;
      const uint32_t site = (s0 + P.V - 1 + k) % P.V;
      C v[12];
      in.load(v, site * (uint32_t)P.N + rr);
#pragma unroll
      for (int c = 0; c < 12; c++) Sp[(k * 12 + c) * (uint32_t)P.N + rr] = v[c];
    }
    __syncthreads();
  }
  // 1.0f that the compiler does not know (see project_half)
  R one = (R)1;
  if constexpr (IsHalf<IOI>::value) asm volatile("" : "+v"(one));
  const NbLoader<IOI, LDSS> ld{in, Sp, (uint32_t)P.N, r, s0, S, one};
  if (active) {
    const uint32_t i = q.v * (uint32_t)P.N + r;
    C acc[12];
#pragma unroll
    for (int c = 0; c < 12; c++) acc[c] = mk<R>(0, 0);
    // t first: its neighbours are the farthest apart, and this order hits L2
    // most often (9.4 M KiB fetched against 12.4 M with t last, 12 rhs FP64)
    if constexpr (PIPE) {
#define CVC_HOP(H) hop_pipelined<IOI, RECON, H, EO>(acc, raw, in, own_f, one, Ul, P, q, r, sl)
      CVC_HOP(0); CVC_HOP(1); CVC_HOP(2); CVC_HOP(3); CVC_HOP(4); CVC_HOP(5); CVC_HOP(6); CVC_HOP(7);
#undef CVC_HOP
    } else {
#define CVC_HOP(H) hop_plain<IOI, RECON, H, LDSL, LDSS, EO, FEW>(acc, ld, U, Ul, P, q, sl)
      CVC_HOP(0); CVC_HOP(1); CVC_HOP(2); CVC_HOP(3); CVC_HOP(4); CVC_HOP(5); CVC_HOP(6); CVC_HOP(7);
#undef CVC_HOP
    }

    // the shadow residual of the <r2, out> epilogue is read once per launch:
    // streaming loads, issued beside the own spinor's (the latencies overlap)
    C w2[12];
    if constexpr (dot_shadow(DM)) r2.load_nt(w2, i);
    C own[12];
    if constexpr (!EO) {
      if constexpr (PIPE) raw.full(own);
      else ld.full(own, q.v, true);
      const R mh = (R)-0.5;
#pragma unroll
      for (int c = 0; c < 12; c++) {
        // -1/2 hop + phi/(2 kappa) + i mutm gamma5 phi  (gamma5 = +1 on spins 0,1, -1 on 2,3)
        const R m = c < 6 ? P.mutm : -P.mutm;
        C o;
        o.x = fmar(mh, acc[c].x, fmar(P.k2, own[c].x, -(m * own[c].y)));
        o.y = fmar(mh, acc[c].y, fmar(P.k2, own[c].y, m * own[c].x));
        if (G5OUT && c >= 6) { o.x = -o.x; o.y = -o.y; }
        acc[c] = o;
      }
    } else {
      if (P.dmode != 1) {
        if constexpr (PIPE) raw.full(own);
        else own_f.load(own, i);
      }
#pragma unroll
      for (int c = 0; c < 12; c++) {
        const R m = c < 6 ? P.mutm : -P.mutm;
        C o;
        if (P.dmode == 0) {
          o.x = fmar(P.hopc, acc[c].x, fmar(P.k2, own[c].x, -(m * own[c].y)));
          o.y = fmar(P.hopc, acc[c].y, fmar(P.k2, own[c].y, m * own[c].x));
        } else {
          C h = mk<R>(P.hopc * acc[c].x, P.hopc * acc[c].y);
          if (P.dmode >= 2) h = mk<R>(fmar(P.hopc, acc[c].x, own[c].x), fmar(P.hopc, acc[c].y, own[c].y));
          if (P.dmode == 2) {
            o = h;
          } else {
            // A^-1 h = (1/(2 kappa) - i mutm gamma5) h / ((1/(2 kappa))^2 + mutm^2)
            o.x = fmar(P.k2, h.x, m * h.y) * P.dinv;
            o.y = fmar(P.k2, h.y, -(m * h.x)) * P.dinv;
          }
        }
        if (G5OUT && c >= 6) { o.x = -o.x; o.y = -o.y; }
        acc[c] = o;
      }
    }
    if (P.nt) out.store_nt(acc, i);
    else out.store(acc, i);
    add_dots<DM>(dv, acc, own, w2);
  }
  if constexpr (DM != DOT_NONE) block_reduce_store<dot_rows(DM)>(dv, part, P.N);
}

// ------------------------------------------------------- t-marching operator
//
// Multi-rhs operator on the whole lattice in which each workgroup owns S
// columns (sites of one (x, y, z) cross-section, all N rhs) and walks them
// through M consecutive time slices.  The backward t hop of slice t+1,
// (1 + gamma_0) U_0(t)^dagger phi(t), is formed from the own spinor phi(t)
// while slice t is processed and carried to the next step in registers as the
// six complex numbers it depends on, so the t neighbours are not read again
// from memory: per step a thread reads phi(t) (its own, which the same thread
// read one step before as the forward neighbour, so it comes from L2), the six
// spatial neighbours and phi(t+1).  Columns are grouped in patches of
// XP x YP x LZ sites; XCD j takes the patches p = j mod 8, and the workgroups
// of one XCD run the chunks of one patch over one range of M slices side by
// side, so the spatial neighbours of a chunk are read by neighbouring
// workgroups of the same XCD at about the same step.  The links of a step
// (U_0(t), U_k(t), U_k(t - k) for k = x, y, z) are staged in LDS once per
// workgroup and shared by the N rhs lanes of a column.
//
// Accumulation: acc starts at -2 (1/(2 kappa) + i mutm gamma5) phi(t), the
// eight hops are added, and the output is -acc/2 (the factors -2 and -1/2 are
// exact), i.e. phi/(2 kappa) + i mutm gamma5 phi - hop/2 as in Q_phi.c:58-174
// with a different rounding order.

// w_a = link row . h_a for the three rows (w[a][i]), the boundary phase
// applied (PHASE) as in link_apply; expand_w adds the hop's four spin rows.
template <typename R, int RECON, bool FWD, bool PHASE>
__device__ __forceinline__ void link_mul(cplx<R> w[2][3], const cplx<R> h[2][3], const cplx<R> *__restrict__ base,
                                         uint32_t stride, cplx<R> ph) {
  using C = cplx<R>;
  C u[9];
  if constexpr (RECON == 12) {
#pragma unroll
    for (int k = 0; k < 6; k++) u[k] = base[(size_t)k * stride];
    rebuild_row3(u);
  }
#pragma unroll
  for (int i = 0; i < 3; i++) {
    C w0 = mk<R>(0, 0), w1 = mk<R>(0, 0);
#pragma unroll
    for (int j = 0; j < 3; j++) {
      const int k = FWD ? 3 * i + j : 3 * j + i;
      const C e = RECON == 18 ? base[(size_t)k * stride] : u[k];
      if constexpr (FWD) {
        w0 = cfma(w0, e, h[0][j]);
        w1 = cfma(w1, e, h[1][j]);
      } else {
        w0 = cfmac(w0, e, h[0][j]);
        w1 = cfmac(w1, e, h[1][j]);
      }
    }
    if constexpr (!PHASE) {
    } else if constexpr (FWD) {
      w0 = cmul(ph, w0);
      w1 = cmul(ph, w1);
    } else {
      w0 = cmulc(ph, w0);
      w1 = cmulc(ph, w1);
    }
    w[0][i] = w0;
    w[1][i] = w1;
  }
}

// the scale of an FP16 spinor, on its link product
template <typename IO, typename C, typename R>
__device__ __forceinline__ void scale_w(C w[2][3], R n) {
  if constexpr (IsHalf<IO>::value) {
#pragma unroll
    for (int i = 0; i < 3; i++) {
      w[0][i] = cscale(w[0][i], n);
      w[1][i] = cscale(w[1][i], n);
    }
  }
}

template <typename C, int MU, bool FWD>
__device__ __forceinline__ void expand_w(C acc[12], const C w[2][3]) {
  constexpr int q2 = GCOL[MU][2], q3 = GCOL[MU][3];
  constexpr int l2 = FWD ? uneg(GVAL[MU][2]) : GVAL[MU][2];
  constexpr int l3 = FWD ? uneg(GVAL[MU][3]) : GVAL[MU][3];
#pragma unroll
  for (int i = 0; i < 3; i++) {
    acc[i] = cadd(acc[i], w[0][i]);
    acc[3 + i] = cadd(acc[3 + i], w[1][i]);
    acc[6 + i] = cadd(acc[6 + i], cunit<l2>(q2 == 0 ? w[0][i] : w[1][i]));
    acc[9 + i] = cadd(acc[9 + i], cunit<l3>(q3 == 0 ? w[0][i] : w[1][i]));
  }
}

// the links of one step, staged per column: slot 0 U_0(t), slots 1-3 U_k(t),
// slots 4-6 U_k(t - k)
constexpr int kMarchSlots = 7;

#ifndef CVC_MARCH_WAVES64
#define CVC_MARCH_WAVES64 3
#endif
#ifndef CVC_MARCH_WAVES32
#define CVC_MARCH_WAVES32 4
#endif
template <typename R> struct MarchWaves {
  static constexpr int value = sizeof(R) == 8 ? CVC_MARCH_WAVES64 : CVC_MARCH_WAVES32;
};

template <typename IOI, typename IOO, int RECON, bool G5OUT, int DM, typename IOR = IOI>
__global__ void __launch_bounds__(256, MarchWaves<typename IOI::real>::value)
k_dslash_march(IOO out, IOI in, const cplx<typename IOI::real> *__restrict__ U, DParams<typename IOI::real> P,
               IOR r2, double *__restrict__ part) {
  using R = typename IOI::real;
  using C = cplx<R>;
  constexpr int KL = RECON == 18 ? 9 : 6;
  // FP32 with 2-row links: staged whole with the phase applied (as in k_dslash)
  constexpr bool FOLD = RECON == 12 && sizeof(R) == 4;
  constexpr int KS = FOLD ? 9 : KL;
  constexpr int RL = FOLD ? 18 : RECON;
  const uint32_t S = P.mS;
  // workgroup -> (patch, range of slices, chunk of the patch's columns)
  uint32_t k = blockIdx.x, xcd = 0;
  if (P.mXcd) {
    xcd = blockIdx.x % kXcds;
    k = blockIdx.x / kXcds;
  }
  const uint32_t ch = k % P.mCP, q = k / P.mCP;
  const uint32_t rng = q % P.mNR, pl = q / P.mNR;
  const uint32_t patch = P.mXcd ? pl * kXcds + xcd : pl;
  const uint32_t px = patch % P.mNPX, py = patch / P.mNPX;
  const uint32_t r = threadIdx.x % (uint32_t)P.N, cl = threadIdx.x / (uint32_t)P.N;
  // column cl of the chunk: z fastest, then y, then x inside the patch
  auto column = [&](uint32_t c, uint32_t &sxyz) -> bool {
    const uint32_t j = ch * S + c;
    if (c >= S || j >= P.mXP * P.mYP * (uint32_t)P.LZ) return false;
    const uint32_t z = j % (uint32_t)P.LZ, j2 = j / (uint32_t)P.LZ;
    const uint32_t y = py * P.mYP + j2 % P.mYP, x = px * P.mXP + j2 / P.mYP;
    sxyz = (x * (uint32_t)P.LY + y) * (uint32_t)P.LZ + z;
    return true;
  };
  uint32_t sxyz = 0;
  const bool active = column(cl, sxyz) && !(P.done && P.done[(size_t)r * P.dstride]);
  uint32_t cx = 0, cy = 0, cz = 0;
  if (active) {
    cz = sxyz % (uint32_t)P.LZ;
    cy = (sxyz / (uint32_t)P.LZ) % (uint32_t)P.LY;
    cx = sxyz / P.sX;
  }
  const uint32_t t0 = rng * P.mM;
  extern __shared__ unsigned char dyn_lds[];
  C *Ul = reinterpret_cast<C *>(dyn_lds);   // [kMarchSlots][KS][S]
  R one = (R)1;   // opaque to the compiler (see project_half)
  if constexpr (IsHalf<IOI>::value) asm volatile("" : "+v"(one));
  const NbLoader<IOI, false> ld{in, nullptr, (uint32_t)P.N, r, 0, 0, one};
  double dv[dot_rows(DM) > 0 ? dot_rows(DM) : 1] = {};

  // carry: (U_0^dagger (1 + gamma_0) phi)(t - 1) as the six complex numbers w
  C carry[2][3];
  if (active) {
    const uint32_t tm = t0 == 0 ? (uint32_t)P.T - 1 : t0 - 1;
    const uint32_t sm = tm * P.sT + sxyz;
    C h[2][3];
    const R n = ld.template proj<0, false>(h, sm, false);
    link_mul<R, RECON, false, true>(carry, h, U + sm, P.V, P.ph[0]);
    scale_w<IOI>(carry, n);
  }

  for (uint32_t step = 0; step < P.mM; step++) {
    const uint32_t t = t0 + step;
    __syncthreads();   // the previous step's links are no longer read
    for (uint32_t e = threadIdx.x; e < (uint32_t)kMarchSlots * S; e += blockDim.x) {
      const uint32_t slot = e / S, c = e - slot * S;
      uint32_t cs;
      if (!column(c, cs)) continue;
      const int mu = slot < 4 ? (int)slot : (int)slot - 3;
      uint32_t ls = t * P.sT + cs;
      if (slot >= 4) {   // U_k(t - k)
        const uint32_t str = mu == 1 ? P.sX : mu == 2 ? (uint32_t)P.LZ : 1u;
        const uint32_t L = (uint32_t)(mu == 1 ? P.LX : mu == 2 ? P.LY : P.LZ);
        const uint32_t crd = (cs / str) % L;
        ls = crd == 0 ? ls + (L - 1) * str : ls - str;
      }
      if constexpr (FOLD) {
        C u[9];
#pragma unroll
        for (int kk = 0; kk < 6; kk++) u[kk] = U[((size_t)mu * 6 + kk) * P.V + ls];
        rebuild_row3(u);
#pragma unroll
        for (int kk = 0; kk < 9; kk++) Ul[(slot * 9 + kk) * S + c] = cmul(u[kk], P.ph[mu]);
      } else {
#pragma unroll
        for (int kk = 0; kk < KL; kk++) Ul[(slot * KL + kk) * S + c] = U[((size_t)mu * KL + kk) * P.V + ls];
      }
    }
    __syncthreads();
    if (!active) continue;
    const uint32_t s = t * P.sT + sxyz;
    const uint32_t i = s * (uint32_t)P.N + r;
    // the shadow residual of the <r2, out> epilogue is read once per launch:
    // streaming loads, issued with the own spinor's
    C w2[12];
    if constexpr (dot_shadow(DM)) r2.load_nt(w2, i);
    C acc[12];
    {
      C own[12];
      ld.full(own, s, false);
      // acc = -2 (1/(2 kappa) + i mutm gamma5) phi   (gamma5 = +1 on spins 0,1, -1 on 2,3)
#pragma unroll
      for (int c = 0; c < 12; c++) {
        const R m = c < 6 ? P.mutm : -P.mutm;
        acc[c].x = (R)-2 * fmar(P.k2, own[c].x, -(m * own[c].y));
        acc[c].y = (R)-2 * fmar(P.k2, own[c].y, m * own[c].x);
      }
      // backward t hop from the carry, then the carry for slice t+1 from phi(t)
      expand_w<C, 0, false>(acc, carry);
      C h[2][3];
      project<0, false>(h, [&](int c) { return own[c]; });
      link_mul<R, RL, false, !FOLD>(carry, h, Ul + cl, S, P.ph[0]);
    }
    pin_regs(acc, 12);
    pin_regs(&carry[0][0], 6);
    // spatial hops
#define CVC_MHOP(MU, CRD, L, STR)                                                                              \
    {                                                                                                          \
      const uint32_t sm_ = (CRD) == 0 ? s + (uint32_t)((L) - 1) * (STR) : s - (STR);                          \
      const uint32_t sp_ = (CRD) == (uint32_t)(L) - 1 ? s - (uint32_t)((L) - 1) * (STR) : s + (STR);           \
      C h[2][3], w[2][3];                                                                                      \
      R n = ld.template proj<MU, false>(h, sm_, false);                                                        \
      pin_regs(&h[0][0], 6);                                                                                   \
      link_mul<R, RL, false, !FOLD>(w, h, Ul + (3 + MU) * KS * S + cl, S, P.ph[MU]);                           \
      scale_w<IOI>(w, n);                                                                                      \
      expand_w<C, MU, false>(acc, w);                                                                          \
      pin_regs(acc, 12);                                                                                       \
      n = ld.template proj<MU, true>(h, sp_, false);                                                           \
      pin_regs(&h[0][0], 6);                                                                                   \
      link_mul<R, RL, true, !FOLD>(w, h, Ul + (MU)*KS * S + cl, S, P.ph[MU]);                                  \
      scale_w<IOI>(w, n);                                                                                      \
      expand_w<C, MU, true>(acc, w);                                                                           \
      pin_regs(acc, 12);                                                                                       \
    }
    CVC_MHOP(1, cx, P.LX, P.sX);
    CVC_MHOP(2, cy, P.LY, (uint32_t)P.LZ);
    CVC_MHOP(3, cz, P.LZ, 1u);
#undef CVC_MHOP
    // forward t hop: (1 - gamma_0) U_0(t) phi(t+1), last, so that phi(t+1) is
    // still in L2 when the next step reads it as its own spinor
    {
      const uint32_t sp = t == (uint32_t)P.T - 1 ? sxyz : s + P.sT;
      C h[2][3], w[2][3];
      const R n = ld.template proj<0, true>(h, sp, false);
      pin_regs(&h[0][0], 6);
      link_mul<R, RL, true, !FOLD>(w, h, Ul + cl, S, P.ph[0]);
      scale_w<IOI>(w, n);
      expand_w<C, 0, true>(acc, w);
    }
    const R mh = (R)-0.5;
#pragma unroll
    for (int c = 0; c < 12; c++) {
      acc[c].x *= mh;
      acc[c].y *= mh;
      if (G5OUT && c >= 6) { acc[c].x = -acc[c].x; acc[c].y = -acc[c].y; }
    }
    if (P.nt) out.store_nt(acc, i);
    else out.store(acc, i);
    C own[12];
    if constexpr (DM == DOT_TS || DM == DOT_TSR) in.load(own, i);
    add_dots<DM>(dv, acc, own, w2);
  }
  if constexpr (DM != DOT_NONE) block_reduce_store<dot_rows(DM)>(dv, part, P.N);
}

// ------------------------------------------------------------- launcher

static int log2_exact(uint32_t v) {   // -1 unless v is a power of two
  if (v == 0 || (v & (v - 1))) return -1;
  int l = 0;
  while ((1u << l) < v) l++;
  return l;
}

template <typename R>
static DParams<R> make_params(const cvchip_ctx *c, int N, double mutm) {
  DParams<R> P;
  P.V = (uint32_t)c->lat.V;
  P.N = N;
  P.VN = (uint32_t)(c->lat.V * N);
  P.T = c->lat.T;
  P.LX = c->lat.LX;
  P.LY = c->lat.LY;
  P.LZ = c->lat.LZ;
  P.sX = (uint32_t)(c->lat.LY * c->lat.LZ);
  P.sT = (uint32_t)(c->lat.LX * c->lat.LY * c->lat.LZ);
  P.invN = 1.0f / (float)N;
  P.invS = 0.f;
  P.k2 = (R)(0.5 / c->kappa);
  P.mutm = (R)mutm;
  for (int m = 0; m < 4; m++) P.ph[m] = mk<R>((R)c->ph.re[m], (R)c->ph.im[m]);
  return P;
}

template <typename IO> static IO make_io(const Field &f);
template <> IOPlain<double> make_io<IOPlain<double>>(const Field &f) {
  return IOPlain<double>{(double2 *)f.data, (uint32_t)(f.V * f.nrhs)};
}
template <> IOPlain<float> make_io<IOPlain<float>>(const Field &f) {
  return IOPlain<float>{(float2 *)f.data, (uint32_t)(f.V * f.nrhs)};
}
template <> IOHalf make_io<IOHalf>(const Field &f) {
  return IOHalf{(__half2 *)f.data, f.norm, (uint32_t)(f.V * f.nrhs)};
}

// t-march geometry (mode 6) for N rhs on the whole lattice L; bits 8-15 of the
// policy give the march length M (0: 16; the largest divisor of T not above
// it is used), bits 16-19 and 20-23 the patch's x and y extents (0: 8; a
// value that does not divide LX or LY falls back to 1).
static bool march_geometry(const cvchip_ctx *c, int N, Traversal &t, bool explicit_policy, uint32_t M_auto) {
  const Lattice &L = c->lat;
  if (N < 1 || N > 192) return false;
  uint32_t S = 192u / (uint32_t)N;
  if (S > 48) S = 48;
  const int pol = explicit_policy ? c->dslash_policy : 0;
  uint32_t M = (uint32_t)((pol >> 8) & 255);
  if (M == 0) M = explicit_policy ? 16 : M_auto;
  while (M > 1 && L.T % (int)M) M--;
  uint32_t XP = (uint32_t)((pol >> 16) & 15), YP = (uint32_t)((pol >> 20) & 15);
  if (XP == 0) XP = 8;
  if (YP == 0) YP = 8;
  if (L.LX % (int)XP) XP = 1;
  if (L.LY % (int)YP) YP = 1;
  t.mode = 6;
  t.mS = S;
  t.mM = M;
  t.mXP = XP;
  t.mYP = YP;
  t.mNPX = (uint32_t)L.LX / XP;
  const uint32_t npatch = t.mNPX * ((uint32_t)L.LY / YP);
  t.mCP = (XP * YP * (uint32_t)L.LZ + S - 1) / S;
  t.mNR = (uint32_t)L.T / M;
  t.mXcd = npatch % kXcds == 0 ? 1 : 0;
  t.nblk = npatch * t.mNR * t.mCP;
  t.threads = S * (uint32_t)N;
  return true;
}


// Sites per operator block for runs of len of a lattice's V sites: at most
// launch_block's, the count that costs the run least, in lanes: the padded sites', a
// quarter of those that idle in a block's last wave, half a site for each block
// (its prologue), and a thirty-second where S N is not a multiple of 8, so that
// a block's stores do not begin and end on 128-byte lines (a line shared by two blocks
// is written twice, in halves).  36 rhs, FP16: 7 sites (252 lanes) 201 us at 32x16^3,
// 3115 us at 64x32^3; 4 sites (144 lanes), the choice without the idle lanes, 220-230
// and 3400-3500 us.  Twenty counts from 8 to 96 on eight lattices, geometric mean of
// the former over the present time: FP64 1.012, FP32 1.008, FP16 1.020.
static uint32_t op_sites(int N, uint32_t len, int64_t V) {
  const uint32_t S0 = (uint32_t)(launch_block(V, N) / N);
  if (N < 8) return S0;   // links from memory: blocks of 256 threads win although their last one is padded more
  auto cost = [&](uint32_t S) {   // in 1/16 lanes
    const uint64_t nb = (len + S - 1) / S, used = S * (uint64_t)N, lanes = (used + 63) / 64 * 64;
    return nb * (12 * used + 4 * lanes + 8 * N) + (used % 8 ? nb * used / 2 + 16 * N : 0);
  };
  uint32_t best = S0;
  for (uint32_t S = S0; S > 0 && 2 * S >= S0; S--)
    if (cost(S) < cost(best)) best = S;
  return best;
}

// The columns of the automatic traversal (mode 4): bx planes x yb rows of the
// lattice L (its half for the even/odd operator) for N rhs.  A step in t should still find the last
// slice's cross-section in the XCD's 4 MB L2 beside what streams through (the
// outputs, the links, the neighbours of the columns' sides), so of the divisors
// of LX and LY those are taken that read the fewest sides again (weight hw per
// unit of 2/bx + 2/yb) while the cross-section's spinors stay below `budget`
// bytes, corrected for padded blocks and for XCDs that get a pair less; a plane of
// the column above it reads the x neighbours inside the column again too (whole
// slices, without that term, at 48 FP64 rhs: 64x32^3 20.8 ms against 16.0 ms for
// the 2 x 2 columns).  Sweep
// of 0.6-9 MB and hw 0.1-0.7 over 24 operators (FP64, FP64 / FP32 / FP16
// even/odd on six lattices): geometric mean 1.5 % above the best of each at
// 1.5 MB and 0.3, 4-6 % at 1.2 and 2.4 MB.  1.8 MB against 1.5 MB, FP64: whole lattice, 48
// rhs 64x32^3 14.7 / 16.5 ms (2 x 4 columns), 24 rhs 7.06 / 7.27 ms, 24 rhs 40x20^3 1.02 /
// 1.09 ms, but even/odd, 12 rhs 40x20^3, 285 / 265 us.
// bx and yb that the policy gives (not 0) stay; only the other is chosen.
static void best_columns(const Lattice &L, int N, int K, bool eo, uint32_t &bx, uint32_t &yb) {
  const double site = 12. * 16 / K * N;   // bytes of a site's spinors
  const double budget = eo ? 1.5e6 : 1.8e6, hw = 0.3;   // even/odd forms stream own spinors too
  double best = 0.;
  const uint32_t bx0 = bx, yb0 = yb;
  for (int cx = 1; cx <= L.LX; cx++) {
    if (L.LX % cx || (bx0 && (uint32_t)cx != bx0)) continue;
    for (int cy = 1; cy <= L.LY; cy++) {
      if (L.LY % cy || (yb0 && (uint32_t)cy != yb0)) continue;
      const uint32_t len = (uint32_t)(cy * L.LZ), S = op_sites(N, len, L.V);
      const double pad = (double)((len + S - 1) / S * S) / len;
      const double npair = (double)(L.LX / cx) * (L.LY / cy) * L.T, npx = ceil(npair / kXcds);
      const double halo = (cx < L.LX ? 2. / cx : 0.) + (cy < L.LY ? 2. / cy : 0.);
      auto missed = [&](double bytes) { return bytes > budget ? 2. * (1. - budget / bytes) : 0.; };
      const double again = halo + missed(site * cx * len) + (1. - 1. / cx) * missed(site * len);
      const double cost = (1. + hw * again) * pad * (npx * kXcds / npair);
      if (best == 0. || cost < best) {
        best = cost;
        bx = (uint32_t)cx;
        yb = (uint32_t)cy;
      }
    }
  }
}

// Block-to-site mapping; the policy's bits 4-7 pick the mode (0: automatic),
// bits 8-15 the y-block height of modes 2, 4 and 5 and of the automatic columns (0:
// automatic), bits 20-23 the x extent of mode 4's and the automatic columns (0: 4 or
// 1 in mode 4; its t extent in bits 16-19 does not change the order); for mode 5, bits 16-19 are log2 of the column's z extent
// (0: 8) and bits 20-23 its x extent (0: 4).
// Automatic: N >= 8 the columns of best_columns; below, XCD chunks of a slice: over 1,
// 2, 4 and 7 rhs in each precision on six lattices (16^4 to 64x32^3) the best columns
// of each case take 0.97 to 1.04 times as long in the geometric mean (0.81 to 1.15).
// K: complexes per 16 bytes of the operator's spinors (1 FP64, 2 FP32, 4
// FP16+norm).  The FP32 operator of 8 to 20 rhs on the whole lattice marches in t
// (mode 6, marches of 4 slices) where the 8 x 8 patches of a cross-section divide
// among the XCDs and a set is 256 MB or more: 12 rhs 32^4 845 against 940 us for the
// columns, 64x32^3 1.68 against 1.87 ms, 32x32x16^2 (302 MB) 211 against 219 us; over
// 8, 10, 12, 13, 16, 18 and 20 rhs on such lattices the columns take 1.03 times as
// long (0.90 to 1.14).  Below 256 MB the columns win (16x32x16^2, 12 rhs, 151 MB: 80
// against 90 us), and where the XCDs share patches unevenly (40x20^3, 12 rhs, 261
// against 431 us; 20x40^3, 25 patches, 12 rhs, 1.47 GB, 1.14 against 1.63 ms; 48x24^3, 9
// patches, 0.58 against 0.85 ms).
static Traversal plan_traversal(const cvchip_ctx *c, int N, bool eo, int K) {
  Lattice L = c->lat;
  if (eo) {   // the half lattice of one parity: LZ/2 half-sites per z line
    L.LZ /= 2;
    L.V /= 2;
  }
  const uint32_t V = (uint32_t)L.V, slice = (uint32_t)(L.LX * L.LY * L.LZ);
  int want = (c->dslash_policy >> 4) & 15;
  if (want == 6) {
    Traversal t{};
    if (!eo && march_geometry(c, N, t, true, 16)) return t;
    want = 4;   // the even/odd operator does not march
  }
  if (want == 0 && K == 2 && !eo && N >= 8 && N <= 20 && (uint64_t)V * N * 96 >= ((uint64_t)1 << 28) &&
      L.LX % 8 == 0 && L.LY % 8 == 0 && L.LX / 8 * (L.LY / 8) % (int)kXcds == 0) {
    Traversal t{};
    if (march_geometry(c, N, t, false, 4)) return t;
  }
  uint32_t yb = (uint32_t)((c->dslash_policy >> 8) & 255);
  uint32_t bx = (uint32_t)((c->dslash_policy >> 20) & 15);
  if (want == 0 && N >= 8) {
    best_columns(L, N, K, eo, bx, yb);
    want = 4;
  }
  if (want == 0) want = 1;
  if (yb == 0) {
    yb = 1;
    for (uint32_t y : {16u, 8u, 4u, 2u})
      if (L.LY % (int)y == 0) { yb = y; break; }
  }
  if (bx == 0) bx = L.LX % 4 == 0 ? 4 : 1;
  Traversal t{};
  uint32_t S = 1;
  // blocks of S sites over runs of len sites
  auto runs = [&](uint32_t len) {
    S = op_sites(N, len, L.V);
    t.threads = S * (unsigned)N;
    return (len + S - 1) / S;
  };
  if (want == 5) {
    const uint32_t cyb = (c->dslash_policy >> 8) & 255 ? yb : 4u;
    const uint32_t lz = (c->dslash_policy >> 16) & 15;
    const uint32_t czb = lz ? (1u << lz) : 8u;
    const uint32_t cbx = (c->dslash_policy >> 20) & 15 ? bx : 4u;
    const int l1 = log2_exact(cbx), l2 = log2_exact(cyb), l3 = log2_exact(czb);
    if (l1 >= 0 && l2 >= 0 && l3 >= 0 && L.LX % (int)cbx == 0 && L.LY % (int)cyb == 0 && L.LZ % (int)czb == 0) {
      const uint32_t ncol = (uint32_t)(L.LX / (int)cbx) * (uint32_t)(L.LY / (int)cyb) * (uint32_t)(L.LZ / (int)czb);
      if (ncol % kXcds == 0) {
        t.mode = 5;
        t.bx = cbx;
        t.yb = cyb;
        t.zb = czb;
        t.ncy = (uint32_t)L.LY / cyb;
        t.ncz = (uint32_t)L.LZ / czb;
        t.lzb = (uint32_t)l3;
        t.lyz = (uint32_t)(l2 + l3);
        t.lA = (uint32_t)(l1 + l2 + l3);
        t.colsz = (uint32_t)L.T << t.lA;
        t.bpcol = runs(t.colsz);
        t.nblk = ncol * t.bpcol;
        return t;
      }
    }
    want = 4;   // a column request that does not tile the lattice falls back to mode 4
  }
  if (want == 4 && L.LX % (int)bx == 0 && L.LY % (int)yb == 0) {
    t.mode = 4;
    t.yb = yb;
    t.bx = bx;
    t.ncx = (uint32_t)L.LX / bx;
    t.runlen = yb * (uint32_t)L.LZ;
    t.bpr = runs(t.runlen);
    t.bpp = bx * t.bpr;
    t.npair = t.ncx * ((uint32_t)L.LY / yb) * (uint32_t)L.T;
    t.npx = (t.npair + kXcds - 1) / kXcds;
    t.nblk = kXcds * t.npx * t.bpp;
    return t;
  }
  // (a mode 4 request that does not tile the lattice falls back to mode 2)
  if ((want == 2 || want == 4) && L.T % (int)kXcds == 0 && L.LY % (int)yb == 0) {
    t.mode = 2;
    t.yb = yb;
    t.runlen = yb * (uint32_t)L.LZ;
    t.bpr = runs(t.runlen);
    t.nrun = (uint32_t)(L.LY / (int)yb) * (uint32_t)L.LX;
    t.nblk = (uint32_t)L.T * t.nrun * t.bpr;
    return t;
  }
  if (slice % kXcds == 0) { t.csz = slice / kXcds; t.mode = 1; }
  else if (V % kXcds == 0) { t.csz = V / kXcds; t.mode = 1; }
  else { t.csz = V; t.mode = 0; }
  if (want == 3) t.mode = 0;
  t.bpc = runs(t.csz);
  t.nblk = (V / t.csz) * t.bpc;
  return t;
}

// planned once per context, policy, rhs count and precision (a launch on a small
// lattice is shorter than the plan)
static const Traversal &traversal(const cvchip_ctx *c, int N, bool eo, int K) {
  const uint64_t key = ((uint64_t)c->dslash_policy << 16) | ((uint64_t)N << 4) | ((uint64_t)eo << 3) | (uint64_t)K;
  const auto it = c->plans.find(key);
  if (it != c->plans.end()) return it->second;
  return c->plans.emplace(key, plan_traversal(c, N, eo, K)).first->second;
}

template <typename R>
static void set_traversal(DParams<R> &P, const Traversal &tr, uint32_t LZt) {
  P.LZt = LZt;
  P.invS = 1.0f / (float)(tr.threads / (unsigned)P.N);   // sites per block
  P.csz = tr.csz;
  P.bpc = tr.bpc;
  P.mode = tr.mode;
  P.yb = tr.yb;
  P.runlen = tr.runlen;
  P.bpr = tr.bpr;
  P.nrun = tr.nrun;
  P.bx = tr.bx;
  P.ncx = tr.ncx;
  P.bpp = tr.bpp;
  P.npx = tr.npx;
  P.npair = tr.npair;
  P.bpcol = tr.bpcol;
  P.zb = tr.zb;
  P.ncy = tr.ncy;
  P.ncz = tr.ncz;
  P.lzb = tr.lzb;
  P.lyz = tr.lyz;
  P.lA = tr.lA;
  P.colsz = tr.colsz;
  P.sXt = (uint32_t)P.LY * LZt;
  P.sTt = (uint32_t)P.LX * P.sXt;
  P.mS = tr.mS;
  P.mM = tr.mM;
  P.mXP = tr.mXP;
  P.mYP = tr.mYP;
  P.mCP = tr.mCP;
  P.mNR = tr.mNR;
  P.mNPX = tr.mNPX;
  P.mXcd = tr.mXcd;
  auto div = [](uint32_t d) { return make_fdiv(d ? d : 1); };   // 0: a quotient of another mode
  P.fLZt = div(LZt);
  P.fLY = div((uint32_t)P.LY);
  P.fLX = div((uint32_t)P.LX);
  P.fbpc = div(tr.bpc);
  P.fbpcol = div(tr.bpcol);
  P.fT = div((uint32_t)P.T);
  P.fbpp = div(tr.bpp);
  P.fbpr = div(tr.bpr);
  P.fncx = div(tr.ncx);
  P.fslice = div(tr.nrun * tr.bpr);
  P.fncy = div(tr.ncy);
  P.fncz = div(tr.ncz);
}

unsigned dslash_blocks(const cvchip_ctx *c, int N) {
  unsigned m = 0;
  for (int K : {1, 2, 4}) {
    m = std::max(m, traversal(c, N, false, K).nblk);
    if (c->lat.LZ % 2 == 0) m = std::max(m, traversal(c, N, true, K).nblk);
  }
  return m;
}

struct EOArgs {
  const Field *own;
  int par, dmode;
  double hopc;
};

// IOR differs from IOI only for the <r2, out> epilogue (DOT_R2) with an FP16 r2
template <typename IOI, typename IOO, int RECON, bool EO, typename IOR = IOI>
static int launch(cvchip_ctx *c, Field &out, const Field &in, double mutm, int g5, DotMode dm,
                  const Field *r2, int *nblk_out, const EOArgs *eo = nullptr) {
  constexpr bool kSameR = std::is_same<IOR, IOI>::value;
  constexpr bool k64 = sizeof(typename IOI::real) == 8;
  if (!kSameR && (dm != DOT_R2 || !r2)) {
    set_error("operator: a shadow residual of another precision serves only the <r2, out> epilogue");
    return CVCHIP_ERR_ARG;
  }
  if ((dot_shadow(dm) && !r2) || (g5 ? dm == DOT_TS || dm == DOT_TSR : dm == DOT_NN || dm == DOT_NNR) ||
      (!k64 && (dm == DOT_TSR || dm == DOT_NNR))) {
    set_error("operator: no such fused dot products (%d)", (int)dm);
    return CVCHIP_ERR_ARG;
  }
  using R = typename IOI::real;
  const int N = in.nrhs;
  DParams<R> P = make_params<R>(c, N, mutm);
  P.par = eo ? eo->par : 0;
  P.dmode = eo ? eo->dmode : 0;
  P.hopc = (R)(eo ? eo->hopc : -0.5);
  P.dinv = (R)(1.0 / (0.25 / (c->kappa * c->kappa) + mutm * mutm));
  const Traversal &tr = traversal(c, N, EO, IOI::K);
  set_traversal(P, tr, EO ? (uint32_t)c->lat.LZ / 2 : (uint32_t)c->lat.LZ);
  const int B = (int)tr.threads;
  P.done = c->op_mask;
  P.dstride = c->op_mask_stride;
  // Streaming stores only for outputs that would not stay in the 256 MB MALL
  // beside the other fields (bit 3: for every output), and streaming loads for
  // own spinors, which the even/odd forms read once, that do not stay in the caches
  // anyway: both leave the L2 to the neighbours.  Per iteration (FP32 28x18x14x20,
  // FP16 40x20^3, FP32 24x14x14x16 with 48 rhs): 908 / 1460 / 1881 us with stores
  // from 256 MB and cached loads, 875 / 1410 / 1775 us with these; stores from 64
  // MB 890 / 1409 / 1780; own loads of 40 MB sets slow the operator by 10 %.
  P.nt = (((c->dslash_policy >> 2) & 1) && out.bytes >= ((size_t)128 << 20)) || ((c->dslash_policy >> 3) & 1);
  P.nt_own = eo && eo->own && eo->own->bytes >= ((size_t)64 << 20);
  const unsigned nblk = tr.nblk;
  double *part = nullptr;
  if (dm != DOT_NONE) {
    CVC_TRY(ensure_red(c, sizeof(double) * (c->red_off + (size_t)nblk * dot_rows(dm) * N + 64 * 256)));
    part = (double *)c->red.ptr + c->red_off;
  }
  const cplx<R> *U;
  if constexpr (sizeof(R) == 8) U = (RECON == 18) ? c->gauge64 : c->gauge64r12;
  else U = c->gauge32r12;
  IOO o = make_io<IOO>(out);
  IOI ii = make_io<IOI>(in);
  IOR rr;
  if constexpr (kSameR) rr = r2 ? make_io<IOI>(*r2) : ii;
  else rr = make_io<IOR>(*r2);
  IOI ow = (eo && eo->own) ? make_io<IOI>(*eo->own) : ii;
  dim3 g(nblk), b(B);
  if (!EO && tr.mode == 6) {
    using CR = cplx<R>;
    constexpr int KSM = (RECON == 12 && sizeof(R) == 4) ? 9 : (RECON == 18 ? 9 : 6);
    // bits 24-27: extra LDS per block in 8 KiB units (caps the blocks per CU)
    const size_t lds = (size_t)kMarchSlots * KSM * tr.mS * sizeof(CR) + (size_t)((c->dslash_policy >> 24) & 15) * 8192;
    dim3 bm(tr.threads);
#define CVC_MLAUNCH(G5, DMV) \
    hipLaunchKernelGGL((k_dslash_march<IOI, IOO, RECON, G5, DMV, IOR>), g, bm, lds, c->stream, o, ii, U, P, rr, part)
    if (g5) {
      if (dm == DOT_R2) CVC_MLAUNCH(true, DOT_R2);
      else if constexpr (kSameR) {
        if (dm == DOT_NONE) CVC_MLAUNCH(true, DOT_NONE);
        else if (dm == DOT_NN) CVC_MLAUNCH(true, DOT_NN);
        else if constexpr (k64) CVC_MLAUNCH(true, DOT_NNR);
      }
    } else {
      if (dm == DOT_R2) CVC_MLAUNCH(false, DOT_R2);
      else if constexpr (kSameR) {
        if (dm == DOT_NONE) CVC_MLAUNCH(false, DOT_NONE);
        else if (dm == DOT_TS) CVC_MLAUNCH(false, DOT_TS);
        else if constexpr (k64) CVC_MLAUNCH(false, DOT_TSR);
      }
    }
#undef CVC_MLAUNCH
    CVC_HIP(hipGetLastError());
    if (nblk_out) *nblk_out = (int)nblk;
    return 0;
  }
  const bool multi = block_for(N) / N <= LDS_SITES;
  const bool ldsl = multi && (c->dslash_policy & 1);
  const bool ldss = !EO && multi && (c->dslash_policy & 2) && tr.mode != 5;
  // bits 24-27: extra LDS per block in 8 KiB units (caps the blocks per CU)
  const size_t pad = (size_t)((c->dslash_policy >> 24) & 15) * 8192;
  const size_t dyn = (ldss ? (size_t)(B / N + 2) * N * 12 * sizeof(cplx<R>) : 0) + pad;
  constexpr bool kFew = IOI::K <= 2;   // kernels of their own for the fewest rhs (see hop_plain)
  const bool few = kFew && N <= (k64 ? 2 : 1);
#define CVC_LAUNCH(G5, DMV)                                                                                     \
  do {                                                                                                          \
    if constexpr (EO) {                                                                                         \
      if (ldsl) hipLaunchKernelGGL((k_dslash<IOI, IOO, RECON, G5, DMV, true, false, true, IOR>), g, b, dyn, c->stream, o, ii, ow, U, P, rr, part); \
      else if (few) hipLaunchKernelGGL((k_dslash<IOI, IOO, RECON, G5, DMV, false, false, true, IOR, kFew>), g, b, dyn, c->stream, o, ii, ow, U, P, rr, part); \
      else hipLaunchKernelGGL((k_dslash<IOI, IOO, RECON, G5, DMV, false, false, true, IOR>), g, b, dyn, c->stream, o, ii, ow, U, P, rr, part); \
    } else {                                                                                                    \
      if (ldsl && ldss) hipLaunchKernelGGL((k_dslash<IOI, IOO, RECON, G5, DMV, true, true, false, IOR>), g, b, dyn, c->stream, o, ii, ii, U, P, rr, part); \
      else if (ldsl) hipLaunchKernelGGL((k_dslash<IOI, IOO, RECON, G5, DMV, true, false, false, IOR>), g, b, dyn, c->stream, o, ii, ii, U, P, rr, part); \
      else if (ldss) hipLaunchKernelGGL((k_dslash<IOI, IOO, RECON, G5, DMV, false, true, false, IOR>), g, b, dyn, c->stream, o, ii, ii, U, P, rr, part); \
      else if (few) hipLaunchKernelGGL((k_dslash<IOI, IOO, RECON, G5, DMV, false, false, false, IOR, kFew>), g, b, dyn, c->stream, o, ii, ii, U, P, rr, part); \
      else hipLaunchKernelGGL((k_dslash<IOI, IOO, RECON, G5, DMV, false, false, false, IOR>), g, b, dyn, c->stream, o, ii, ii, U, P, rr, part); \
    }                                                                                                           \
  } while (0)
  if (g5) {
    if (dm == DOT_R2) CVC_LAUNCH(true, DOT_R2);
    else if constexpr (kSameR) {
      if (dm == DOT_NONE) CVC_LAUNCH(true, DOT_NONE);
      else if (dm == DOT_NN) CVC_LAUNCH(true, DOT_NN);
      else if constexpr (k64) CVC_LAUNCH(true, DOT_NNR);
    }
  } else {
    if (dm == DOT_R2) CVC_LAUNCH(false, DOT_R2);
    else if constexpr (kSameR) {
      if (dm == DOT_NONE) CVC_LAUNCH(false, DOT_NONE);
      else if (dm == DOT_TS) CVC_LAUNCH(false, DOT_TS);
      else if constexpr (k64) CVC_LAUNCH(false, DOT_TSR);
    }
  }
#undef CVC_LAUNCH
  CVC_HIP(hipGetLastError());
  if (nblk_out) *nblk_out = (int)nblk;
  return 0;
}

int dslash(cvchip_ctx *c, Field &out, const Field &in, double mutm, int gamma5_out, DotMode dm,
           const Field *r2, int *nblocks_out) {
  if (!c->gauge_set) {
    set_error("gauge field not set (call cvchip_set_gauge first)");
    return CVCHIP_ERR_STATE;
  }
  // r2 may be FP16 for FP32 fields in the <r2, out> epilogue (the FP32 mixed solver's shadow residual)
  const bool r2_half = r2 && dm == DOT_R2 && in.prec == CVCHIP_PREC_F32 && r2->prec == CVCHIP_PREC_F16;
  if (out.nrhs != in.nrhs || out.V != in.V ||
      (r2 && (r2->nrhs != in.nrhs || r2->V != in.V || (r2->prec != in.prec && !r2_half)))) {
    set_error("operator fields do not match (nrhs %d vs %d)", out.nrhs, in.nrhs);
    return CVCHIP_ERR_ARG;
  }
  if (out.data == in.data) {
    set_error("operator output must not alias its input");
    return CVCHIP_ERR_ARG;
  }
  if (in.prec == CVCHIP_PREC_F64 && out.prec == CVCHIP_PREC_F64) {
    if (c->link_recon == 12)
      return launch<IOPlain<double>, IOPlain<double>, 12, false>(c, out, in, mutm, gamma5_out, dm, r2, nblocks_out);
    return launch<IOPlain<double>, IOPlain<double>, 18, false>(c, out, in, mutm, gamma5_out, dm, r2, nblocks_out);
  }
  if (in.prec == CVCHIP_PREC_F32 && out.prec == CVCHIP_PREC_F32) {
    if (r2_half)
      return launch<IOPlain<float>, IOPlain<float>, 12, false, IOHalf>(c, out, in, mutm, gamma5_out, dm, r2,
                                                                       nblocks_out);
    return launch<IOPlain<float>, IOPlain<float>, 12, false>(c, out, in, mutm, gamma5_out, dm, r2, nblocks_out);
  }
  if (in.prec == CVCHIP_PREC_F16 && out.prec == CVCHIP_PREC_F16)
    return launch<IOHalf, IOHalf, 12, false>(c, out, in, mutm, gamma5_out, dm, r2, nblocks_out);
  set_error("unsupported operator precision pair %d -> %d", in.prec, out.prec);
  return CVCHIP_ERR_ARG;
}

// Even/odd operator pieces on half-lattice fields (V/2 sites, half-site order
// of DParams): out_par = dmode form of (own, hopc x hopping sum of in), in at
// the opposite parity.  With H the hopping sum and A = 1/(2 kappa) + i mutm g5,
// D = A - H/2 splits as D_ee = A, D_eo = -H_eo/2 (Q_phi.c:58-174 restricted to
// one parity of the output).
int dslash_eo(cvchip_ctx *c, Field &out, const Field &in, const Field *own, double mutm, int par, int dmode,
              double hopc, int gamma5_out, DotMode dm, const Field *r2, int *nblocks_out) {
  if (!c->gauge_set) {
    set_error("gauge field not set (call cvchip_set_gauge first)");
    return CVCHIP_ERR_STATE;
  }
  if (c->lat.LZ % 2) {
    set_error("even/odd operator needs an even LZ (got %d)", c->lat.LZ);
    return CVCHIP_ERR_ARG;
  }
  const int64_t Vh = c->lat.V / 2;
  const bool r2_half = r2 && dm == DOT_R2 && in.prec == CVCHIP_PREC_F32 && r2->prec == CVCHIP_PREC_F16;
  if (out.V != Vh || in.V != Vh || out.nrhs != in.nrhs || out.prec != in.prec ||
      (dmode != 1 && (!own || own->V != Vh || own->nrhs != in.nrhs || own->prec != in.prec)) ||
      (r2 && (r2->V != Vh || r2->nrhs != in.nrhs || (r2->prec != in.prec && !r2_half))) || dmode < 0 || dmode > 3 ||
      (par != 0 && par != 1)) {
    set_error("even/odd operator: fields must be half-lattice sets of one size and precision");
    return CVCHIP_ERR_ARG;
  }
  if (out.data == in.data) {
    set_error("operator output must not alias its input");
    return CVCHIP_ERR_ARG;
  }
  const EOArgs eo{own, par, dmode, hopc};
  if (in.prec == CVCHIP_PREC_F64) {
    if (c->link_recon == 12)
      return launch<IOPlain<double>, IOPlain<double>, 12, true>(c, out, in, mutm, gamma5_out, dm, r2, nblocks_out, &eo);
    return launch<IOPlain<double>, IOPlain<double>, 18, true>(c, out, in, mutm, gamma5_out, dm, r2, nblocks_out, &eo);
  }
  if (in.prec == CVCHIP_PREC_F32) {
    if (r2_half)
      return launch<IOPlain<float>, IOPlain<float>, 12, true, IOHalf>(c, out, in, mutm, gamma5_out, dm, r2,
                                                                      nblocks_out, &eo);
    return launch<IOPlain<float>, IOPlain<float>, 12, true>(c, out, in, mutm, gamma5_out, dm, r2, nblocks_out, &eo);
  }
  return launch<IOHalf, IOHalf, 12, true>(c, out, in, mutm, gamma5_out, dm, r2, nblocks_out, &eo);
}

// ------------------------------------------------------- reductions

// Two fixed-order stages: G blocks per (q, rhs) row each sum a contiguous
// segment of the row (four independent accumulators per thread, so several
// loads are in flight), then one block per row sums the G segment totals.
__global__ void __launch_bounds__(256) k_reduce_seg(const double *__restrict__ part, int nblk, int G,
                                                    double *__restrict__ seg) {
  __shared__ double sh[256];
  const int row = blockIdx.x / G, g = blockIdx.x - row * G;
  const int len = (nblk + G - 1) / G;
  const int b0 = g * len, b1 = min(nblk, b0 + len);
  const double *p = part + (size_t)row * nblk;
  double a0 = 0., a1 = 0., a2 = 0., a3 = 0.;
  int b = b0 + (int)threadIdx.x;
  for (; b + 768 < b1; b += 1024) {
    a0 += p[b];
    a1 += p[b + 256];
    a2 += p[b + 512];
    a3 += p[b + 768];
  }
  for (; b < b1; b += 256) a0 += p[b];
  sh[threadIdx.x] = (a0 + a1) + (a2 + a3);
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) sh[threadIdx.x] += sh[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) seg[blockIdx.x] = sh[0];
}

__global__ void k_reduce_partials(const double *__restrict__ part, int nblk, int Q, int N,
                                  double *__restrict__ res) {
  __shared__ double sh[256];
  (void)Q;
  (void)N;
  const double *row = part + (size_t)blockIdx.x * nblk;   // (q, rhs) = (blockIdx / N, blockIdx % N)
  double a = 0.;
  for (int b = threadIdx.x; b < nblk; b += blockDim.x) a += row[b];
  sh[threadIdx.x] = a;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) sh[threadIdx.x] += sh[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) res[blockIdx.x] = sh[0];
}

// segments of at least 4096 partials, at most kSegMax per row
constexpr int kSegMax = 64;

int reduce_stage1(cvchip_ctx *c, const double *part, int nblk, int rows, int slot, const double **out, int *n) {
  const int G = std::min(nblk / 4096, kSegMax);
  if (G < 2) {
    *out = part;
    *n = nblk;
    return 0;
  }
  if (slot < 0 || slot >= kReduceSlots || rows > kReduceRows) {
    set_error("partial sums: slot %d of %d, %d rows of %d", slot, kReduceSlots, rows, kReduceRows);
    return CVCHIP_ERR_STATE;
  }
  // every slot at the size of a full set of rows, so that no call grows the
  // scratch under another's result
  const size_t room = (size_t)kReduceRows * kSegMax;
  CVC_TRY(ensure_red2(c, sizeof(double) * kReduceSlots * room));
  double *seg = (double *)c->red2.ptr + slot * room;
  hipLaunchKernelGGL(k_reduce_seg, dim3(rows * G), dim3(256), 0, c->stream, part, nblk, G, seg);
  CVC_HIP(hipGetLastError());
  *out = seg;
  *n = G;
  return 0;
}

int reduce_partials(cvchip_ctx *c, const double *part, int nblk, int Q, int N, double *res) {
  const double *p = nullptr;
  int n = 0;
  CVC_TRY(reduce_stage1(c, part, nblk, Q * N, 0, &p, &n));
  hipLaunchKernelGGL(k_reduce_partials, dim3(Q * N), dim3(256), 0, c->stream, p, n, Q, N, res);
  CVC_HIP(hipGetLastError());
  return 0;
}

}  // namespace cvchip

using namespace cvchip;

extern "C" int cvchip_field_dslash(cvchip_ctx *c, cvchip_field *out, const cvchip_field *in,
                                   double mutm, int gamma5_out) {
  return cvchip::guarded("cvchip_field_dslash", [&]() -> int {
    if (!c || !out || !in) return CVCHIP_ERR_NULL;
    CVC_TRY(dslash(c, out->f, in->f, mutm, gamma5_out));
    CVC_HIP(hipStreamSynchronize(c->stream));
    return CVCHIP_OK;
  });
}

extern "C" int cvchip_field_dslash_timed(cvchip_ctx *c, cvchip_field *out, const cvchip_field *in,
                                         double mutm, int reps, double *ms) {
  return cvchip::guarded("cvchip_field_dslash_timed", [&]() -> int {
    if (!c || !out || !in || !ms) return CVCHIP_ERR_NULL;
    if (reps < 1) {
      set_error("reps must be positive");
      return CVCHIP_ERR_ARG;
    }
    CVC_HIP(hipEventRecord(c->ev0, c->stream));
    for (int k = 0; k < reps; k++) CVC_TRY(dslash(c, out->f, in->f, mutm, 0));
    CVC_HIP(hipEventRecord(c->ev1, c->stream));
    CVC_HIP(hipEventSynchronize(c->ev1));
    float t = 0.f;
    CVC_HIP(hipEventElapsedTime(&t, c->ev0, c->ev1));
    *ms = (double)t / reps;
    return CVCHIP_OK;
  });
}

extern "C" int cvchip_Q_phi(cvchip_ctx *c, double *xi, const double *phi, double mutm, int gamma5_out) {
  return cvchip::guarded("cvchip_Q_phi", [&]() -> int {
    if (!c || !xi || !phi) {
      set_error("NULL argument to cvchip_Q_phi");
      return CVCHIP_ERR_NULL;
    }
    TmpField a, b;
    int rc = field_alloc(c, a, 1, CVCHIP_PREC_F64);
    if (!rc) rc = field_alloc(c, b, 1, CVCHIP_PREC_F64);
    if (!rc) rc = upload_aos(c, a, phi, 0, 1);
    if (!rc) rc = dslash(c, b, a, mutm, gamma5_out);
    if (!rc) rc = download_aos(c, b, xi, 0, 1);
    return rc;
  });
}
