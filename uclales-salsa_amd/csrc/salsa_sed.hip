// salsa_sed.hip -- sedimentation of the SALSA categories (sedim_SALSA,
// mcrp.f90:745-921) on device: the liquid categories at levels 4 and 5, ice
// at level 5.
//
//   k_sed_zero   rrate, sfcrrate, VtPrc (level 5: irate, sfcirate, VtIce) to
//                zero (sedim_SALSA :792-795, DepositionFast :1127)
//   k_sed_slow   DepositionSlow (:926-1069) of one category, one workgroup
//                per interior column and one lane per level, one pass over
//                the bins: each bin's fall speeds (with the dry deposition
//                velocity at the lowest level) and fluxes, the level above's
//                fluxes through LDS, their divergence into the tendencies,
//                the water divergence into tlt (:810-816, :833-839), the rain
//                rate and at the lowest level the surface rate.  One launch
//                per category, so the accumulation into rrate / tlt keeps the
//                reference's order.
//   k_sed_prc    DepositionFast (:1073-1275) and its part of sedim_SALSA
//                (:862-878, :884-904) for precipitation (flag 3) or ice
//                (flag 4), one workgroup per interior column and one lane
//                per level: fall speeds into VtPrc / VtIce, the fall-distance
//                redistribution of every bin and moved quantity with each
//                level's changes summed in the reference's top-down order,
//                tendencies += change / dtlt, rate (bins in order), tlt and
//                the surface rate from the deposited mass.
// Terminal velocities: terminal_vel (mo_particle_external_properties.f90:
// 43-100), liquid and ice branches.  Contraction is off so that the products and
// sums round as the oracle's; the reference's x**(1./3.), x**1.5 and x**3. are
// formed as a cube root (FP32 seed and one Halley step), x*sqrt(x) and x*x*x,
// which differ from pow in the last bit only.
#include <hip/hip_runtime.h>

#include <stdint.h>

// (before the shared headers, so that their inline physics rounds the same way here)
#pragma clang fp contract(off)

#include "salsa_internal.h"
#include "salsa_physics.h"

namespace salsa {

namespace {

constexpr int kSedMaxZ = 256;                 // levels per column (SedArgs::dzt)
constexpr int kSedSpec = 3;                   // mass rows of a liquid bin that a context holds; ice has one more
constexpr double kPiFull = 3.14159265358979323846, kKb = 1.3807e-23, kG = 9.81, kCp = 1005., kAlvl = 2.5e6;
constexpr double kLn10 = 2.302585092994045684;

// x / d from the reciprocal r of d (to a few units in its last place): the
// residual of the product, formed exactly, corrects it to the correctly rounded
// quotient.  A divisor that many quotients share costs each of them three
// operations instead of a division's eleven.
__device__ __forceinline__ double sd_quot(double x, double d, double r) {
  const double q = x * r;
  return __builtin_fma(__builtin_fma(-q, d, x), r, q);
}

// Air at one level: viscosity, twice the mean free path, their reciprocals (every
// bin's fall speed divides by them), the viscosity over the density.
struct Air { double avis, iv, l2, il, nu; };
__device__ __forceinline__ Air sd_air(double tk, double adn) {
  Air a;
  const double tr = tk / 296.16;
  a.avis = 1.8325e-5 * (416.16 / (tk + 120.0)) * (tr * ::sqrt(tr));
  const double va = ::sqrt(8 * kKb * tk / (kPiFull * 4.8096e-26));
  a.l2 = 2. * (2 * a.avis / (adn * va));
  a.il = 1. / a.l2;
  a.iv = 1. / a.avis;
  a.nu = a.avis / adn;
  return a;
}

// rdiam: 1 / diam, as sd_quot takes it
__device__ __forceinline__ double sd_terminal_vel(double diam, double rdiam, double rhop, double rhoa, const Air &air,
                                                  double beta) {
  if (diam <= 19e-6) return sd_quot((diam * diam) * (rhop - rhoa) * kGrav * beta, 18. * air.avis, air.iv * (1. / 18.));
  if (diam > 19e-6 && diam < 1.07e-3) {
    const double NDa = sd_quot(4. / 3. * (diam * diam * diam) * kGrav * (rhop - rhoa) * rhoa, air.avis * air.avis, air.iv * air.iv);
    const double X = ::log(NDa);
    const double X2 = X * X, X3 = X2 * X, X4 = X2 * X2, X5 = X4 * X, X6 = X3 * X3;
    const double Y = -0.318657e1 + 0.992696 * X - 0.153193e-2 * X2 - 0.987059e-3 * X3 - 0.578878e-3 * X4 +
                     0.855176e-4 * X5 - 0.327815e-5 * X6;
    const double Re2 = beta * ::exp(Y);
    return sd_quot(air.nu, diam, rdiam) * Re2;
  }
  // Np**(1/6) through log(Np) / 6: X3 = log(Bo) + log(Np) / 6 and
  // Re3 = exp(log(Np) / 6 + Y3), within a few 1e-16 of the powers
  const double v2 = air.avis * air.avis;
  const double Np = (kSurfw0 * kSurfw0 * kSurfw0) * (rhoa * rhoa) / ((v2 * v2) * (rhop - rhoa) * kGrav);
  const double L6 = ::log(Np) / 6.;
  const double Bo = 4. / 3. * (rhop - rhoa) * kGrav / kSurfw0 * (diam * diam);
  const double X3 = ::log(Bo) + L6;
  const double Z2 = X3 * X3, Z3 = Z2 * X3, Z4 = Z2 * Z2, Z5 = Z4 * X3;
  const double Y3 = -0.500015e1 + 0.523778e1 * X3 - 0.204914e1 * Z2 + 0.475294 * Z3 - 0.542819e-1 * Z4 +
                    0.238449e-2 * Z5;
  const double Re3 = ::exp(L6 + Y3);
  return fmin(sd_quot(air.nu, diam, rdiam) * Re3, 9.2);
}

// the bin's wet diameter, density, slip correction and fall speed from the
// bin's number zpn >= 1e-15, volume v = sum m_s / rho_s and mass ms = sum m_s.
// (The density is formed with the diameter although it is ms / v: in the product
// of the diameter's cube and the density the rounding of the cube root cancels.)
__device__ __forceinline__ double sd_vc_sums(double zpn, double v, double ms, double adn, const Air &air,
                                             double *dwet_out, double *gg_out) {
  const double rn = rcp_nr(zpn);
  const double dwet = cbrt_fast(sd_quot(sd_quot(v, zpn, rn), kPi6, 1. / kPi6)), rdwet = rcp_nr(dwet);
  const double vp = kPi6 * (dwet * dwet * dwet);
  const double zdn = sd_quot(sd_quot(ms, zpn, rn), vp, rcp_nr(vp));
  const double Kn = dwet == 0. ? HUGE_VAL : sd_quot(air.l2, dwet, rdwet);
  const double GG = 1. + Kn * (1.249 + 0.42 * ::exp(sd_quot(-0.87 * dwet, air.l2, air.il)));
  if (dwet_out) *dwet_out = dwet;
  if (gg_out) *gg_out = GG;
  return sd_terminal_vel(dwet, rdwet, zdn, adn, air, GG);
}

__device__ __forceinline__ bool sd_interior(const SedArgs &a, int i, int j) {
  return i >= 2 && i <= a.nxp - 3 && j >= 2 && j <= a.nyp - 3;
}

__global__ void __launch_bounds__(256) k_sed_zero(SedArgs a) {
  const int64_t n3 = a.n3, ncol = (int64_t)a.nxp * a.nyp, nb = a.nb[2];
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n3; e += (int64_t)gridDim.x * blockDim.x) {
    a.rrate[e] = 0.;
    for (int b = 0; b < nb; ++b) a.vt_prc[b * n3 + e] = 0.;
    if (e < ncol) a.sfcrrate[e] = 0.;
    if (a.level == 5) {                         // irate, sfcirate, VtIce (:793-795, :1127)
      a.irate[e] = 0.;
      for (int b = 0; b < a.nb[3]; ++b) a.vt_ice[b * n3 + e] = 0.;
      if (e < ncol) a.sfcirate[e] = 0.;
    }
  }
}

// DepositionSlow (:926-1069) for category cat (0 aerosol, 1 cloud) on one
// interior column: one workgroup per column, one lane per level, one pass over
// the bins in order.  Per bin, every interior level reads its number and mass
// rows once, evaluates the fall speed (0 below the number limit; capped at
// half a level per step and 2 m/s; at the lowest level plus the dry
// deposition velocity) and publishes its fluxes times the air density in LDS
// (two buffers by bin parity, one barrier per bin); each level then takes the
// level above's from there (:1036-1049; 0 above the top interior level) and
// forms their divergence into the tendencies and, for the water row, into
// tlt (:810-816, :833-839).  The rain rate sums the flux entries
// (ns-1)*nb .. ns*nb (1-based, one entry early, as written) at the lane's
// level: the water rows' terms wait in LDS until the bin loop has produced
// the early entry (the last dry row of the last bin), which comes first; at
// the lowest level also the surface rate.  One launch per category keeps the
// reference's category order of the rrate / tlt accumulation.
template <int MS>
__global__ void __launch_bounds__(kSedMaxZ, MS <= 3 ? 3 : 1) k_sed_slow(SedArgs a, int cat) {
  extern __shared__ double sm[];
  const int Z = (int)blockDim.x;
  double *flx = sm;                             // [2][1 + MS][Z]: flux * adn of each level, by bin parity
  double *rt = sm + 2 * (1 + MS) * Z;           // [nb][Z]: the water rows' rain-rate terms of each level
  const int nx = a.nxp - 4;
  const int i = 2 + (int)blockIdx.x % nx, j = 2 + (int)blockIdx.x / nx;
  const int64_t col = (int64_t)i + (int64_t)a.nxp * j, n3 = a.n3;
  const int k = threadIdx.x, nzp = a.nzp;
  const int nb = a.nb[cat], ns = a.ns, iw = a.iwa;
  const bool src = k >= 1 && k <= nzp - 2;
  const int64_t x = col * nzp + k;
  const double *__restrict__ N = a.n_p[cat];
  const double *__restrict__ M = a.m_p[cat];
  double *__restrict__ Nt = a.n_t[cat];
  double *__restrict__ Mt = a.m_t[cat];
  double ad = 1., dz = 0., cap = 0., tkx = 0., ust = 0.;
  Air ar{};
  if (src) {
    ad = a.adn[x];
    tkx = a.tk[x];
    ar = sd_air(tkx, ad);
    dz = a.dzt[k];
    cap = fmin(0.5 * (1. / dz) / a.dtlt, 2.0);
    if (k == 1) ust = a.ustar[col];
  }
  // per-lane factor of the flux divergence (x * dz / adn rounded as x * (dz / adn))
  const double dza = dz / ad;
  double sdw = 0., t0 = 0.;
  uint64_t onm = 0;                             // bins at or above the number limit
  // the rows of bin b (number, masses, their tendencies), loaded one bin
  // ahead so that a bin's loads are in flight while the previous bin computes
  double qn = 0., qnt = 0., qm[MS], qmt[MS];
  auto load = [&](int b, double &n_, double &nt_, double *m_, double *mt_) {
    n_ = N[(int64_t)b * n3 + x];
    nt_ = Nt[(int64_t)b * n3 + x];
#pragma unroll
    for (int s = 0; s < MS; ++s) {
      const int64_t r = ((int64_t)s * nb + b) * n3 + x;
      m_[s] = s < ns ? M[r] : 0.;
      mt_[s] = s < ns ? Mt[r] : 0.;
    }
  };
#pragma unroll
  for (int s = 0; s < MS; ++s) qm[s] = qmt[s] = 0.;
  if (src) load(0, qn, qnt, qm, qmt);
  for (int b = 0; b < nb; ++b) {
    double *F = flx + (b & 1) * (1 + MS) * Z;
    const double zpn = qn, znt = qnt;
    double m[MS], mt[MS];
#pragma unroll
    for (int s = 0; s < MS; ++s) {
      m[s] = qm[s];
      mt[s] = qmt[s];
    }
    if (src && b + 1 < nb) load(b + 1, qn, qnt, qm, qmt);
    double vc = 0.;
    const bool on = src && !(zpn < kNlim);
    if (on) {
      double v = 0., ms = 0.;
#pragma unroll
      for (int s = 0; s < MS; ++s)
        if (s < ns) v = v + sd_quot(m[s], a.rholiq[s], a.rrholiq[s]);
#pragma unroll
      for (int s = 0; s < MS; ++s)
        if (s < ns) ms = ms + m[s];
      double dwet, GG;
      vc = sd_vc_sums(zpn, v, ms, ad, ar, &dwet, &GG);
      vc = fmin(vc, cap);
      if (k == 1) {                               // the level just above the surface
        // Sc**(-2/3) and 10**(-3/St) as exponentials of logarithms (a few
        // 1e-15 from the powers; Sc is the Schmidt number, 10**(-3/St) >= 1e-300)
        const double mdiff = (kKb * tkx * GG) / (3.0 * kPiFull * ar.avis * dwet);
        const double Sc = (ar.avis / ad) / mdiff;
        double St = vc * (ust * ust) / kG * (ar.avis / ad);
        if (St < 0.01) St = 0.01;
        const double rtr = 1.0 / fmax(kEpsR8, (ust * (::exp(-2.0 / 3.0 * ::log(Sc)) + ::exp(-3.0 / St * kLn10))));
        vc = (1. / rtr) + vc;
      }
      onm |= (uint64_t)1 << b;
#pragma unroll
      for (int s = 0; s < MS; ++s) {
        if (s == ns - 1) rt[b * Z + k] = -m[s] * vc;
        if (s == ns - 2 && b == nb - 1) t0 = -m[s] * vc;
      }
    }
    // the fluxes rfn, rfm (0 below the limit and outside the interior) times adn
    const double Pn = (on ? -zpn * vc : 0.) * ad;
    double Pm[MS];
#pragma unroll
    for (int s = 0; s < MS; ++s) Pm[s] = (on ? -m[s] * vc : 0.) * ad;
    F[k] = Pn;
#pragma unroll
    for (int s = 0; s < MS; ++s)
      if (s < ns) F[(1 + s) * Z + k] = Pm[s];
    __syncthreads();
    if (src) {
      const double dn = (F[k + 1] - Pn) * dza;
      Nt[(int64_t)b * n3 + x] = znt - dn;
#pragma unroll
      for (int s = 0; s < MS; ++s) {
        if (s < ns) {
          const double dm = (F[(1 + s) * Z + k + 1] - Pm[s]) * dza;
          Mt[((int64_t)s * nb + b) * n3 + x] = mt[s] - dm;
          if (s == iw) sdw = sdw + dm;
        }
      }
    }
  }
  if (!src) return;                             // no barrier below
  // rain rate over the flux entries (ns-1)*nb .. ns*nb (1-based), as written
  double sw = 0.;
  if ((onm >> (nb - 1)) & 1) sw = sw + t0;
  for (int b = 0; b < nb; ++b)
    if ((onm >> b) & 1) sw = sw + rt[b * Z + k];
  a.rrate[x] = a.rrate[x] - sw * ad * kAlvl;
  a.tlt[x] = a.tlt[x] + sdw * (kAlvl / kCp) * a.th[x] / a.tk[x];
  if (k == 1) a.sfcrrate[col] = a.sfcrrate[col] - sw * ad * kAlvl;
}

// LDS of k_sed_slow<MS> for blockDim Z and nb bins: the flux buffers and the
// rain-rate terms
size_t sed_slow_lds_bytes(int Z, int nb, int MS) {
  return ((size_t)2 * (1 + MS) * Z + (size_t)nb * Z) * sizeof(double);
}

// DepositionFast for one category on one interior column: one workgroup per
// column, one lane per level (blockDim = nzp rounded up to 64).  Per bin, in
// order:
//   1. every source level k (1 <= k <= nzp-2 with N >= prlim) evaluates its
//      fall speed (VtPrc / VtIce) and its fall-distance decision
//      (:1188-1225): the landing level kf, one or two receiving levels and
//      their shares;
//   2. per moved quantity (the number, then the mass species), every level L
//      sums what lands on it from the sources above it, in decreasing source
//      level as the reference's top-down walk adds them, then its own
//      departure (-q) and, when the particles stay within the level, its own
//      share; the change goes straight into the tendency (/ dtlt).  Only
//      sources within the column's largest fall distance of L are scanned.
// Deposited mass (sources whose walk reaches the surface) is summed per
// species and bin by lane 0 over those sources, top down.  Rate (bins in
// order), tlt and the surface rate as in sedim_SALSA (:862-878, :884-904).
// ICE: flag 4 -- the fall speed of non-spherical ice (calcDiamLES both ways,
// getShapeCoefficients, terminal_vel's ice branch), water and rime in the
// rate, the surface rate and tlt, latent heat alvi; MS: the most mass rows
// per bin (registers per level).

// The ice fall speed of one bin (DepositionFast flag 4: calcDiamLES,
// getShapeCoefficients and getDiameter, mo_ice_shape.f90:47-86, 145-191;
// terminal_vel's ice branch, mo_particle_external_properties.f90:91-98)
// with its powers taken in the log domain: the mass thresholds Mth, Mgr,
// Mcr and the non-spherical diameter as logarithms (Mgr = rho_b pi6 Dgr**3,
// Dgr = (alpha / (pi6 rho_b))**(1/(3-beta)), Dcr = Dgr h**(1/(3-beta))),
// the Best number X = 2 vb (rhop-rhoa) g / (gamma rhoa visc**2) D**(2-sigma)
// and the speed Are / X**bre * visc**(1-2 bre) * (2 alpha g / (rhoa gamma))**bre
// * D**bv as one exponential: five logarithms and two exponentials per bin
// instead of eight powers, within a few 1e-14 of the power form.  The constants
// and the level's viscosity and density go into the arguments of the logarithms
// of X and of the factor, not in as logarithms of their own, whose roundings are
// larger than the result.  numc: the number, v, ms: volume sum m / rho and mass
// sum m of the bin; visc, lvisc, rv2: the level's viscosity, its logarithm and
// 1 / visc**2; rrhoa: 1 / rhoa; c: of the constants.
struct IceLogC { double lmth, lia, lpi6ic, rga, inv, rib; };   // rga 1 / gamma, inv 1 / (3 - beta), rib 1 / beta
__device__ __forceinline__ double ice_vc_log(const SedArgs &a, const IceLogC &c, double v, double ms, double rhoa,
                                             double visc, double lvisc, double rv2, double rrhoa, double mpri, double mrim,
                                             double numc) {
  double al = kPi6 * kRhoic, be = 3., ga = kPi / 4., rga = 4. / kPi, si = 2.;
  double Ld = -20.72326583694641;               // log(1e-9): getDiameter's value below the number limit
  const double rn = rcp_nr(numc);
  if (!(numc < 1.e-6)) {
    const double mtot = sd_quot(mpri + mrim, numc, rn), mt = mtot * numc;
    const double fr = fmax(fmin(sd_quot(mrim, mt, rcp_nr(mt)), 0.9999), 0.0001);
    const double rho_b = fr * kRhori + (1. - fr) * kRhoic;
    const double Lm = ::log(mtot), Lrb = ::log(kPi6 * rho_b);
    const double lmgr = Lrb + 3. * ((c.lia - Lrb) * c.inv);
    const double h = sd_quot(1., 1. - fr, rcp_nr(1. - fr)), Lh = ::log(h);
    const double lmcr = lmgr + 3. * (Lh * c.inv);
    if (Lm >= c.lmth && Lm < lmgr) {
      al = a.ice_alpha; be = a.ice_beta; ga = a.ice_gamma; rga = c.rga; si = a.ice_sigma;
    } else if (Lm > lmcr) {
      al = a.ice_alpha * h; be = a.ice_beta; si = a.ice_sigma * (1. - fr) + 2. * fr;
      ga = a.ice_gamma * (1. - fr) + kPi / 4. * fr;
      rga = rcp_nr(ga);
    }
    if (Lm < c.lmth) Ld = sd_quot(Lm - c.lpi6ic, 3., 1. / 3.);
    else if (Lm < lmgr) Ld = sd_quot(Lm - c.lia, a.ice_beta, c.rib);
    else if (Lm < lmcr) Ld = sd_quot(Lm - Lrb, 3., 1. / 3.);
    else if (Lm >= lmcr) Ld = sd_quot(Lm - Lh - c.lia, a.ice_beta, c.rib);
  }
  const double c1 = 0.0902, delta0 = 9.06;
  const double dsph = cbrt_fast(sd_quot(sd_quot(v, numc, rn), kPi6, 1. / kPi6)), vb = kPi6 * cubed(dsph);
  const double zdn = sd_quot(sd_quot(ms, numc, rn), vb, rcp_nr(vb)), rgr = rga * rrhoa;
  const double LX = ::log(sd_quot(2. * vb * (zdn - rhoa) * kGrav, ga * rhoa * visc * visc, rgr * rv2)) + (2. - si) * Ld;
  const double sX = ::sqrt(::exp(LX));
  const double k1213 = ::sqrt(1. + c1 * sX), k1 = k1213 - 1.;
  const double bre = 0.5 * c1 * sX / k1 / k1213;
  const double bv = bre * (be - si + 2.) - 1.;
  const double Lc = ::log(sd_quot(2. * al * kGrav, rhoa * ga, rgr));
  return 0.25 * delta0 * delta0 * k1 * k1 * ::exp(-bre * LX + (1. - 2. * bre) * lvisc + bre * Lc + bv * Ld);
}

// LDS of one column (Z = blockDim.x levels), carved from the dynamic buffer
// in this order: dz, rdz [Z]; by bin parity f1, f0 (shares of a source's
// content that land one level below kf and on it), av (air density times fall
// speed) [2][Z] and q (its number and masses) [2][1 + MS][Z]; rem [ns*nb]
// (deposited mass per species and bin); then the ints dec [2][Z] (bit 0
// source, 1 two levels, 2 deposits; (d + 1) << 8) and wmax [2][4] (largest
// fall distance per wavefront).
__host__ __device__ inline size_t sed_prc_lds_bytes(int Z, int nb, int ns, int MS) {
  return (size_t)((8 + 2 * (1 + MS)) * Z + ns * nb) * sizeof(double) + (size_t)(2 * Z + 8) * sizeof(int);
}

// Bound by the fall speed's FP64 arithmetic and, at level 4, HBM.  One barrier
// per bin: a source publishes its content and the two shares, and every level
// scans the sources above it once for all quantities.  With a barrier and a
// scan per bin and moved quantity (35 and 21 of them) the ice launch took 929 us
// at 128 x 128 x 100 cells and the precipitation launch 127 us at 64 x 64 x 120;
// now 694 and 106 us, with the fall speeds' bits as they were.  (Reciprocals
// without sd_quot's correction: 617 and 98 us, but fall speeds further from the
// exact value, 5.3 against 4.6 units of 2^-53 rms.  Four wavefronts per SIMD,
// with 14 to 34 spills, 698 and 124 us before the ice speed took its
// diameter again, three 652 and 108 us.)
template <int MS, bool ICE>
__global__ void __launch_bounds__(kSedMaxZ, 3) k_sed_prc(SedArgs a) {
  extern __shared__ double smem[];
  constexpr int cat = ICE ? 3 : 2;
  constexpr double alv = ICE ? kAls : kAlvl;
  const int nx = a.nxp - 4;
  const int i = 2 + (int)blockIdx.x % nx, j = 2 + (int)blockIdx.x / nx;
  const int64_t col = (int64_t)i + (int64_t)a.nxp * j, n3 = a.n3;
  const int k = threadIdx.x, nzp = a.nzp, ktop = nzp - 2, nw = blockDim.x / 64;
  const int nb = a.nb[cat], ns = ICE ? a.ns_ice : a.ns, iw = a.iwa, ir = a.irim;
  const int Z = blockDim.x;
  double *const Sdz = smem, *const Srdz = smem + Z, *const Sf1 = smem + 2 * Z, *const Sf0 = smem + 4 * Z;
  double *const Sav = smem + 6 * Z, *const Sq = smem + 8 * Z, *const Srem = Sq + 2 * (1 + MS) * Z;
  int *const Sdec = reinterpret_cast<int *>(Srem + ns * nb);
  int *const Swmax = Sdec + 2 * Z;
  const double *__restrict__ Np = a.n_p[cat];
  const double *__restrict__ Mp = a.m_p[cat];
  double *__restrict__ Nt = a.n_t[cat];
  double *__restrict__ Mt = a.m_t[cat];
  double *__restrict__ vt = ICE ? a.vt_ice : a.vt_prc;
  double *__restrict__ rate = ICE ? a.irate : a.rrate;
  double *__restrict__ srate = ICE ? a.sfcirate : a.sfcrrate;
  const bool lev = k < nzp, src = k >= 1 && k <= ktop;
  const int64_t x = col * nzp + k;
  const double dtlt = a.dtlt, rdt = 1. / dtlt;
  // the bin's rows at this level, quantity u: 0 the number, 1 + s species s
  // (the next bin's are loaded while the current one is worked on)
  double qv[MS + 1], tv[MS + 1], qn[MS + 1], tn[MS + 1];
  auto load = [&](int b, double *q, double *t) {
#pragma unroll
    for (int u = 0; u <= MS; ++u) {
      const bool use = lev && b < nb && u <= ns;
      const int64_t r = u == 0 ? (int64_t)b * n3 : ((int64_t)(u - 1) * nb + b) * n3;
      q[u] = use ? (u == 0 ? Np : Mp)[r + x] : 0.;
      t[u] = use ? (u == 0 ? Nt : Mt)[r + x] : 0.;
    }
  };
  load(0, qv, tv);
  Air air{};
  double rr = 0., sw = 0., sr = 0., ad = 0., lvisc = 0., rv2 = 0., rrhoa = 0.;
  IceLogC ilc{};                                        // ice: log Mth (pristine threshold), log alpha, log(pi6 rhoic), ..
  if (ICE) {
    const double dth = ::pow(kPi6 * kRhoic / a.ice_alpha, 1. / (a.ice_beta - 3.));
    ilc.lmth = ::log(kRhoic * kPi6 * cubed(dth));
    ilc.lia = ::log(a.ice_alpha);
    ilc.lpi6ic = ::log(kPi6 * kRhoic);
    ilc.rga = 1. / a.ice_gamma;
    ilc.inv = 1. / (3. - a.ice_beta);
    ilc.rib = 1. / a.ice_beta;
  }
  if (lev) {
    Sdz[k] = a.dzt[k];
    Srdz[k] = 1. / a.dzt[k];
    ad = a.adn[x];
  }
  if (src) {
    air = sd_air(a.tk[x], ad);
    if (ICE) {
      lvisc = ::log(air.avis);
      rv2 = air.iv * air.iv;
      rrhoa = 1. / ad;
    }
    rr = rate[x];
  }
  __syncthreads();
  for (int b = 0; b < nb; ++b) {
    const int pb = b & 1;
    double *const Q = Sq + pb * (1 + MS) * Z;
    load(b + 1, qn, tn);
    const double zpn = qv[0];
    const bool on = src && !(zpn < kPrlim);
    double f1 = 0., f0 = 0.;
    int d = -1;
    bool two = false, dep = false;
    if (on) {
      double v = 0., ms = 0., vc, wv = 0., rv = 0.;
#pragma unroll
      for (int s = 0; s < MS; ++s)
        if (s < ns) {
          v = v + sd_quot(qv[1 + s], (ICE ? a.rhoice : a.rholiq)[s], (ICE ? a.rrhoice : a.rrholiq)[s]);
          ms = ms + qv[1 + s];
        }
#pragma unroll
      for (int s = 0; s < MS; ++s) {
        if (s == iw) wv = qv[1 + s];
        if (s == ir) rv = qv[1 + s];
      }
      if (ICE) {
        // calcDiamLES (mo_particle_external_properties.f90:169-201) both
        // ways, getShapeCoefficients, the bulk density, terminal_vel flag 4
        double mpri = 0., mrim = 0.;
#pragma unroll
        for (int s = 0; s < MS; ++s) {
          if (s < ns - 1) mpri = mpri + qv[1 + s];
          if (s == ns - 1) mrim = qv[1 + s];
        }
        vc = ice_vc_log(a, ilc, v, ms, ad, air.avis, lvisc, rv2, rrhoa, mpri, mrim, zpn);
      } else {
        vc = sd_vc_sums(zpn, v, ms, ad, air, nullptr, nullptr);
      }
      vt[(int64_t)b * n3 + x] = vc;
      // the rate: water (and, for ice, rime) falling out of the level (:1206-1212)
      rr = ICE ? rr + (wv + rv) * ad * vc * alv : rr + wv * ad * vc * alv;
      const double fdmax = dtlt * vc;
      double fd = 0.;
      int fi = 0;
      while (fd < fdmax) {                      // bounded: ends at the lowest level
        fd = fd + Srdz[k - fi];
        fi = fi + 1;
        if (k - fi <= 0) { dep = true; break; }
      }
      fi = fi - 1;
      const int kf = k - fi;                    // kf - 1 >= 0; kf <= k + 1 <= nzp - 1
      fd = fd - Srdz[kf];
      const double fdos = fmin(fmax(fdmax - fd, 0.), Srdz[kf]);
      const double pre = fdos * Sdz[kf];
      two = !(pre > 0.5);
      // the shares (:1229-1246), thinner or thicker levels included
      const int kb = two ? kf : k;
      f1 = sd_quot((two ? pre : 1.) * Sdz[kf - 1], Sdz[kb], Srdz[kb]);
      f0 = two ? 1. - pre : 0.;
      d = k - kf;                               // >= -1
      Sf1[pb * Z + k] = f1;
      Sf0[pb * Z + k] = f0;
      Sav[pb * Z + k] = ad * vc;
#pragma unroll
      for (int u = 0; u <= MS; ++u) Q[u * Z + k] = qv[u];
    }
    Sdec[pb * Z + k] = on ? (1 | (two ? 2 : 0) | (dep ? 4 : 0) | ((d + 1) << 8)) : 0;
    int wm = d;
    for (int o = 32; o > 0; o >>= 1) wm = max(wm, __shfl_xor(wm, o));
    if ((k & 63) == 0) Swmax[pb * 4 + (k >> 6)] = wm;
    __syncthreads();
    int dmax = -1;
    for (int w = 0; w < nw; ++w) dmax = max(dmax, Swmax[pb * 4 + w]);
    double out[MS + 1];
#pragma unroll
    for (int u = 0; u <= MS; ++u) out[u] = 0.;
    if (lev && k <= ktop) {
      // what lands here, from the top down as the reference adds it
      for (int s = min(ktop, k + dmax + 1); s > k; --s) {
        const int ds = Sdec[pb * Z + s], kf = s - ((ds >> 8) - 1);
        const bool l1 = kf - 1 == k, l0 = (ds & 2) && kf == k;
        if (!(ds & 1) || !(l1 || l0)) continue;
        const double f = l1 ? Sf1[pb * Z + s] : Sf0[pb * Z + s];
#pragma unroll
        for (int u = 0; u <= MS; ++u) out[u] = out[u] + f * Q[u * Z + s];
      }
      if (on) {
        // what leaves, and what does not leave the level
        const double own = d == -1 ? f1 : (two && d == 0 ? f0 : 0.);
#pragma unroll
        for (int u = 0; u <= MS; ++u) {
          out[u] = out[u] - qv[u];
          if (d <= 0) out[u] = out[u] + own * qv[u];
        }
      }
    }
    if (lev) {
#pragma unroll
      for (int u = 0; u <= MS; ++u) {
        if (u > ns) break;
        const int64_t r = u == 0 ? (int64_t)b * n3 : ((int64_t)(u - 1) * nb + b) * n3;
        (u == 0 ? Nt : Mt)[r + x] = tv[u] + sd_quot(out[u], dtlt, rdt);
        if (u - 1 == iw) sw = sw + out[u];
        if (ICE && u - 1 == ir) sr = sr + out[u];
      }
    }
    if (k == 0) {                               // lane 0 (level 0 is never a source)
      double r[MS];
#pragma unroll
      for (int s = 0; s < MS; ++s) r[s] = 0.;
      for (int s = min(ktop, dmax + 1); s >= 1; --s)
        if ((Sdec[pb * Z + s] & 5) == 5)
#pragma unroll
          for (int u = 0; u < MS; ++u) r[u] = r[u] + Q[(1 + u) * Z + s] * Sav[pb * Z + s];
#pragma unroll
      for (int u = 0; u < MS; ++u)
        if (u < ns) Srem[u * nb + b] = r[u];
    }
#pragma unroll
    for (int u = 0; u <= MS; ++u) {
      qv[u] = qn[u];
      tv[u] = tn[u];
    }
  }
  if (src) rate[x] = rr;
  // the water rows and, for ice, the rime rows
  if (lev && k <= ktop) a.tlt[x] = a.tlt[x] - ((sw + sr) / dtlt) * (alv / kCp) * a.th[x] / a.tk[x];
  if (k == 0) {
    // SUM(remprc((ns-1)*nb:ns*nb)) (ice: (ns-2)*nb:ns*nb), 1-based, one entry
    // before the water rows as written (:1256-1260)
    double s2 = 0.;
    for (int q = (ICE ? ns - 2 : ns - 1) * nb - 1; q < ns * nb; ++q) s2 = s2 + Srem[q];
    srate[col] = srate[col] + s2 * alv;
  }
}

}  // namespace

int launch_sedim(const SedArgs &a, int sed_aero, int sed_cloud, int sed_precp, int sed_ice, hipStream_t s) {
  const unsigned g256 = (unsigned)((a.n3 + 255) / 256);
  hipLaunchKernelGGL(k_sed_zero, dim3(g256 < 65536 ? g256 : 65536), dim3(256), 0, s, a);
  for (int cat = 0; cat < 2; ++cat) {
    if (!(cat == 0 ? sed_aero : sed_cloud)) continue;
    // one workgroup per interior column, one lane per level; the fluxes of
    // one bin and the column's rain-rate terms in LDS
    const unsigned ncol = (unsigned)((a.nxp - 4) * (a.nyp - 4)), nthr = (unsigned)((a.nzp + 63) / 64 * 64);
    const size_t lds = sed_slow_lds_bytes((int)nthr, a.nb[cat], kSedSpec);
    if (a.nzp > kSedMaxZ || a.nb[cat] > 64 || a.ns < 2 || a.ns > kSedSpec || lds > 65536) return (int)hipErrorInvalidValue;
    hipLaunchKernelGGL(k_sed_slow<kSedSpec>, dim3(ncol), dim3(nthr), lds, s, a, cat);
  }
  if (sed_precp) {
    // one workgroup per interior column, one lane per level
    const unsigned ncol = (unsigned)((a.nxp - 4) * (a.nyp - 4)), nthr = (unsigned)((a.nzp + 63) / 64 * 64);
    const size_t lds = sed_prc_lds_bytes((int)nthr, a.nb[2], a.ns, kSedSpec);
    if (a.nzp > kSedMaxZ || a.ns > kSedSpec || lds > 65536) return (int)hipErrorInvalidValue;
    hipLaunchKernelGGL((k_sed_prc<kSedSpec, false>), dim3(ncol), dim3(nthr), lds, s, a);
  }
  if (sed_ice && a.level == 5) {
    const unsigned ncol = (unsigned)((a.nxp - 4) * (a.nyp - 4)), nthr = (unsigned)((a.nzp + 63) / 64 * 64);
    const size_t lds = sed_prc_lds_bytes((int)nthr, a.nb[3], a.ns_ice, kSedSpec + 1);
    if (a.nzp > kSedMaxZ || a.ns_ice > kSedSpec + 1 || lds > 65536) return (int)hipErrorInvalidValue;
    hipLaunchKernelGGL((k_sed_prc<kSedSpec + 1, true>), dim3(ncol), dim3(nthr), lds, s, a);
  }
  return (int)hipGetLastError();
}

}  // namespace salsa
