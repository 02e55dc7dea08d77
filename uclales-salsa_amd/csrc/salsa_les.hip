// salsa_les.hip -- the LES side of a SALSA step on device: what cfll does
// after run_SALSA (step.f90:330-333) for the SALSA tracers, so that the
// prognostic fields never leave HBM between steps.
//
//   k_les_cells   interior columns, one lane per cell, every row once:
//                 tend_constrain2 (constrain_SALSA.f90:18-36), update
//                 (step.f90:470-489), tend0 (step.f90:379-396), the bottom and
//                 top rows of sclrset 'mixd' (util.f90:71-107: the bottom
//                 copies k = 2, the top extrapolates with dzf2 =
//                 dzt(nzp-2)/dzt(nzp-1)), SALSA_diagnostics' clamps
//                 (constrain_SALSA.f90:88-100) and diagnostic sums (:370-400),
//                 and a list of the cells that its removals may change;
//                 a column at an edge writes its periodic images too
//                 (cyclics/cyclicc of a process that owns the whole grid).
//   k_les_remove  SALSA_diagnostics' removals (:103-366) on the listed cells:
//                 particles with number but no mass, cloud / precipitation /
//                 ice bins that evaporated back to the aerosol bins
//                 (findDry4Wet :408-470 for precipitation and ice), aerosols
//                 below 0.1 nm dry diameter; each cell's rows staged in LDS
//                 where they fit, the bins in the reference's order.
//   k_les_start   the list empty; a_indefp clamped when registered (:33-34).
//
// The passes are HBM-bound byte movers, coalesced along k (the fastest LES
// index).  Floating-point contraction is off so that every sum
// and product rounds as written.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <type_traits>

#include "salsa_internal.h"

#pragma clang fp contract(off)

namespace salsa {

namespace {

constexpr double kMassTH = 1.e-25;    // constrain_SALSA.f90:65
constexpr int kLesCells = 64;         // listed cells per workgroup of the LDS removal pass
constexpr int kLesLdsRows = 128;      // rows per cell that fit its 64 KiB of LDS

// The list of this call starts empty; a_indefp to [0, 1] (tend_constrain2, :33-34).
__global__ void __launch_bounds__(256) k_les_start(LesArgs a, int64_t nind) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *a.count = 0;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < nind; e += (int64_t)gridDim.x * blockDim.x)
    a.indef[e] = fmin(fmax(a.indef[e], 0.), 1.);
}

// One cell's tracer rows, either in the LES arrays (row stride n3) or staged
// in LDS (row stride = cells per workgroup): N(c, b) = n[c][b * rs],
// M(c, s, b) = m[c][(s * nb[c] + b) * rs].
struct LesCell {
  double *n[4], *m[4];
  int64_t rs;
  __device__ __forceinline__ double &N(const LesArgs &a, int c, int b) const { return n[c][b * rs]; }
  __device__ __forceinline__ double &M(const LesArgs &a, int c, int s, int b) const {
    return m[c][((int64_t)s * a.nb[c] + b) * rs];
  }
};

// findDry4Wet for an evaporating bin (number ne, dry masses md[s * mstride])
__device__ __forceinline__ int les_dry4wet(const LesArgs &a, const LesCell &C, double ne, const double *md,
                                           int64_t mstride) {
  const int ndry = a.ndry;
  double cd = 0.;
  for (int s = 0; s < ndry; ++s) cd = cd + md[s * mstride] / a.rholiq[s];
  cd = cd / ne;
  cd = ::pow(cd / kPi6, 1. / 3.);
  int cnt = 0;
  for (int b = a.in2a; b <= a.fn2a; ++b) cnt += cd > a.aerobins[b];
  int ba = a.in2a + cnt - 1;
  ba = ba < a.in2a ? a.in2a : ba;
  ba = ba > a.fn2a ? a.fn2a : ba;
  const int bb = a.fn2a + (ba - a.in2a);   // as written in the reference (:443)
  if (C.N(a, 0, bb) <= kNlim) return ba;
  if (C.N(a, 0, ba) <= kNlim) return bb;
  // calc_correlation of the dry masses; sxy keeps the last product only
  // (util.f90:1017)
  double r[2];
  for (int q = 0; q < 2; ++q) {
    const int bx = q ? bb : ba;
    double sx = 0., sy = 0., sx2 = 0., sy2 = 0., sxy = 0.;
    for (int s = 0; s < ndry; ++s) {
      const double xv = C.M(a, 0, s, bx), yv = md[s * mstride];
      sx = sx + xv;
      sy = sy + yv;
      sx2 = sx2 + xv * xv;
      sy2 = sy2 + yv * yv;
      sxy = xv * yv;
    }
    const double n = (double)ndry;
    r[q] = (sx2 * n - sx * sx < kEpsR8 || sy2 * n - sy * sy < kEpsR8)
               ? 0.
               : (sxy * n - sx * sy) / (::sqrt(sx2 * n - sx * sx) * ::sqrt(sy2 * n - sy * sy));
  }
  return r[0] < r[1] ? bb : ba;
}

// SALSA_diagnostics' removals on an interior cell (constrain_SALSA.f90:
// 103-366) in the reference's order; x is the cell's LES index (for the
// charge-time rows).  Returns whether any value changed.
__device__ __forceinline__ bool les_remove(const LesArgs &a, const LesCell &C, int64_t x, double T, double rh,
                                           double rhi) {
  const int nwet = a.nwet, ndry = a.ndry, iwa = a.iwa, irim = a.irim;
  const int64_t n3 = a.n3;
  bool mod = false;
  auto N = [&](int c, int b) -> double & { return C.N(a, c, b); };
  auto M = [&](int c, int s, int b) -> double & { return C.M(a, c, s, b); };
  auto ctime = [&](int row) {
    if (a.charge_time) a.charge_time[(int64_t)row * n3 + x] = 0.;
  };
  // particles with number but no mass (:103-154)
#pragma unroll
  for (int c = 0; c < 2; ++c)
    for (int b = 0; b < a.nb[c]; ++b) {
      double sm = 0.;
      for (int s = 0; s < nwet; ++s) sm = sm + M(c, s, b);
      if (N(c, b) > 0. && sm <= 0.) {
        N(c, b) = 0.;
        for (int s = 0; s < nwet; ++s) M(c, s, b) = 0.;
        ctime(c == 0 ? b : a.nb[0] + b);
        mod = true;
      }
    }
  for (int b = 0; b < a.nb[2]; ++b)
    if (N(2, b) > 0. && M(2, iwa, b) <= 0.) {
      N(2, b) = 0.;
      for (int s = 0; s < nwet; ++s) M(2, s, b) = 0.;
      ctime(a.nb[0] + a.nb[1] + b);
      mod = true;
    }
  if (a.level == 5)
    for (int b = 0; b < a.nb[3]; ++b) {
      const double mt = M(3, iwa, b) + M(3, irim, b);
      if (N(3, b) > 0. && mt < kMassTH) {
        N(3, b) = 0.;
        for (int s = 0; s <= irim; ++s) M(3, s, b) = 0.;
        mod = true;
      }
    }
  // cloud droplets that evaporated (:156-207)
  for (int bc = a.ica_cur; bc <= a.fcb_cur; ++bc) {
    if (!(N(1, bc) > kNlim && rh < 0.999 && M(1, iwa, bc) < 1.e-5)) continue;
    double ns = 0.;
    for (int s = 0; s < ndry; ++s) ns = ns + a.diss[s] * M(1, s, bc) / a.mm[s];
    ns = ns / N(1, bc);
    const double zbb = 6. * kMwa * ns / (kPi * kRhowa);
    const double zaa = 4. * kMwa * kSurfw0 / (kRg * kRhowa * T);
    const double cdcld = ::sqrt(3. * zbb / zaa);
    double zvol = 0.;
    for (int s = 0; s < nwet; ++s) zvol = zvol + M(1, s, bc) / a.rholiq[s];
    zvol = zvol / N(1, bc);
    const double zdh2o = ::pow(zvol / kPi6, 1. / 3.);
    if (zdh2o < fmin(0.7 * cdcld, 1.3e-5) || M(1, iwa, bc) < kMassTH * N(1, bc)) {
      const int ba = bc <= a.fca_cur ? a.ica_par + (bc - a.ica_cur) : a.icb_par + (bc - a.icb_cur);
      N(0, ba) = N(0, ba) + N(1, bc);
      N(1, bc) = 0.;
      for (int s = 0; s < nwet; ++s) {
        M(0, s, ba) = M(0, s, ba) + M(1, s, bc);
        M(1, s, bc) = 0.;
      }
      ctime(a.nb[0] + bc);
      mod = true;
    }
  }
  // precipitation that evaporated (:209-258)
  for (int bc = 0; bc < a.nb[2]; ++bc) {
    if (!(N(2, bc) > kPrlim && rh < 0.999 && M(2, iwa, bc) < 1.e-6)) continue;
    double ns = 0.;
    for (int s = 0; s < ndry; ++s) ns = ns + a.diss[s] * M(2, s, bc) / a.mm[s];
    ns = ns / N(2, bc);
    const double zbb = 6. * kMwa * ns / (kPi * kRhowa);
    const double zaa = 4. * kMwa * kSurfw0 / (kRg * kRhowa * T);
    const double cdprc = ::sqrt(3. * zbb / zaa);
    double zvol = 0.;
    for (int s = 0; s < nwet; ++s) zvol = zvol + M(2, s, bc) / a.rholiq[s];
    zvol = zvol / N(2, bc);
    const double zdh2o = ::pow(zvol / kPi6, 1. / 3.);
    if (zdh2o < fmin(0.2 * cdprc, 10.e-6) || M(2, iwa, bc) < kMassTH * N(2, bc)) {
      const int ba = les_dry4wet(a, C, N(2, bc), &M(2, 0, bc), (int64_t)a.nb[2] * C.rs);
      N(0, ba) = N(0, ba) + N(2, bc);
      N(2, bc) = 0.;
      for (int s = 0; s < nwet; ++s) {
        M(0, s, ba) = M(0, s, ba) + M(2, s, bc);
        M(2, s, bc) = 0.;
      }
      ctime(a.nb[0] + a.nb[1] + bc);
      mod = true;
    }
  }
  // ice that sublimated (:260-315)
  if (a.level == 5) {
    for (int bc = 0; bc < a.nb[3]; ++bc) {
      const double mt = M(3, iwa, bc) + M(3, irim, bc);
      double vt = 0.;
      for (int s = 0; s <= irim; ++s) vt = vt + M(3, s, bc) / a.rhoice[s];
      if (!(N(3, bc) > kPrlim && rhi < 0.999 && mt < 1.e-15)) continue;
      double cdice = vt / N(3, bc);
      cdice = ::pow(cdice / kPi6, 1. / 3.);
      double zdrms = 0., zwams = 0.;
      for (int s = 0; s < ndry; ++s) zdrms = zdrms + M(3, s, bc);
      for (int s = 0; s <= irim; ++s) zwams = zwams + M(3, s, bc);
      const double zvol = zdrms / zwams;
      if (zvol > 0.5 || cdice < 2.e-6) {
        const int ba = les_dry4wet(a, C, N(3, bc), &M(3, 0, bc), (int64_t)a.nb[3] * C.rs);
        N(0, ba) = N(0, ba) + N(3, bc);
        N(3, bc) = 0.;
        for (int s = 0; s < nwet; ++s) {
          M(0, s, ba) = M(0, s, ba) + M(3, s, bc);
          M(3, s, bc) = 0.;
        }
        M(0, iwa, ba) = M(0, iwa, ba) + M(3, irim, bc);
        M(3, irim, bc) = 0.;
        mod = true;
      }
    }
  }
  // aerosols below 0.1 nm dry diameter (:317-366); with the gas field
  // (lscndgas) their SO4, OC, NO and NH go to the gas phase as molecules
  for (int b = 0; b < a.nb[0]; ++b) {
    if (!(N(0, b) > kNlim)) continue;
    double zvol = 0.;
    for (int s = 0; s < ndry; ++s) zvol = zvol + M(0, s, b) / a.rholiq[s];
    zvol = zvol / N(0, b);
    if (zvol < kPi6 * 1.e-30) {
      if (a.gas)
        for (int s = 0; s < ndry; ++s) {
          const int g = a.gas_row[s];
          if (g >= 0) a.gas[(int64_t)g * n3 + x] = a.gas[(int64_t)g * n3 + x] + M(0, s, b) / a.mm[s] * kAvog;
        }
      for (int s = 0; s < nwet; ++s) M(0, s, b) = 0.;
      N(0, b) = 0.;
      mod = true;
    }
  }
  return mod;
}

// diagnostic tracers (:370-400) from the cell's (final) rows
__device__ __forceinline__ void les_sums(const LesArgs &a, const LesCell &C, int64_t x) {
  const int iwa = a.iwa, irim = a.irim;
  const int64_t n3 = a.n3;
  double sa = 0., sc = 0., sp = 0., sn = 0.;
  for (int b = a.in1a; b <= a.fn2b; ++b) sa = sa + C.M(a, 0, iwa, b);
  for (int b = a.ica_cur; b <= a.fcb_cur; ++b) sc = sc + C.M(a, 1, iwa, b);
  for (int b = 0; b < a.nb[2]; ++b) sp = sp + C.M(a, 2, iwa, b);
  for (int b = 0; b < a.nb[2]; ++b) sn = sn + C.N(a, 2, b);
  const double rc = sa + sc;
  double rtot = rc + sp + a.rp[x];
  a.diag[x] = rc;
  a.diag[n3 + x] = sp;
  a.diag[2 * n3 + x] = sn;
  if (a.level == 5) {
    double si = 0., sr = 0.;
    for (int b = 0; b < a.nb[3]; ++b) si = si + C.M(a, 3, iwa, b);
    for (int b = 0; b < a.nb[3]; ++b) sr = sr + C.M(a, 3, irim, b);
    rtot = rtot + si + sr;
    a.diag[4 * n3 + x] = si;
    a.diag[5 * n3 + x] = sr;
  }
  a.diag[3 * n3 + x] = rtot;
}

// Whether a wet bin (number n, masses m) can pass les_remove's evaporation test
// zdh2o < min(f * critical diameter, d) || water < kMassTH * n: the cubes of the
// diameters, which need no power, with a margin far above their rounding.
template <int MS>
__device__ __forceinline__ bool les_may_dry(const LesArgs &a, double n, const double (&m)[MS], double T, double f3,
                                            double d3) {
  double ns = 0., zvol = 0., wv = 0.;
#pragma unroll
  for (int s = 0; s < MS; ++s) {
    if (s < a.ndry) ns = ns + a.diss_mm[s] * m[s];
    if (s < a.nwet) zvol = zvol + m[s] * a.rrholiq[s];
    if (s == a.iwa) wv = m[s];
  }
  const double c2 = (4.5 * kRg / (kPi * kSurfw0)) * T * (ns / n);      // critical diameter squared
  return zvol < fmin(f3 * (c2 * ::sqrt(c2)), d3) * (kPi6 * (1. + 1.e-9)) * n || wv < kMassTH * n;
}

// Wavefronts of a column, each with an even share of its levels (of 4 and
// more: no share splits the three lowest or the three highest levels).
__host__ __device__ inline int les_chunks(int nzp) { return (nzp + 127) / 128; }

// two neighbouring levels of a row, on any 8-byte boundary
typedef double les2 __attribute__((ext_vector_type(2)));
typedef les2 les2u __attribute__((aligned(8)));

// Interior columns: two neighbouring levels per lane, a workgroup per chunk of
// a column and in it a wavefront per category, bin after bin, the next bin's
// rows (number, every mass species, their tendencies) loaded before the current
// one's are stored.  Per row: the tendency floored and added, the bottom and
// top levels from their two neighbours (read lane to lane, before the clamps),
// the clamp, the new value and a zero tendency stored, at an edge also to the
// periodic images; per bin the diagnostic sums in bin order and whether any
// removal test of les_remove can hold on the clamped values (its conditions as
// it meets them on values nothing has changed yet, with a margin where they are
// formed otherwise: false means that it would leave the cell as it is).  The
// first wavefront writes the sums and lists the cells.  MS: the mass rows of an
// ice bin, one more than a liquid bin has.
//
// HBM-bound: 32 B per element, each row touched once (1.42 GB at 64 x 64 x 120
// cells, 352 us; as passes for the update, the bottom and top rows and
// halos, the sums and the removals 212 + 48 + 132 + 65 us).  The loop body has
// no branch around a load or store (lanes past the chunk, and the last of an
// odd one, repeat its last two levels; edge columns take another copy of the
// loop): a wait then leaves the stores behind it in flight, which a count that
// differs by path would not.  Two levels per lane halve the changes of row, each
// of which is another page.  On small grids the chain of bins sets the time: by
// category it has 11 links, with one wavefront for all categories 26 (a call on
// 2 000 cells 82 us, with one wavefront 111, as passes 89; the large grid 389,
// 375 and 486).
template <int MS>
__global__ void __launch_bounds__(256) k_les_cells(LesArgs a) {
  __shared__ les2 sum[6][64];                 // rc's two parts, sp, sn, si, sr
  __shared__ int hit[64];                     // bit u: the lane's level u may be changed
  constexpr int iwa = MS - 2, irim = MS - 1, nwet = MS - 1, ndry = MS - 2;
  const int64_t n3 = a.n3;
  const int nx = a.nxp - 4, ny = a.nyp - 4, nch = les_chunks(a.nzp);
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), unit = (int)blockIdx.x;
  if (wv == 0) hit[lane] = 0;
  __syncthreads();
  // the rows of columns at the y edges first: they have the most images
  const int q = unit / nch, h = unit % nch, i = 2 + q % nx, j = 2 + (q / nx + ny - 2) % ny;
  const int k0 = (int)((int64_t)h * a.nzp / nch), nlev = (int)((int64_t)(h + 1) * a.nzp / nch) - k0;
  const int kk = 2 * lane < nlev - 2 ? 2 * lane : nlev - 2;      // this lane's two levels from k0
  const bool in0 = k0 + kk >= 1, in1 = k0 + kk + 1 <= a.nzp - 2; // interior (nzp >= 4: one end each)
  const bool first = h == 0, last = h == nch - 1;
  const bool bot = k0 + kk == 0, top = k0 + kk == a.nzp - 2;
  const int lt = (nlev + 1) / 2 - 1;          // the lane of the last two levels
  const int64_t x = ((int64_t)i + (int64_t)a.nxp * j) * a.nzp + k0 + kk;
  // the column's periodic images in the halo: bit 3 v + u for the one shifted by
  // u - 1 domains along x and v - 1 along y (several on the smallest grids)
  const int64_t sx = (int64_t)nx * a.nzp, sy = (int64_t)a.nxp * ny * a.nzp;
  const uint32_t ux = (i - nx >= 0 ? 1u : 0u) | 2u | (i + nx < a.nxp ? 4u : 0u);
  const uint32_t vy = (j - ny >= 0 ? 1u : 0u) | 2u | (j + ny < a.nyp ? 4u : 0u);
  const uint32_t im = ((vy & 1u) ? ux : 0u) | (ux & ~2u) << 3 | ((vy & 4u) ? ux << 6 : 0u);
  auto images = [&](auto &&f) {
    for (uint32_t left = im; left; left &= left - 1) {
      const int e = __builtin_ctz(left);
      f((e % 3 - 1) * sx + (e / 3 - 1) * sy);
    }
  };
  auto get = [](const double *p) -> les2 { return *(const les2u *)p; };
  auto set = [](double *p, les2 v) { *(les2u *)p = v; };
  const les2 zero = {0., 0.};
  const les2 rh = get(a.rh + x), rhi = a.level == 5 ? get(a.rhi + x) : zero, T = get(a.temp + x);
  const double rdt = a.dtlt;
  auto from = [](double v, int l) -> double {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l), __builtin_amdgcn_readlane(__double2loint(v), l));
  };
  // the new values of a row of which this lane holds p and t (:18-36, step.f90:470-489, util.f90:71-107), clamped
  auto fresh = [&](les2 pv, les2 tv) -> les2 {
    // the floor is rarely reached: its division only where it is close
    const les2 lo = (-1. + 1.e-8) * pv;
    const bool f0 = tv.x * rdt >= lo.x + fabs(lo.x) * 1.e-12, f1 = tv.y * rdt >= lo.y + fabs(lo.y) * 1.e-12;
    les2 tc = tv;
    if (__any(!f0 || !f1)) {
      tc.x = f0 ? tv.x : fmax(lo.x / rdt, tv.x);
      tc.y = f1 ? tv.y : fmax(lo.y / rdt, tv.y);
    }
    les2 v;
    v.x = in0 ? pv.x + tc.x * rdt : pv.x;
    v.y = in1 ? pv.y + tc.y * rdt : pv.y;
    les2 o = v;
    if (first) {
      const double s1 = from(v.y, 0), s2 = from(v.x, 1);
      if (bot) o.x = s1 - 0. * (s2 - s1);
    }
    if (last) {
      const double sm = from(v.x, lt), sm2 = nlev & 1 ? from(v.x, lt - 1) : from(v.y, lt - 1);
      if (top) o.y = sm + a.dzf2 * (sm - sm2);
    }
    o.x = o.x >= 0. ? o.x : fmax(0., o.x);
    o.y = o.y >= 0. ? o.y : fmax(0., o.y);
    return o;
  };
  bool any[2] = {false, false};
  les2 s1 = zero, s2 = zero;                  // the category's sums: water, and precipitation's number or ice's rime
  struct Bin { les2 n, nt, m[MS], mt[MS]; };
  // bin b of category c
  auto load = [&](int c, int b, Bin &B) {
    const int nb = a.nb[c], nsw = MS - 1 + (c == 3);
    const int64_t o = (int64_t)b * n3 + x;
    B.n = get(a.n_p[c] + o);
    B.nt = get(a.n_t[c] + o);
#pragma unroll
    for (int s = 0; s < MS; ++s) {
      // (a liquid bin has no rime row: that place repeats its water)
      const int64_t r = (int64_t)((s < nsw ? s : nsw - 1) * nb) * n3 + o;
      B.m[s] = get(a.m_p[c] + r);
      B.mt[s] = get(a.m_t[c] + r);
    }
  };
  auto run = [&](auto edge) {
    Bin B, F;
    auto category = [&](auto cc) {
      constexpr int c = decltype(cc)::value;
      const int nb = a.nb[c], nsw = MS - 1 + (c == 3);
      if (nb > 0) load(c, 0, B);
      for (int b = 0; b < nb; ++b) {
        load(c, b + 1 < nb ? b + 1 : b, F);
        const les2 n2 = fresh(B.n, B.nt);
        les2 m2[MS];
#pragma unroll
        for (int s = 0; s < MS; ++s) m2[s] = s < nsw ? fresh(B.m[s], B.mt[s]) : zero;
        auto put = [&](int64_t y) {
          const int64_t o = (int64_t)b * n3 + y;
          set(a.n_p[c] + o, n2);
          set(a.n_t[c] + o, zero);
#pragma unroll
          for (int s = 0; s < MS; ++s)
            if (s < nsw) {
              set(a.m_p[c] + ((int64_t)(s * nb) * n3 + o), m2[s]);
              set(a.m_t[c] + ((int64_t)(s * nb) * n3 + o), zero);
            }
        };
        put(x);
        if constexpr (decltype(edge)::value) images([&](int64_t o) { put(x + o); });
        les2 wv = zero, rv = zero;            // water and rime masses (no dynamic register index)
#pragma unroll
        for (int s = 0; s < MS; ++s) {
          if (s == iwa) wv = m2[s];
          if (s == irim) rv = m2[s];
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const double n = n2[u];
          double m[MS];
#pragma unroll
          for (int s = 0; s < MS; ++s) m[s] = m2[s][u];
          if constexpr (c < 2) {
            double sm = 0.;
#pragma unroll
            for (int s = 0; s < MS; ++s)
              if (s < nwet) sm = sm + m[s];
            any[u] |= n > 0. && sm <= 0.;
          }
          if constexpr (c == 0) {
            double zvol = 0.;
#pragma unroll
            for (int s = 0; s < MS; ++s)
              if (s < ndry) zvol = zvol + m[s] * a.rrholiq[s];
            any[u] |= n > kNlim && zvol < (kPi6 * 1.e-30 * (1. + 1.e-9)) * n;
          } else if constexpr (c == 1) {
            if (b >= a.ica_cur && b <= a.fcb_cur && rh[u] < 0.999 && n > kNlim && wv[u] < 1.e-5)
              any[u] |= les_may_dry<MS>(a, n, m, T[u], 0.343, 2.197e-15);
          } else if constexpr (c == 2) {
            any[u] |= n > 0. && wv[u] <= 0.;
            if (rh[u] < 0.999 && n > kPrlim && wv[u] < 1.e-6) any[u] |= les_may_dry<MS>(a, n, m, T[u], 0.008, 1.e-15);
          } else {
            const double mt = wv[u] + rv[u];
            any[u] |= n > 0. && mt < kMassTH;
            any[u] |= n > kPrlim && rhi[u] < 0.999 && mt < 1.e-15;
          }
        }
        if constexpr (c == 0) {
          if (b >= a.in1a && b <= a.fn2b) s1 = s1 + wv;
        } else if constexpr (c == 1) {
          if (b >= a.ica_cur && b <= a.fcb_cur) s1 = s1 + wv;
        } else {
          s1 = s1 + wv;
          s2 = s2 + (c == 2 ? n2 : rv);
        }
        B = F;
      }
    };
    if (wv == 0) category(std::integral_constant<int, 0>{});
    else if (wv == 1) category(std::integral_constant<int, 1>{});
    else if (wv == 2) category(std::integral_constant<int, 2>{});
    else category(std::integral_constant<int, 3>{});
  };
  if (im) run(std::true_type{});
  else run(std::false_type{});
  if (wv) {
    sum[wv < 2 ? 1 : 2 * wv - 2][lane] = s1;
    if (wv >= 2) sum[2 * wv - 1][lane] = s2;
    if (any[0] || any[1]) atomicOr(hit + lane, (any[0] ? 1 : 0) | (any[1] ? 2 : 0));
  }
  __syncthreads();
  if (wv) return;
  any[0] |= hit[lane] & 1;
  any[1] |= (hit[lane] >> 1) & 1;
  // diagnostic tracers (:370-400), as les_sums forms them
  {
    const les2 rc = s1 + sum[1][lane], sp = sum[2][lane], sn = sum[3][lane];
    auto sums = [&](int64_t y) {
      les2 rtot = rc + sp + get(a.rp + y);
      set(a.diag + y, rc);
      set(a.diag + n3 + y, sp);
      set(a.diag + 2 * n3 + y, sn);
      if (a.level == 5) {
        const les2 si = sum[4][lane], sr = sum[5][lane];
        rtot = rtot + si + sr;
        set(a.diag + 4 * n3 + y, si);
        set(a.diag + 5 * n3 + y, sr);
      }
      set(a.diag + 3 * n3 + y, rtot);
    };
    sums(x);
    images([&](int64_t o) { sums(x + o); });
  }
  // append the cells to the list of cells the removals visit (one atomic
  // per wavefront; the list order does not matter, cells are independent)
  const bool own = 2 * lane < nlev;           // the lanes past it repeat levels, as does the first of a last odd one
  const bool fl0 = own && kk == 2 * lane && any[0], fl1 = own && any[1];
  const unsigned long long m0 = __ballot(fl0), m1 = __ballot(fl1);
  if (m0 | m1) {
    const int n0 = (int)__popcll(m0);
    int base = 0;
    if (lane == 0) base = atomicAdd(a.count, n0 + (int)__popcll(m1));
    base = __builtin_amdgcn_readfirstlane(base);
    const unsigned long long below = (1ull << lane) - 1ull;
    if (fl0) a.list[base + (int)__popcll(m0 & below)] = (int32_t)x;
    if (fl1) a.list[base + n0 + (int)__popcll(m1 & below)] = (int32_t)(x + 1);
  }
}

// Removals on the listed cells, on the LES arrays (layouts whose
// rows do not fit kLesLdsRows); their sums are formed again from the final
// values
__global__ void __launch_bounds__(256) k_les_remove(LesArgs a) {
  const int ncat = a.level == 5 ? 4 : 3;
  const int cnt = *a.count;
  for (int idx = blockIdx.x * blockDim.x + threadIdx.x; idx < cnt; idx += gridDim.x * blockDim.x) {
    const int64_t x = a.list[idx];
    LesCell G;
    G.rs = a.n3;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      G.n[c] = c < ncat ? a.n_p[c] + x : nullptr;
      G.m[c] = c < ncat ? a.m_p[c] + x : nullptr;
    }
    les_remove(a, G, x, a.temp[x], a.rh[x], a.level == 5 ? a.rhi[x] : 0.);
    les_sums(a, G, x);
  }
}

// Removals on the listed cells with each cell's rows staged in LDS
// (one lane per listed cell, its own column lds[row * kLesCells + lane]):
// the sequence of dependent tests runs at LDS latency.  A cell whose
// removals changed something writes all its rows back and its sums again.
__global__ void __launch_bounds__(kLesCells) k_les_remove_lds(LesArgs a) {
  extern __shared__ double lds[];
  const int ncat = a.level == 5 ? 4 : 3;
  const int t = threadIdx.x, cnt = *a.count;
  const int64_t n3 = a.n3;
  for (int idx = blockIdx.x * kLesCells + t; idx - t < cnt; idx += gridDim.x * kLesCells) {
    if (idx >= cnt) continue;                 // lanes work on their own LDS column: no barrier
    const int64_t x = a.list[idx];
    LesCell G, S;
    G.rs = n3;
    S.rs = kLesCells;
    int row = 0;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      G.n[c] = c < ncat ? a.n_p[c] + x : nullptr;
      G.m[c] = c < ncat ? a.m_p[c] + x : nullptr;
      S.n[c] = lds + (int64_t)row * kLesCells + t;
      row += c < ncat ? a.nb[c] : 0;
      S.m[c] = lds + (int64_t)row * kLesCells + t;
      row += c < ncat ? a.nb[c] * a.nsw[c] : 0;
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        if (c >= ncat) continue;
        const double *g = q ? G.m[c] : G.n[c];
        double *l = q ? S.m[c] : S.n[c];
        const int nr = q ? a.nb[c] * a.nsw[c] : a.nb[c];
        for (int r0 = 0; r0 < nr; r0 += 16) {
          double v[16];
#pragma unroll
          for (int u = 0; u < 16; ++u) v[u] = r0 + u < nr ? g[(int64_t)(r0 + u) * n3] : 0.;
#pragma unroll
          for (int u = 0; u < 16; ++u)
            if (r0 + u < nr) l[(r0 + u) * kLesCells] = v[u];
        }
      }
    if (les_remove(a, S, x, a.temp[x], a.rh[x], a.level == 5 ? a.rhi[x] : 0.)) {
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          if (c >= ncat) continue;
          double *g = q ? G.m[c] : G.n[c];
          const double *l = q ? S.m[c] : S.n[c];
          const int nr = q ? a.nb[c] * a.nsw[c] : a.nb[c];
          for (int r = 0; r < nr; ++r) g[(int64_t)r * n3] = l[r * kLesCells];
        }
      les_sums(a, S, x);
    }
  }
}

unsigned grid_for(int64_t n, int block) {
  const int64_t g = (n + block - 1) / block;
  return (unsigned)(g < 65536 ? (g > 0 ? g : 1) : 65536);
}

}  // namespace

int launch_les_update(const LesArgs &a, hipStream_t s) {
  const int ncat = a.level == 5 ? 4 : 3;
  int nrow = 0;
  for (int c = 0; c < ncat; ++c) nrow += a.nb[c] * (1 + a.nsw[c]);
  const int64_t nind = a.indef && a.level == 5 ? (int64_t)a.nindef * a.n3 : 0;
  hipLaunchKernelGGL(k_les_start, dim3(grid_for(nind, 256)), dim3(256), 0, s, a, nind);
  // what k_les_cells takes for granted of a layout: one or two dry species, water, rime
  const int ms = a.nsw[0] + 1;
  if (ms < 3 || ms > 4 || a.nsw[1] != ms - 1 || a.nsw[2] != ms - 1 || (ncat == 4 && a.nsw[3] != ms) ||
      a.nwet != ms - 1 || a.ndry != ms - 2 || a.iwa != ms - 2 || (ncat == 4 && a.irim != ms - 1))
    return (int)hipErrorInvalidValue;
  const int64_t units = (int64_t)(a.nxp - 4) * (a.nyp - 4) * les_chunks(a.nzp);
  const dim3 gc((unsigned)units), tc(64 * ncat);
  if (ms == 3) hipLaunchKernelGGL(k_les_cells<3>, gc, tc, 0, s, a);
  else hipLaunchKernelGGL(k_les_cells<4>, gc, tc, 0, s, a);
  if (nrow <= kLesLdsRows) {
    const int64_t g = (a.n3 + kLesCells - 1) / kLesCells;
    hipLaunchKernelGGL(k_les_remove_lds, dim3((unsigned)(g < 4096 ? g : 4096)), dim3(kLesCells),
                       (size_t)nrow * kLesCells * sizeof(double), s, a);
  } else {
    hipLaunchKernelGGL(k_les_remove, dim3(grid_for(a.n3, 256)), dim3(256), 0, s, a);
  }
  return (int)hipGetLastError();
}

}  // namespace salsa
