// salsa_lanes.hip -- the coagulation + condensation step with one lane per
// grid cell.
//
// The step kernel of salsa_kernels.hip gives every cell 8 to 64 lanes; the
// lanes of a wavefront then hold different bins, so nearly every branch of the
// physics is taken by some lane, every target of the sweep ends in cross-lane
// sums, and the cell records cost a gather and a scatter pass.  Here a
// wavefront's 64 lanes are 64 cells working on the same bin, pair or sweep
// entry: control flow and table reads are uniform (scalar), the LES rows are
// read and written coalesced where they lie (k fastest), and the wavefronts of
// a workgroup share the bins, pairs and entries of the same 64 cells.
//
//   k_lanes_start  counts to zero, and the table of the call's rows
//   k_lanes_class  cost class of every interior cell, and two lists of cell
//                  ids: without and with active hydrometeors
//   k_lanes_pairs  particle terms of every bin (LDS), then the collision
//                  kernel of every pair whose bins are active
//   k_lanes_sweep  the sequential semi-implicit sweep on the state in LDS,
//                  equilibration, condensation substeps, tendencies or new state
//
// The last two run per list, 64 neighbouring entries to a workgroup, in chunks
// that keep the kernels within a bounded work space.  The counts stay on the
// device: a grid covers the workgroups that every cell could need, and those
// past the list's end return at once.  Nothing waits for the device.
//
// Measured with the 120 x 64 x 64 cloud deck (491 520 cells, FP32-mixed): the
// step 2.95 ms with 8 to 16 lanes per cell, 1.32 ms here; classes 0.04,
// pairs 0.13 + 0.26 and sweep 0.50 + 0.38 ms for the cells without + with
// hydrometeors.  100 x 64 x 64 mixed-phase clouds with dust 10.5 and 4.9 ms.
//
// Follows the same reference lines as salsa_kernels.hip (mo_salsa_driver.f90:
// 230-388, mo_salsa_coagulation_kernels.f90:24-420, mo_salsa_coagulation_
// processes.f90:24-1611, mo_salsa_dynamics.f90:92-202, 276-342, 691-1157,
// mo_salsa_properties.f90:73-380).
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <cmath>
#include <cstring>

#include "salsa_internal.h"
#include "salsa_physics.h"

namespace salsa {

int lanes_program(const DevLayout &L, int kt, uint32_t *prog);

namespace {

// The sweep program: per target and wavefront 32 words, one per lane of a
// register, taken from there by lane number (the loop over the targets then
// has no scalar loads, whose waits would be shared with those on LDS).
constexpr int kEnt = 8;                       // words 0..: entries: pair << 15 | bin << 9 | roles
constexpr int kProgT = 8, kProgK = 9, kProgN = 10, kProgS = 12, kProgQ = 13;   // target | flags << 8; pair of its
                                              // self term; nlim (two words); cloud-cloud pair of its self-
                                              // collection, -1 without; parity of the first quad (below)
constexpr int kProgF = 16;                    // words 16..: precipitation-formation entries:
                                              // pair | bin << 16 | own series << 30 | used << 31
constexpr int kProg = 32;
__host__ __device__ constexpr int prog_pf(int VL) { return VL >= 16 ? 12 : 8; }   // at most 8, and 3 to align them
enum : uint32_t {
  SR_SINK = 1u, SR_SRC = 2u, SR_SINK_EAGG = 4u, SR_SRC_EAGG = 8u, SR_PC_WA = 16u, SR_PC_RI = 32u, SR_PF = 64u,
  SR_FIX_OWN = 128u, SR_FIX_OTH = 256u, SR_SPECIAL = 511u & ~3u
};

constexpr int kL = 64;                        // cells per workgroup: one per lane

__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }

__device__ __forceinline__ int64_t lanes_index(const StepArgs &a, int cell) {
  const int k = cell % a.nz, r = cell / a.nz;
  const int i = r % a.nx, j = r / a.nx;
  return (int64_t)(k + a.hz) + (int64_t)a.nzp * ((int64_t)(i + a.hxy) + (int64_t)a.nxp * (j + a.hxy));
}

// Rows that a table names are global memory: plain (not flat) loads and stores.
typedef const __attribute__((address_space(1))) double *grow_in;
typedef __attribute__((address_space(1))) double *grow_out;
__device__ __forceinline__ double row_load(const double *p, int64_t x) { return ((grow_in)p)[x]; }
__device__ __forceinline__ void row_store(double *p, int64_t x, double v) { ((grow_out)p)[x] = v; }

// Block g of a launch: its first entry in the list of the cells with (hyd) or
// without hydrometeors, and the cells it holds.
struct Block { int first, n; };
__device__ __forceinline__ int lanes_count(const LanesArgs &w, bool hyd) {
  return hyd ? w.counts[2] : w.counts[0] + w.counts[1];
}
__device__ __forceinline__ Block lanes_block(const LanesArgs &w, bool hyd, int g) {
  const int left = lanes_count(w, hyd) - g * kL;
  return Block{g * kL, left < kL ? left : kL};
}

// ---------------------------------------------------------------------------
// classes
// ---------------------------------------------------------------------------
constexpr int kClassThreads = 1024;

// Start of a step: counts and fault word to zero, and the rows of the call's
// fields in the order of the state, NC = 1 + volumes per bin (a liquid bin has
// no rime row at level 5: it reads its number row with an infinite density).
__global__ void __launch_bounds__(256) k_lanes_start(const DevLayout *__restrict__ Dp, StepArgs a, LanesArgs w, int NC) {
  const DevLayout &D = *Dp;
  if (threadIdx.x < 4) w.counts[threadIdx.x] = 0;
  if (threadIdx.x == 4) *a.fault_any = 0;
  for (int r = threadIdx.x; r < D.nt * NC; r += 256) {
    const int b = r / NC, q = r % NC, c = D.cat_of[b], nr = 1 + (c < 3 ? D.nwet : D.nspec);
    const int64_t on = a.n3 * D.loc_of[b], om = a.n3 * ((int64_t)(q - 1) * D.nb[c] + D.loc_of[b]);
    LaneRow row;
    row.kind = (q >= nr ? LR_NONE : 0) | (q == 0 ? LR_NUMBER : 0) |
               (q == 1 + D.iwa || (c == 3 && q == 1 + D.irim) ? LR_WATER : 0);
    if (q == 0 || q >= nr) {
      row.in = a.n_p[c] + on;
      row.out = (a.inplace ? a.n_o[c] : a.n_t[c]) + on;
      row.rho = q == 0 ? 1. : HUGE_VAL;
    } else {
      row.in = a.m_p[c] + om;
      row.out = (a.inplace ? a.m_o[c] : a.m_t[c]) + om;
      row.rho = c < 3 ? D.rholiq[q - 1] : (q - 1 == D.irim ? kRhori : D.rhoice[q - 1]);
    }
    w.rows[r] = row;
  }
}

// One thread per interior cell: the class as k_gather forms it, counted; the
// ids of a block's cells go to the list of the cells without hydrometeors
// (classes 0 and 1 together, so that neighbouring cells stay neighbours: their
// rows are then read in whole lines) or with them, in cell order, at a place that the block reserves with one atomic
// per list (the order of the blocks in a list has no effect on a cell's result).
__global__ void __launch_bounds__(kClassThreads) k_lanes_class(const DevLayout *__restrict__ Dp, StepArgs a, LanesArgs w) {
  __shared__ int32_t wc[3][kClassThreads / 64], base[2];
  const DevLayout &D = *Dp;
  const int lane = threadIdx.x & 63, wv = wave_id();
  const int64_t cell = (int64_t)blockIdx.x * kClassThreads + threadIdx.x;
  int cl = -1;
  if (cell < a.ncells) {
    const int64_t x = lanes_index(a, (int)cell);
    const double dn = a.dn[x], rs = a.rsl[x];
    double rv = a.rv_p[x];
    bool hyd = false;
    for (int c = 1; c < D.ncat; ++c) {
      const double *p = a.n_p[c] + x;
      for (int b = 0; b < D.nb[c]; ++b) hyd |= !(p[a.n3 * b] * dn < D.nlim[D.off[c] + b]);
    }
    if (!a.lsfreeRH) rv = fmin(rv, rs * a.rhlim);
    cl = hyd ? 2 : (rv / rs > 0.98 ? 1 : 0);
  }
  const uint64_t mh = __ballot(cl == 2), ma = __ballot(cl == 0 || cl == 1), m1 = __ballot(cl == 1);
  if (lane == 0) {
    wc[0][wv] = __popcll(ma);
    wc[1][wv] = __popcll(mh);
    wc[2][wv] = __popcll(m1);
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    const int k = threadIdx.x;
    int s = 0;
    for (int v = 0; v < kClassThreads / 64; ++v) {
      const int n = wc[k][v];
      wc[k][v] = s;
      s += n;
    }
    if (k == 2) {
      if (s) { atomicAdd(w.counts + 1, s); atomicAdd(w.counts, -s); }   // counts: class 0, 1, 2
    } else {
      if (s && k == 0) atomicAdd(w.counts, s);
      base[k] = s ? atomicAdd(w.counts + (k == 0 ? 3 : 2), s) : 0;      // 3: cells in the first list
    }
  }
  __syncthreads();
  const uint64_t below = (1ull << lane) - 1ull;
  if (cl == 2) w.lists[w.ncells + base[1] + wc[1][wv] + __popcll(mh & below)] = (int32_t)cell;
  else if (cl >= 0) w.lists[base[0] + wc[0][wv] + __popcll(ma & below)] = (int32_t)cell;
}

// ---------------------------------------------------------------------------
// particle terms and pairs
// ---------------------------------------------------------------------------
// LDS of k_lanes_pairs for nb bins of C cells: diameters, the terms of every
// bin and of its self-offset twin, the residuals of the FP32 fall speeds
// (mixed path), the bins' activity masks.
__host__ __device__ inline int pairs_lds(int nb, int kt, int C) {
  return C * (8 * nb + 2 * nb * 4 * kt + (kt == 4 ? 2 * nb * 4 : 0)) + 8 * nb;
}

template <class KT, int NV, int W, int C, bool HYD>
__global__ void __launch_bounds__(64 * W, 3) k_lanes_pairs(const DevLayout *__restrict__ Dp, StepArgs a, LanesArgs w) {
  extern __shared__ __align__(16) char smem[];
  const DevLayout &D = *Dp;
  constexpr int R = 64 / C;                   // bins (pairs) that a wavefront works on at a time
  constexpr int BC = kL / C;                  // workgroup blocks per block of 64 slots
  const int lane = (threadIdx.x & 63) % C, row = (threadIdx.x & 63) / C;
  const int wk = wave_id() * R + row;         // this lane's worker of the W * R
  const int nb = HYD ? D.nt : D.nb[0], np = HYD ? D.npair : D.npair_aa;
  double *sDW = reinterpret_cast<double *>(smem);                            // [nb][C]
  PT4<KT> *sPR = reinterpret_cast<PT4<KT> *>(sDW + nb * C);                  // [2][nb][C]
  KT *sVL = reinterpret_cast<KT *>(sPR + 2 * nb * C);                        // [2][nb][C], mixed path
  uint64_t *sAct = reinterpret_cast<uint64_t *>(sizeof(KT) == 4 ? sVL + 2 * nb * C : sVL);
  const int gend = (lanes_count(w, HYD) + kL - 1) / kL;
  {
    const int g = w.g0 + (int)blockIdx.x / BC, c0 = ((int)blockIdx.x % BC) * C;
    if (g >= gend) return;
    const Block B = lanes_block(w, HYD, g);
    const bool live = c0 + lane < B.n;
    const int icell = w.lists[(HYD ? w.ncells : 0) + B.first + (live ? c0 + lane : 0)];
    const int64_t x = lanes_index(a, icell);
    const int blk = g - w.g0, sl = c0 + lane;   // block of the chunk, place in it
    const double T = a.temp[x], P = a.press[x], dn = a.dn[x];
    const CellC cc = cell_consts(D, T, P);
    for (int b = wk; b < nb; b += W * R) {
      const LaneRow *r = w.rows + b * (1 + NV);
      double v[1 + NV], vs = 0., vwa = 0., vri = 0., sdry = 0.;
#pragma unroll
      for (int q = 0; q <= NV; ++q) v[q] = row_load(r[q].in, x);
      const double n = v[0] * dn;
#pragma unroll
      for (int q = 1; q <= NV; ++q) {
        v[q] = v[q] * dn / r[q].rho;
        vs += v[q];
        if (q == 1 + D.iwa) vwa = v[q];
        if (q == D.nspec) vri = v[q];
        if (q < D.nspec) sdry += v[q] * kRhoic;
      }
      double dw = n > D.nlim[b] ? cbrt_fast(vs / n / kPi6) : D.dmid[b];
      dw = fmin(dw, D.dlim[b]);
      sDW[b * C + lane] = dw;
      if (b < D.nb[0]) w.dwa[((int64_t)blk * D.nb[0] + b) * kL + sl] = dw;
      uint64_t act = __ballot(live && !(n < D.nlim[b]));
      if (C < 64) act = (act >> (row * C)) & ((1ull << (C & 63)) - 1ull);
      if (lane == 0) sAct[b] = act;
      if (!act) continue;
      PT4<KT> p0, p1;
      if (HYD && D.phase[b] == 4) {           // ice (updateRhomean, getShapeCoefficients)
        double rho = kRhoic;
        if (n > D.nlim[b]) {
          const double mp = kRhoic * vwa, mr = kRhori * vri;
          rho = fmin((mp * kRhoic + mr * kRhori) / fmax(mp + mr, 7.e-25), kRhoic);
        }
        const Shape sh = shape_coeffs(D, sdry, vri * kRhori, n);
        const double mass = rho * kPi6 * cubed(dw);
        const PTerms q0 = particle_terms(cc, dw, mass, rho, 4, dw, sh);
        const PTerms q1 = particle_terms(cc, 1.1 * dw, 1.33 * mass, rho, 4, dw, sh);
        p0 = PT4<KT>{(KT)q0.D, (KT)q0.c, (KT)q0.w, (KT)q0.v};
        p1 = PT4<KT>{(KT)q1.D, (KT)q1.c, (KT)q1.w, (KT)q1.v};
        if (sizeof(KT) == 4) {
          sVL[b * C + lane] = (KT)(q0.v - (double)(KT)q0.v);
          sVL[(nb + b) * C + lane] = (KT)(q1.v - (double)(KT)q1.v);
        }
      } else {
        const double rho = kRhowa, mass = rho * kPi6 * cubed(dw);
        if (sizeof(KT) == 4) {
          const PTermsF q0 = particle_terms_liquid_f(cc, dw, mass, rho);
          const PTermsF q1 = particle_terms_liquid_f(cc, 1.1 * dw, 1.33 * mass, rho);
          p0 = PT4<KT>{(KT)q0.D, (KT)q0.c, (KT)q0.w, (KT)q0.v};
          p1 = PT4<KT>{(KT)q1.D, (KT)q1.c, (KT)q1.w, (KT)q1.v};
          sVL[b * C + lane] = (KT)(q0.vd - (double)q0.v);
          sVL[(nb + b) * C + lane] = (KT)(q1.vd - (double)q1.v);
        } else {
          const Shape sh{0., 0., 0., 0.};
          const PTerms q0 = particle_terms(cc, dw, mass, rho, D.phase[b], dw, sh);
          const PTerms q1 = particle_terms(cc, 1.1 * dw, 1.33 * mass, rho, D.phase[b], dw, sh);
          p0 = PT4<KT>{(KT)q0.D, (KT)q0.c, (KT)q0.w, (KT)q0.v};
          p1 = PT4<KT>{(KT)q1.D, (KT)q1.c, (KT)q1.w, (KT)q1.v};
        }
      }
      sPR[b * C + lane] = p0;
      sPR[(nb + b) * C + lane] = p1;
    }
    __syncthreads();
    const KT vkin = (KT)cc.vkin, cshear = (KT)cc.cshear, cinert = (KT)cc.cinert, cfac = (KT)D.charge_factor;
    KT *K = reinterpret_cast<KT *>(w.K) + (int64_t)blk * (np + 1) * kL + sl;           // [pair][64], then a row of zeros
    if (wk == 0) K[np * kL] = KT(0.);
    for (int p = wk; p < np; p += W * R) {
      const uint32_t pw = D.pw[p];
      const int b1 = pw & 255u, b2 = (pw >> 8) & 255u, tw = (pw >> 16) & 1u;
      const uint64_t m = sAct[b1] & sAct[b2];
      KT k = KT(0.);
      uint32_t pfb = 0;
      const bool pf = HYD && p >= D.pf0 && p < D.pf0 + D.ncc;
      if ((m >> lane) & 1ull) {
        // particle 1 is the twin of particle 2 when the bins' dmid agree within 1%
        const double dB = sDW[b2 * C + lane];
        const double dA = tw ? 1.1 * dB : sDW[b1 * C + lane];
        const int ia = (tw ? nb + b2 : b1) * C + lane, ib = b2 * C + lane;
        const PT4<KT> A = sPR[ia], Bq = sPR[ib];
        KT vAl = KT(0.), vBl = KT(0.);
        if (sizeof(KT) == 4) { vAl = sVL[ia]; vBl = sVL[ib]; }
        k = pair_coef<KT>((KT)dA, A.D, A.c, A.w, A.v, (KT)dB, Bq.D, Bq.c, Bq.w, Bq.v, dA >= dB, vkin, cshear, cinert,
                          vAl, vBl);
        k = k * cfac;                         // charge enhancement (kernels.f90:411-416)
        if (pf) {
          // precip bin reached by coalescence (accumulatePrecipFormation, processes.f90:1461-1467)
          const double dnew = cbrt_fast(cubed(sDW[b1 * C + lane]) + cubed(dB));
          int cnt = 0;
          for (int q = 0; q < D.nb[2]; ++q) cnt += dnew > D.precpbins[q];
          pfb = (uint32_t)cnt;
        }
      }
      K[p * kL] = k;
      if (pf) w.pf[((int64_t)blk * D.ncc + (p - D.pf0)) * kL + sl] = (uint8_t)pfb;
    }
  }
}

// ---------------------------------------------------------------------------
// equilibration of one aerosol bin over the lanes (mo_salsa_properties.f90:
// 165-378): the Kelvin fixed point of lanes with on set.  Returns the water
// volume; zke in and out (carried over the 1a bins).
// ---------------------------------------------------------------------------
template <bool REG2>
__device__ __forceinline__ double equil_bin(double n, double zcore, double c1, double c2, double c5, double T,
                                            double zr, double zdwet, double &zke, bool on, uint32_t &flags) {
  const double tol = REG2 ? 1.e-12 : 1.e-2;
  const double kel = 2. * kSurfw0 * kMvwa, kt = kBoltz * T, core = div_nr(zcore, kPi6);
  double zdold = 1., zlwc = 0.;
  int count = 0;
  bool go = on && fabs(zdwet / zdold - 1.) > tol;
  while (__any(go)) {
    if (go) {
      zdold = fmax(zdwet, 1.e-20);
      const double aw = div_nr(zr, zke);
      const double aw2 = aw * aw;
      const double bm1 = 1.1065495e+2 - 3.6759197e+2 * aw + 5.0462934e+2 * aw2
                         - 3.1543839e+2 * (aw2 * aw) + 6.770824e+1 * (aw2 * aw2);
      const double bm2 = rcp_nr(aw * kMwa) - 1. / kMwa;
      double l = div_nr(c1, bm1) + div_nr(c2, bm2);
      if (REG2) {
        const double bm5 = 5.875248e+1 - 1.8781997e+2 * aw + 2.7211377e+2 * aw2
                           - 1.8458287e+2 * (aw2 * aw) + 4.153689e+1 * (aw2 * aw2);
        l = l + div_nr(c5, bm5);
      }
      zlwc = l;
      zdwet = cbrt_fast(div_nr(div_nr(div_nr(zlwc, n), kRhowa), kPi6) + core);
      zke = ::exp(div_nr(kel, kt * zdwet));
      go = fabs(zdwet / zdold - 1.) > tol;
      if (++count > 100) { flags |= SALSA_CELL_NOCONV; go = false; }
    }
  }
  return zlwc;
}

// ---------------------------------------------------------------------------
// sweep, condensation, output
// ---------------------------------------------------------------------------
// Sums over a cell's collectors are taken in VL partial sums, entry e in
// partial e % VL, which are then added as a balanced tree; a wavefront holds
// VL / W neighbouring partials and adds them before the W wavefronts' sums
// meet.  With VL = 16 or 32 that is the order of the general kernel's sums at 16
// or 32 lanes per cell: 94 % of the cells of a level-5 step with ice everywhere
// then have its bits (FP64 with dust 32 %), the others differ by rounding in
// products that the compiler contracts otherwise.
template <int W>
__device__ __forceinline__ double tree_sum(const double *p, int stride) {
  static_assert(W == 4 || W == 8, "wavefronts per workgroup");
  double q[W / 4];
#pragma unroll
  for (int v = 0; v < W / 4; ++v)
    q[v] = (p[(4 * v) * stride] + p[(4 * v + 1) * stride]) + (p[(4 * v + 2) * stride] + p[(4 * v + 3) * stride]);
  if constexpr (W == 4) return q[0];
  else return q[0] + q[1];
}
// the same over the V values of each of a cell's VL / V lanes
template <int VL, int V>
__device__ __forceinline__ double tree_lanes(const double (&x)[V]) {
  static_assert(V == 1 || V == 2 || V == 4, "partials per lane");
  if constexpr (V == 1) return cell_sum<VL>(x[0]);
  else if constexpr (V == 2) return cell_sum<VL / 2>(x[0] + x[1]);
  else return cell_sum<VL / 4>((x[0] + x[1]) + (x[2] + x[3]));
}

// LDS of k_lanes_sweep for nb bins of NV volumes, nice of them ice, and ncc
// cloud-cloud pairs: the state, the wavefronts' sums (sink, sources, two
// fix_coag sums), rime fractions, vapour, flags, precipitation-formation bins.
__host__ __device__ constexpr int sweep_parts(int NV) { return NV + 3; }
__host__ __device__ inline int sweep_lds(int nb, int NV, int W, int ncc, int nice) {
  return kL * (8 * nb * (1 + NV) + 8 * W * sweep_parts(NV) + 8 * nice + 8 + 4 + 1 + ncc);
}

// wavefronts per SIMD that the LDS of a shape leaves room for
__host__ __device__ constexpr int sweep_waves(bool hyd, int NV) { return !hyd ? 4 : NV == 2 ? 3 : 2; }

template <class KT, int NV, bool L5, int W, int VL, int NR, bool HYD>
__global__ void __launch_bounds__(64 * W, sweep_waves(HYD, NV)) k_lanes_sweep(const DevLayout *__restrict__ Dp, StepArgs a,
                                                                        LanesArgs w) {
  extern __shared__ __align__(16) char smem[];
  const DevLayout &D = *Dp;
  constexpr int A = VL / W;                   // partial sums of a wavefront
  constexpr int V = VL / W, NQ = V * NR;      // substeps, W lanes per cell: partial sums and bins per lane
  constexpr int NC = 1 + NV;                  // components of a bin's state: number, volumes
  constexpr int NP = sweep_parts(NV), NF = HYD ? prog_pf(VL) : 1;
  constexpr int nwet = L5 ? NV - 1 : NV, ndry = nwet - 1, iwa = nwet - 1, irim = NV - 1;
  const int lane = threadIdx.x & 63, wv = wave_id();
  const int nb = HYD ? D.nt : D.nb[0], ncc = HYD ? D.ncc : 0;
  double *sS = reinterpret_cast<double *>(smem);       // [nb][NC][64]
  double *sP = sS + nb * NC * kL;                      // [W][NP][64]
  double *sRV = sP + W * NP * kL;                      // [64]
  double *sRF = sRV + kL;                              // [ice bins][64]
  int *sF = reinterpret_cast<int *>(sRF + (HYD && L5 ? D.nb[3] : 0) * kL);   // [64]
  uint8_t *sL = reinterpret_cast<uint8_t *>(sF + kL);  // [64] cells of a stage, side by side
  uint8_t *sPF = sL + kL;                              // [ncc][64]
  const double dt = a.dt;
#define SC(b, q) sS[((b) * NC + (q)) * kL + lane]      // component q of bin b: 0 number, 1 + s species s
  const int g = w.g0 + (int)blockIdx.x;
  if (g * kL >= lanes_count(w, HYD)) return;
  const Block B = lanes_block(w, HYD, g);
  const int32_t *ids = w.lists + (HYD ? w.ncells : 0) + B.first;
  const bool live = lane < B.n;
  const int icell = ids[live ? lane : 0];
  const int64_t x = lanes_index(a, icell);
  const int64_t blk = g - w.g0;               // block of the chunk
  const double T = a.temp[x], P = a.press[x], dn = a.dn[x], rs = a.rsl[x];
  double rv0 = a.rv_p[x];
  if (!a.lsfreeRH) rv0 = fmin(rv0, rs * a.rhlim);     // mo_salsa_driver.f90:193-197
  // kernels of the block's cells: [pair][64], the last row zeros
  const char *K = reinterpret_cast<const char *>(w.K) + blk * ((HYD ? D.npair : D.npair_aa) + 1) * (kL * sizeof(KT));
  const uint32_t kl = lane * sizeof(KT);
  auto kernel_at = [&](uint32_t off) -> KT { return *reinterpret_cast<const KT *>(K + (off + kl)); };
  uint32_t flags = 0;

  // ---- pack ----
  constexpr int RB = 8;                       // rows that a wavefront loads together
  const int nrow = nb * NC;
  for (int r0 = wv * RB; r0 < nrow; r0 += W * RB) {
    double v[RB];
#pragma unroll
    for (int u = 0; u < RB; ++u) v[u] = row_load(w.rows[r0 + u < nrow ? r0 + u : 0].in, x);
#pragma unroll
    for (int u = 0; u < RB; ++u)
      if (r0 + u < nrow) sS[(r0 + u) * kL + lane] = live ? v[u] * dn / w.rows[r0 + u].rho : 0.;
  }
  for (int p = wv; p < ncc; p += W) sPF[p * kL + lane] = w.pf[(blk * ncc + p) * kL + lane];
  // hydrometeor bins below their limits keep their contents; their water
  // counts towards the cell's total, and a block without any skips them
  bool some = false;
  if (!HYD) {
    double wat = 0.;
    const int nall = D.nt * NC;
    for (int r0 = nrow + wv * RB; r0 < nall; r0 += W * RB) {
      double v[RB];
#pragma unroll
      for (int u = 0; u < RB; ++u) v[u] = row_load(w.rows[r0 + u < nall ? r0 + u : nrow].in, x);
#pragma unroll
      for (int u = 0; u < RB; ++u)
        if (r0 + u < nall) {
          some |= live && !(v[u] == 0.);
          if (w.rows[r0 + u].kind & LR_WATER) wat += fmax(0., v[u] * dn) / kMwa;   // (as the clamp leaves it)
        }
    }
    some = __any(some);
    sP[(wv * NP + NP - 1) * kL + lane] = live ? wat : 0.;   // a place that the sweep without hydrometeors leaves alone
  }
  if (wv == 0) {
    sRV[lane] = rv0;
    sF[lane] = 0;
  }
  __syncthreads();

  // ---- sweep: the wavefronts split a target's entries, then its components ----
  const int nt_ = HYD ? D.ntarget : D.it_aero1 - D.it_aero0;
  const int Roff = D.off[2], Ioff = D.off[3];
  const double emax = D.Eiagg_max, emin = D.Eiagg_min;
  // rime fraction of an ice bin (classSection.f90:202-224); kept per bin, as
  // a target's update is the only change to it
  auto rime = [](double n, double nlim, double wa, double ri) -> double {
    return wa > 1.e-23 && ri > 1.e-23 && n > nlim ? ri * kRhori / (wa * kRhoic + ri * kRhori) : 0.;
  };
  if constexpr (HYD && L5) {
    for (int q = wv; q < D.nb[3]; q += W) sRF[q * kL + lane] =
        rime(SC(Ioff + q, 0), D.nlim[Ioff + q], SC(Ioff + q, 1 + iwa), SC(Ioff + q, 1 + irim));
    __syncthreads();
  }
  // x / d for a constant d with reciprocal r: the correctly rounded quotient
  auto quot = [](double x, double d, double r) -> double {
    const double q = x * r;
    return __builtin_fma(__builtin_fma(-q, d, x), r, q);
  };
  // This wavefront's program words of a target, and its kernels: the words are
  // loaded three targets ahead, the kernels two (an unused place has the row
  // of zeros).
  const uint32_t *prog = w.prog + wv * kProg + (lane & (kProg - 1));
  auto words = [&](int it) -> uint32_t { return prog[(it < nt_ ? it : nt_ - 1) * (W * kProg)]; };
  auto word = [](uint32_t pv, int i) -> uint32_t { return (uint32_t)__builtin_amdgcn_readlane((int)pv, i); };
  struct Kern { KT e[kEnt], self; };
  auto fetch = [&](uint32_t pv, Kern &k) {
#pragma unroll
    for (int u = 0; u < kEnt; ++u) k.e[u] = kernel_at((word(pv, u) >> 15) * (uint32_t)(kL * sizeof(KT)));
    k.self = kernel_at(word(pv, kProgK) * (uint32_t)(kL * sizeof(KT)));
  };
  uint32_t pv_n = 0, pv_f = 0, pv_l = 0;      // program words of the next target, the one after, and the one in flight
  uint32_t pv_c = 0;
  Kern kc, kn;
  if (nt_ > 0) {
    pv_n = words(0);
    pv_f = words(1);
    pv_l = words(2);
    fetch(pv_n, kc);
    fetch(pv_f, kn);
  }
  for (int it = 0; it < nt_; ++it) {
    pv_c = pv_n;
    const Kern k = kc;
    pv_n = pv_f; pv_f = pv_l; kc = kn;
    pv_l = words(it + 3);
    fetch(pv_f, kn);
    const uint32_t tf = word(pv_c, kProgT);
    const int t = tf & 255u;
    const uint32_t fl = tf >> 8;
    const double nlim_t = __hiloint2double((int)word(pv_c, kProgN + 1), (int)word(pv_c, kProgN));
    const double Nt = SC(t, 0);
    bool act = live && !(Nt < nlim_t);
    if (HYD && (fl & TF_ICE)) act = act && T < 273.15;  // mo_salsa_dynamics.f90:166
    if (!__any(act)) continue;                          // the same in every wavefront of the block
    const bool ice = HYD && L5 && (fl & TF_ICE);
    const double rft = ice ? sRF[(t - Ioff) * kL + lane] : 0.;
    // the last wavefront forms the target's new rime fraction from its old water
    // and rime, which their owners overwrite beyond the next barrier
    const bool rimer = ice && wv == W - 1;
    const double old_w = rimer ? SC(t, 1 + iwa) : 0., old_r = rimer ? SC(t, 1 + irim) : 0.;
    const int nu = ice ? NV : nwet;                     // components that the target updates
    // a component's owner also moves what coalesces into precipitation
    KT kf[NF];
    if (HYD && wv <= nwet && (fl & (TF_PF | TF_PF_SELF)))
#pragma unroll
      for (int u = 0; u < NF; ++u) kf[u] = kernel_at((word(pv_c, kProgF + u) & 0xffffu) * (uint32_t)(kL * sizeof(KT)));
    double part[A][NC], so[A], sx[A];                   // part: sink, then the sources
#pragma unroll
    for (int v = 0; v < A; ++v) {
      so[v] = sx[v] = 0.;
#pragma unroll
      for (int q = 0; q < NC; ++q) part[v][q] = 0.;
    }
#pragma unroll
    for (int h = 0; h < kEnt; h += 4) {
      uint32_t en[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) en[u] = word(pv_c, h + u);
      if (h && !(en[0] & 511u)) break;                  // a wavefront's entries are filled from the front
      double S[4][NC];
      uint8_t pfb[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const double *sj = sS + ((en[u] >> 9) & 63u) * (NC * kL) + lane;
#pragma unroll
        for (int q = 0; q < NC; ++q) S[u][q] = sj[q * kL];
        if (HYD && (fl & TF_PF)) pfb[u] = sPF[((en[u] & SR_PF) ? (int)(en[u] >> 15) - D.pf0 : 0) * kL + lane];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int v = (h + u) % A;
        const uint32_t role = en[u];
        const double kj = (double)k.e[h + u];
        if (role & SR_SINK) part[v][0] += kj * S[u][0];
        if (role & SR_SRC)                              // (a liquid bin's rime is zero)
#pragma unroll
          for (int q = 1; q < NC; ++q) part[v][q] += kj * S[u][q];
        if (HYD && (role & SR_SPECIAL)) {
          if constexpr (L5) {
            if (role & (SR_SINK_EAGG | SR_SRC_EAGG)) {  // ice aggregation efficiency (processes.f90:758-769)
              const int j = (int)((role >> 9) & 63u);
              const double eg = emax - fmax(sRF[(j - Ioff) * kL + lane], rft) * (emax - emin);
              if (role & SR_SINK_EAGG) part[v][0] += eg * kj * S[u][0];
              if (role & SR_SRC_EAGG)
#pragma unroll
                for (int q = 1; q < NC; ++q) part[v][q] += eg * kj * S[u][q];
            }
            if (role & (SR_PC_WA | SR_PC_RI)) {         // accumulateSourcePhaseChange (:1236-1266)
#pragma unroll
              for (int q = 1; q <= ndry; ++q) part[v][q] += kj * S[u][q];
              if (role & SR_PC_WA) part[v][1 + iwa] += quot(kj * S[u][1 + iwa] * kRhowa, kRhoic, 1. / kRhoic);
              else part[v][1 + irim] += quot(kj * S[u][1 + iwa] * kRhowa, kRhori, 1. / kRhori);
            }
          }
          if (role & SR_PF) {                           // accumulatePrecipFormation (:1458-1576)
            const double kp = pfb[u] ? kj : 0., kr = pfb[u] ? 0. : kj;
            part[v][0] += kp * S[u][0];
#pragma unroll
            for (int q = 1; q < NC; ++q) part[v][q] += kr * S[u][q];
          }
          if (role & SR_FIX_OWN) so[v] += kj * S[u][0];
          if (role & SR_FIX_OTH) sx[v] += kj * S[u][0];
        }
      }
    }
    {
      double *p = sP + wv * NP * kL + lane;
#pragma unroll
      for (int q = 0; q < NC; ++q) {
        double y = part[0][q];
        if constexpr (A == 2) y = y + part[1][q];
        if constexpr (A == 4) y = (y + part[1][q]) + (part[2][q] + part[3][q]);
        p[q * kL] = y;
      }
      if (HYD && (fl & TF_PF)) {
        if constexpr (A == 2) { so[0] = so[0] + so[1]; sx[0] = sx[0] + sx[1]; }
        if constexpr (A == 4) {
          so[0] = (so[0] + so[1]) + (so[2] + so[3]);
          sx[0] = (sx[0] + sx[1]) + (sx[2] + sx[3]);
        }
        p[(NP - 2) * kL] = so[0];
        p[(NP - 1) * kL] = sx[0];
      }
    }
    __syncthreads();
    // components: a wavefront owns whole components, so what it moves to
    // another bin meets no other wavefront
    const double kself = (double)k.self;
    if constexpr (HYD && L5) {
      if (rimer) {                                      // the target's rime fraction after its update
        const double *pp = sP + lane;
        const double sk = tree_sum<W>(pp, NP * kL), ss = (emax - rft * (emax - emin)) * 0.5 * kself * Nt;
        const double nn = Nt * rcp_nr(1. + dt * (sk + ss)), rd = rcp_nr(1. + dt * sk);
        const double vw = (old_w + dt * tree_sum<W>(pp + (1 + iwa) * kL, NP * kL) * Nt) * rd;
        const double vr = (old_r + dt * tree_sum<W>(pp + (1 + irim) * kL, NP * kL) * Nt) * rd;
        if (act) sRF[(t - Ioff) * kL + lane] = rime(nn, nlim_t, vw, vr);
      }
    }
    for (int q = wv; q <= nu; q += W) {
      const double *pp = sP + lane;
      const double sk = tree_sum<W>(pp, NP * kL), sr = tree_sum<W>(pp + q * kL, NP * kL);
      const double Vt = SC(t, q);
      double nw;                                        // the component's new value
      if (q == 0) {
        double ss = 0.;
        if (fl & (TF_SELF_HALF | TF_PF_SELF)) ss = 0.5 * kself * Nt;
        if (HYD && L5 && (fl & TF_SELF_HALF_EAGG)) ss = (emax - rft * (emax - emin)) * 0.5 * kself * Nt;
        nw = Nt * rcp_nr(1. + dt * (sk + ss));
      } else {
        nw = (Vt + dt * sr * Nt) * rcp_nr(1. + dt * sk);
      }
      if (HYD && (fl & TF_PRECIP_SELFCOLL)) {           // precipSelfCoag (:1588-1611)
        const double mv = q ? Vt * Nt * kself : 0.5 * kself * Nt * Nt;
        if (act) {
          SC(t + 1, q) = SC(t + 1, q) + dt * mv;
          nw = nw - dt * mv;
        }
      }
      if (!(HYD && (fl & (TF_PF | TF_PF_SELF)))) {
        if (act) SC(t, q) = nw;
        continue;
      }
      if constexpr (HYD) {
        // coalesced cloud drops into precipitation bins (applyCoagPrecipFormation :649-703),
        // one precipitation bin at a time
        double Nj[NF], Vj[NF];
        int pb_[NF];
        const int ps = (int)word(pv_c, kProgS);
#pragma unroll
        for (int u = 0; u < NF; ++u) {
          const uint32_t e = word(pv_c, kProgF + u);
          const int j = (e >> 16) & 63u;
          Nj[u] = SC(j, 0);
          Vj[u] = SC(j, q);
          pb_[u] = sPF[(e >> 31 ? (int)(e & 0xffffu) - D.pf0 : 0) * kL + lane];
        }
        double fixs = 1., self = 0.;
        int pself = -1;
        if (fl & TF_PF_SELF) {
          fixs = fmax(1. - dt * (0.5 * kself * (Nt * Nt) / Nt), 0.1);
          if (ps >= 0 && act) pself = (int)sPF[ps * kL + lane] - 1;
          if (q && pself >= 0) {
            self = Vt * Nt * kself * fixs;
            nw = nw - dt * self;
          }
        }
        double f_own = 1., f_oth = 1.;                  // fix_coag
        if (fl & TF_PF) {
          f_own = fmax(1. - dt * tree_sum<W>(pp + (NP - 2) * kL, NP * kL), 0.1);
          f_oth = fmax(1. - dt * tree_sum<W>(pp + (NP - 1) * kL, NP * kL), 0.1);
        }
        uint32_t pm = pself >= 0 ? 1u << pself : 0u;
        double mv[NF];
#pragma unroll
        for (int u = 0; u < NF; ++u) {
          const uint32_t e = word(pv_c, kProgF + u);
          pb_[u] = (e >> 31) && act ? pb_[u] - 1 : -1;
          if (pb_[u] >= 0) pm |= 1u << pb_[u];
          const double kj = (double)kf[u], fx = (e >> 30) & 1u ? f_own : f_oth;
          mv[u] = q ? (Vj[u] * Nt + Vt * Nj[u]) * kj * fx : kj * Nj[u] * Nt * fx;
        }
        if (act) SC(t, q) = nw;
        const bool odd = word(pv_c, kProgQ);
        for (int pb = 0; pb < D.nb[2]; ++pb) {
          if (!__any((pm >> pb) & 1u)) continue;
          double y[NF / 4];
#pragma unroll
          for (int u = 0; u < NF; u += 4)
            y[u / 4] = ((pb_[u] == pb ? mv[u] : 0.) + (pb_[u + 1] == pb ? mv[u + 1] : 0.)) +
                       ((pb_[u + 2] == pb ? mv[u + 2] : 0.) + (pb_[u + 3] == pb ? mv[u + 3] : 0.));
          double vp = y[0] + y[1];
          if constexpr (NF == 12) vp = odd ? y[0] + (y[1] + y[2]) : vp + y[2];
          if (pb == pself) {
            if (q) vp += self;
            else vp += 0.5 * kself * Nt * Nt * fixs;
          }
          if ((pm >> pb) & 1u) SC(Roff + pb, q) = SC(Roff + pb, q) + dt * vp;
        }
      }
    }
    __syncthreads();
  }
  // clamp (mo_salsa_dynamics.f90:189-198), and which kinds of bins hold particles
  {
    uint32_t any = 0;   // bit 0 cloud > nlim, 1 precip > prlim, 2 ice > prlim, 3 aero > nlim
    for (int b = wv; b < nb; b += W) {
      const double nv = SC(b, 0);
      if (nv < -1.e-6) flags |= SALSA_CELL_NEG_NUMC;
      const int c = D.cat_of[b];
      if (nv > (c < 2 ? kNlim : kPrlim)) any |= c == 0 ? 8u : 1u << (c - 1);
#pragma unroll
      for (int q = 0; q < NC; ++q) SC(b, q) = fmax(0., SC(b, q));
    }
    if (any) atomicOr(sF + lane, (int)(any << 8));
  }
  __syncthreads();

  // ---- condensation (mo_salsa_dynamics.f90:276-342, 691-1125) ----
  const double zrh = rv0 / rs;
  if (D.lscnd && (D.lscndh2oae || D.lscndh2ocl || D.lscndh2oic)) {
    auto aero_water = [&]() -> double {                 // per partial the bins v, v + VL, ...
      double y[VL / 4];
#pragma unroll
      for (int v = 0; v < VL; v += 4) {
        double z[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          z[u] = 0.;
          for (int b = v + u; b < D.nb[0]; b += VL) z[u] += SC(b, 1 + iwa);
        }
        y[v / 4] = (z[0] + z[1]) + (z[2] + z[3]);
      }
      if constexpr (VL == 32) return ((y[0] + y[1]) + (y[2] + y[3])) + ((y[4] + y[5]) + (y[6] + y[7]));
      else if constexpr (VL == 16) return (y[0] + y[1]) + (y[2] + y[3]);
      else return y[0];
    };
    double w1 = 0.;
    if (wv == W - 1) w1 = aero_water() * kRhowa;
    __syncthreads();                          // read before the equilibration writes
    // equilibration: the 1a chain on the first wavefront, the 2a/2b bins
    // (zrh < 0.98, or without aerosol condensation) over all of them
    int isu = -1, ioc = -1, iss = -1, ibc = -1, idu = -1;
    for (int s = 0; s < ndry; ++s) {
      const int id = D.dry_id[s];
      if (id == 0) isu = s;
      if (id == 1) ioc = s;
      if (id == 2) ibc = s;
      if (id == 3) idu = s;
      if (id == 4) iss = s;
    }
    auto vol = [&](int b, int s) -> double { return s >= 0 ? SC(b, 1 + s) : 0.; };
    if (wv == 0) {
      double zke = 1.001;
      for (int b = D.in1a; b <= D.fn1a; ++b) {
        const double n = SC(b, 0);
        const bool on = live && n > kNlim;
        if (!__any(on)) continue;
        const double v1 = vol(b, isu), v2 = vol(b, ioc), z0 = zke;
        const double lw = equil_bin<false>(n, v1 / n + v2 / n, v1 * (kRhosu / kMsu), kEpsoc * v2 * (kRhooc / kMoc), 0.,
                                           T, fmin(fmax(zrh, 0.05), 0.98), w.dwa[(blk * D.nb[0] + b) * kL + lane], zke, on,
                                           flags);
        if (on) SC(b, 1 + iwa) = lw / kRhowa;
        else zke = z0;
      }
    }
    // (cell, bin) tasks of the cells that need it, side by side
    const uint64_t r2 = __ballot(live && (zrh < 0.98 || !D.lscndh2oae));
    const int n2 = (int)__popcll(r2);
    if (wv == 0 && ((r2 >> lane) & 1ull)) sL[__popcll(r2 & ((1ull << lane) - 1ull))] = (uint8_t)lane;
    if (n2) {
      __syncthreads();
      const int nq = n2 * (D.fn2b - D.in2a + 1);
      for (int q0 = (wv ? wv - 1 : W - 1) * kL; q0 < nq; q0 += W * kL) {
        const int q = q0 + lane, b = D.in2a + (q < nq ? q / n2 : 0), cell = sL[q < nq ? q % n2 : 0];
        const double *S = sS + b * (NC * kL) + cell;
        const double n = S[0];
        const bool on = q < nq && n > kNlim;
        if (!__any(on)) continue;
        auto at = [&](int s) -> double { return s >= 0 ? S[(1 + s) * kL] : 0.; };
        const double z0 = at(isu), z1 = at(ioc), z2 = at(ibc), z3 = at(idu), z4 = at(iss);
        const int64_t xc = lanes_index(a, ids[cell]);
        const double Tc = a.temp[xc], rsc = a.rsl[xc];
        double rvc = a.rv_p[xc];
        if (!a.lsfreeRH) rvc = fmin(rvc, rsc * a.rhlim);
        double zke = 1.02;
        uint32_t fl = 0;
        const double lw = equil_bin<true>(n, z0 / n + z1 / n + z2 / n + z3 / n + z4 / n, z0 * (kRhosu / kMsu),
                                          kEpsoc * (z1 * (kRhooc / kMoc)), z4 * (kRhoss / kMss), Tc,
                                          fmin(fmax(rvc / rsc, 0.37), 0.98), w.dwa[(blk * D.nb[0] + b) * kL + cell], zke,
                                          on, fl);
        if (on) sS[(b * NC + 1 + iwa) * kL + cell] = lw / kRhowa;
        if (fl) atomicOr(sF + cell, (int)fl);
      }
    }
    __syncthreads();
    // the cells that take the substeps (cell-skip predicate, :784-788; .AND. binds before .OR.)
    const uint32_t any = (uint32_t)sF[lane] >> 8;
    const uint64_t pm = __ballot(live && ((any & 1u) || ((any & 2u) && D.lscndh2ocl) || ((any & 4u) && D.lscndh2oic) ||
                                          ((any & 8u) && zrh > 0.98 && D.lscndh2oae)));
    if (wv == W - 1) sRV[lane] = rv0 - (aero_water() * kRhowa - w1) / (P * kMair / (kRg * T));
    if (wv == 0 && ((pm >> lane) & 1ull)) sL[__popcll(pm & ((1ull << lane) - 1ull))] = (uint8_t)lane;
    __syncthreads();

    // substeps: W neighbouring lanes per cell, the updated bins dealt over
    // their VL partials and kept in registers
    if ((int)threadIdx.x / W < (int)__popcll(pm) || wv * kL / W < (int)__popcll(pm)) {
      const bool lq = (int)threadIdx.x / W < (int)__popcll(pm);
      const int cq = lq ? (int)sL[threadIdx.x / W] : (int)(__ffsll((long long)pm) - 1), sub = (int)threadIdx.x % W;
      const int64_t xq = lanes_index(a, ids[cq]);
      const double Tq = a.temp[xq], Pq = a.press[xq], rsq = a.rsl[xq], rsiq = L5 ? a.rsi[xq] : 0.;
      double rvq = a.rv_p[xq];
      if (!a.lsfreeRH) rvq = fmin(rvq, rsq * a.rhlim);
      const double zrhq = rvq / rsq;
      rvq = sRV[cq];
#define QC(b, q) sS[((b) * NC + (q)) * kL + cq]
      const bool aon = zrhq > 0.98 && D.lscndh2oae, ion = D.lscndh2oic && Tq < 273.15, con = D.lscndh2ocl;
      uint64_t upd = 0;   // bins that the substeps update
      double st_[V], sf_[V];                   // all water, and that of the other bins (moles)
#pragma unroll
      for (int v = 0; v < V; ++v) {
        st_[v] = sf_[v] = 0.;
        for (int b = sub * V + v; b < nb; b += VL) {
          const int c = D.cat_of[b];
          const double n = QC(b, 0);
          const double wb = c == 3 ? QC(b, 1 + iwa) * kRhoic / kMwa + QC(b, 1 + irim) * kRhori / kMwa
                                   : QC(b, 1 + iwa) * kRhowa / kMwa;
          st_[v] += wb;
          if (n > D.nlim[b] && (c == 0 ? aon && b >= D.in2a : c == 3 ? ion : con)) upd |= 1ull << b;
          else sf_[v] += wb;
        }
      }
      upd = (uint64_t)cell_or<W>((uint32_t)upd) | ((uint64_t)cell_or<W>((uint32_t)(upd >> 32)) << 32);
      {
        const double rhoair = kMair * Pq / (kRg * Tq);
        double zdf = (5. / (16. * kAvog * rhoair * 1.e-3 * (3.11e-8 * 3.11e-8))) *
                     ::sqrt(kRg * 1.e7 * Tq * kMair * 1.e3 * (kMwa + kMair) * 1.e3 / (2. * kPi * kMwa * 1.e3));
        zdf = zdf * 1.e-4;
        const double zmfp = 3. * zdf * ::sqrt(kPi * kMwa / (8. * kRg * Tq));
        const double zthc = 0.023807 + 7.1128e-5 * (Tq - 273.16);
        const double hl = ((kAlv * kMwa) / (kRg * Tq)) - 1., hs = ((kAls * kMwa) / (kRg * Tq)) - 1.;
        const double csul = rsq * rhoair / kMwa, csui = rsiq * rhoair / kMwa;
        // the r-th updated bin goes to partial r % VL; a lane's slot q = v * NR + k
        // holds the k-th bin of its partial v
        int bin[NQ];
        {
          uint64_t m = upd;
#pragma unroll
          for (int r = 0; r < VL * NR; ++r) {
            const int b = m ? __builtin_ctzll(m) : -1;
            m &= m - 1;
            const int q = (r % V) * NR + r / VL;
            if ((r % VL) / V == 0) bin[q] = b;          // lane 0's; the others overwrite theirs
            else if ((r % VL) / V == sub) bin[q] = b;
          }
        }
        double zcw[NQ], zmt[NQ], zkl[NQ], zns[NQ], zws[NQ], s1_[V], s2_[V];
        uint32_t on_ = 0, ice_ = 0, qw = 0;
#pragma unroll
        for (int v = 0; v < V; ++v) s1_[v] = s2_[v] = 0.;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
          __builtin_amdgcn_sched_barrier(0);            // one bin's transcendental chains at a time
          zcw[q] = 0.; zmt[q] = 0.; zkl[q] = 1.; zns[q] = 0.; zws[q] = 0.;
          const bool on = bin[q] >= 0;
          if (!__any(on)) continue;
          qw |= 1u << q;
          if (on) {
            const int b = bin[q], c = D.cat_of[b];
            const double n = QC(b, 0);
            double vs = 0.;
#pragma unroll
            for (int s = 0; s < NV; ++s) vs += QC(b, 1 + s);
            double dw = cbrt_fast(vs / n / kPi6);
            dw = fmin(dw, D.dlim[b]);                   // updateDiameter (:803-806); dnsp == dwet
            double zn = 0.;
            for (int s = 0; s < ndry; ++s) zn += D.diss[s] * QC(b, 1 + s) * D.rholiq[s] / D.mm[s];
            const double zknud = 2. * zmfp / dw;
            const double zbeta = (zknud + 1.) / (0.377 * zknud + 1. + 4. / 3. * (zknud + zknud * zknud));
            const bool ic = HYD && c == 3;              // :892-930 (capacitance 0.5*dnsp, activity 1), :826-890, :932-955
            const double wa = QC(b, 1 + iwa);
            zcw[q] = ic ? wa * kRhoic / kMwa + QC(b, 1 + irim) * kRhori / kMwa : wa * kRhowa / kMwa;
            const double kl = ::exp(4. * (ic ? kSurfi0 : kSurfw0) * kMwa / (kRg * Tq * kRhowa * dw));
            const double ws = ic ? kl : act_h2o<false>(wa * D.rholiq[iwa] / D.mm[iwa], zn) * kl;
            const double h1 = ic ? n * 4. * kPi * (0.5 * dw) * zdf * zbeta : n * 2. * kPi * dw * zdf * zbeta;
            const double h2 = kMwa * zdf * (ic ? kAls : kAlv) * ws * (ic ? csui : csul) / (zthc * Tq);
            const double mt = h1 / (h2 * (ic ? hs : hl) + 1.);
            zkl[q] = kl; zws[q] = ws; zns[q] = zn; zmt[q] = mt;
            on_ |= 1u << q;
            if (ic) ice_ |= 1u << q;
            s1_[q / NR] += mt * ws * (ic ? csui : csul);
            s2_[q / NR] += mt;
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        double sfix = tree_lanes<VL>(sf_), stot = tree_lanes<VL>(st_), s1 = tree_lanes<VL>(s1_);
        const double s2 = tree_lanes<VL>(s2_);
        if (!HYD) {
          double hw = 0.;
          for (int v = 0; v < W; ++v) hw += sP[(v * NP + NP - 1) * kL + cq];
          sfix += hw;
          stot += hw;
        }
        double zcwc = rvq * rhoair / kMwa;
        const double zcwtot = zcwc + stot;
        // substeps of adt = 0.02 s (:986-1053)
        const double adt = 2.e-2;
        double zcwint = 0.;
        const int nsub = a.nsub;
        const double rz = rcp_nr(1. + adt * s2);
        if constexpr (!L5) {
          // the same substep with its constants folded: a = adt zmt, and the
          // saturation ratio's constants zkl csu and zmt zkl csu
#pragma unroll
          for (int q = 0; q < NQ; ++q) {
            zws[q] = zkl[q] != 0. ? zws[q] / zkl[q] : 0.;          // activity
            zkl[q] *= csul;
          }
          double zme[NQ];
#pragma unroll
          for (int q = 0; q < NQ; ++q) {
            zme[q] = zmt[q] * zkl[q];
            zmt[q] *= adt;
          }
          for (int st = 0; st < nsub; ++st) {
            zcwint = fmin(__builtin_fma(adt, s1, zcwc) * rz, zcwtot);
            double tsum = 0., s1n = 0.;
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
              if ((qw >> q) & 1u) {
                const double lim = 0.1 * zcw[q], d = zmt[q] * __builtin_fma(-zws[q], zkl[q], zcwint);
                const double nw = fmax(zcw[q] + fmin(fmax(d, -lim), lim), 0.);
                const double den = fmax(kEpsR8, nw + zns[q]);
                const double r = __builtin_amdgcn_rcp(den), e = __builtin_fma(-den, r, 1.);
                zws[q] = fmax(0.1, nw * __builtin_fma(r, __builtin_fma(e, e, e), r));
                zcw[q] = nw;
                tsum += nw;
                s1n = __builtin_fma(zme[q], zws[q], s1n);
              }
            }
            tsum = cell_sum<W>(tsum);
            s1 = cell_sum<W>(s1n);
            zcwint = zcwtot - (sfix + tsum);
            zcwc = zcwint;
          }
        } else for (int st = 0; st < nsub; ++st) {
          const double zhlp1 = zcwc + adt * s1;
          zcwint = fmin(zhlp1 * rz, zcwtot);
          double t_[V];
#pragma unroll
          for (int v = 0; v < V; ++v) t_[v] = s1_[v] = 0.;
#pragma unroll
          for (int q = 0; q < NQ; ++q) {
            if ((qw >> q) & 1u) {
              const bool ic = HYD && ((ice_ >> q) & 1u);
              const double csu = ic ? csui : csul;
              const double d = adt * zmt[q] * (zcwint - zws[q] * csu);
              double nw = zcw[q] + fmin(fmax(d, -1.e-1 * zcw[q]), 1.e-1 * zcw[q]);
              nw = fmax(nw, 0.);
              zcw[q] = nw;
              zws[q] = ic ? zkl[q] : act_h2o<true>(nw, zns[q]) * zkl[q];
              t_[q / NR] += nw;
              s1_[q / NR] += zmt[q] * zws[q] * csu;
            }
          }
          const double tsum = tree_lanes<VL>(t_);
          s1 = tree_lanes<VL>(s1_);
          zcwint = zcwtot - (sfix + tsum);
          zcwc = zcwint;
        }
        if (lq) {
          if (sub == 0) {
            sRV[cq] = zcwint * kMwa / rhoair;
            if (nsub > 100) atomicOr(sF + cq, (int)SALSA_CELL_SUBSTEPS);
          }
          // write-back (:1058-1117): the other bins' water goes through moles and back
          for (int b = sub; b < nb; b += W)
            if (!((upd >> b) & 1ull) && D.cat_of[b] != 3)
              QC(b, 1 + iwa) = fmax(0., QC(b, 1 + iwa) * kRhowa / kMwa * kMwa / kRhowa);
#pragma unroll
          for (int q = 0; q < NQ; ++q) {
            if (!((on_ >> q) & 1u)) continue;
            const int b = bin[q];
            if (!((ice_ >> q) & 1u)) {
              QC(b, 1 + iwa) = fmax(0., zcw[q] * kMwa / kRhowa);
            } else {
              const double org_i = QC(b, 1 + iwa) * kRhoic / kMwa, org_r = QC(b, 1 + irim) * kRhori / kMwa;
              const double orig = org_i + org_r;
              const double dvt = zcw[q] - orig;
              if (dvt > 0.) {
                QC(b, 1 + iwa) = QC(b, 1 + iwa) + dvt * kMwa / kRhoic;
              } else if (dvt < 0.) {
                const double fr = (zcw[q] / orig) - 1.;
                QC(b, 1 + iwa) = QC(b, 1 + iwa) + (fr * org_i) * kMwa / kRhoic;
                QC(b, 1 + irim) = QC(b, 1 + irim) + (fr * org_r) * kMwa / kRhori;
              }
            }
          }
        }
      }
#undef QC
    }
    __syncthreads();
  }

  // ---- output (mo_salsa_driver.f90:310-388): tendency += (new - old) / dt, or the new state ----
  const bool inp = a.inplace;
  if (live) {
    // RB rows at a time: their old values and tendencies are loaded together
    auto put_rows = [&](int from, int to, auto &&value) {
      for (int r0 = from; r0 < to; r0 += W * RB) {
        double o[RB], tn[RB];
#pragma unroll
        for (int u = 0; u < RB; ++u) {
          const LaneRow &r = w.rows[r0 + u < to ? r0 + u : r0];
          o[u] = tn[u] = 0.;
          if (!inp) {
            o[u] = row_load(r.in, x);
            tn[u] = row_load(r.out, x);
          }
        }
#pragma unroll
        for (int u = 0; u < RB; ++u) {
          if (r0 + u >= to) break;
          const LaneRow &r = w.rows[r0 + u];
          if (r.kind & LR_NONE) continue;
          const double nv = value(r0 + u, r);
          if (!isfinite(nv)) flags |= SALSA_CELL_NONFINITE;
          row_store(r.out, x, inp ? nv : tn[u] + (nv - o[u]) / dt);
        }
      }
    };
    put_rows(wv * RB, nrow, [&](int r, const LaneRow &row) { return sS[r * kL + lane] * row.rho / dn; });
    if (wv == 0) {
      const double rvn = sRV[lane];
      if (!isfinite(rvn)) flags |= SALSA_CELL_NONFINITE;
      if (inp) a.rv_o[x] = rvn;
      else a.rv_t[x] = a.rv_t[x] + (rvn - rv0) / dt;
    }
    if (!HYD && some)                         // what the inactive bins hold, through the same unit changes
      put_rows(nrow + wv * RB, D.nt * NC, [&](int, const LaneRow &row) {
        const double m = row_load(row.in, x) * dn;
        if ((row.kind & LR_NUMBER) && m < -1.e-6) flags |= SALSA_CELL_NEG_NUMC;
        return fmax(0., m / row.rho) * row.rho / dn;
      });
  }
  if (flags) atomicOr(sF + lane, (int)flags);
  __syncthreads();
  if (wv == 0 && live) {
    const int f = sF[lane] & 0xff;
    a.cell_flags[icell] = (uint8_t)f;
    if (f) atomicOr(a.fault_any, f);
  }
#undef SC
}

template <class KT, int NV, bool L5, int WP, int C, int W, int VL, int NR, bool HYD>
int launch_pair_sweep(const DevLayout &L, const DevLayout *d, const StepArgs &a, LanesArgs w, hipStream_t s) {
  const int nb = HYD ? L.nt : L.nb[0];
  const size_t lp = pairs_lds(nb, sizeof(KT), C), ls = sweep_lds(nb, NV, W, HYD ? L.ncc : 0, HYD && L5 ? L.nb[3] : 0);
  const int64_t most = (a.ncells + kL - 1) / kL, gn = HYD ? w.gn_hyd : w.gn_aero;
  for (int64_t g0 = 0; g0 < most; g0 += gn) {
    const unsigned grid = (unsigned)(most - g0 < gn ? most - g0 : gn);
    w.g0 = (int)g0;
    hipLaunchKernelGGL((k_lanes_pairs<KT, NV, WP, C, HYD>), dim3(grid * (kL / C)), dim3(64 * WP), lp, s, d, a, w);
    hipLaunchKernelGGL((k_lanes_sweep<KT, NV, L5, W, VL, NR, HYD>), dim3(grid), dim3(64 * W), ls, s, d, a, w);
  }
  return (int)hipGetLastError();
}

constexpr int kMaxLds = 160 * 1024;
// The sweep's shape: wavefronts per workgroup (also the lanes per cell of the
// substeps), partial sums per cell, bins of the substeps per partial.  A for
// the cells without hydrometeors; 2 for two volumes per bin (one dry species
// and water), 4 for more.
constexpr int kWavesA = 4, kPartA = 4, kBinsA = 12 / 4;
constexpr int kWaves2 = 4, kPart2 = 4, kBins2 = 24 / 4;
constexpr int kWaves4 = 8, kPart4 = 16, kBins4 = 2;
// level 5 in FP64: the order of 32 lanes per cell, at which the general kernel
// runs there (see tree_sum)
constexpr int kPart5d = 32, kBins5d = 1;

inline int lanes_volumes(const DevLayout &L) { return L.level == 5 ? L.nspec : L.nwet; }

// The sweep program of the layout (prog null: nothing written); returns its
// words, -1 where the layout does not fit.  Entry e of a target is in partial e % VL, which belongs to
// wavefront (e % VL) / (VL / W).  The precipitation-formation entries are at
// most 8 neighbours: they start at their partial's place in a quad of the
// tree, and the parity of that quad says how the (up to three) quads add up.
int sweep_program(const DevLayout &L, int kt, bool hyd, uint32_t *prog) {
  const int NV = lanes_volumes(L), W = !hyd ? kWavesA : NV > 2 ? kWaves4 : kWaves2, VL = !hyd ? kPartA : NV == 2 ? kPart2 : L.level == 5 && kt == 8 ? kPart5d : kPart4, A = VL / W;
  const int i0 = hyd ? 0 : L.it_aero0, nt = hyd ? L.ntarget : L.it_aero1 - L.it_aero0;
  const uint32_t zero = hyd ? L.npair : L.npair_aa;
  if (zero > 1023u || nt < 1) return -1;
  auto set = [&](int it, int v, int q, uint32_t x) { if (prog) prog[((size_t)it * W + v) * kProg + q] = x; };
  for (int it = 0; it < nt; ++it) {
    const DevTarget &T = L.tgt[i0 + it];
    const bool self = T.flags & (TF_SELF_HALF | TF_SELF_HALF_EAGG | TF_PF_SELF | TF_PRECIP_SELFCOLL);
    const int pid = self ? L.pidx[T.t][T.t] : -1, ne = hyd ? T.nent : T.nent_aero;
    uint64_t bits;
    std::memcpy(&bits, &L.nlim[T.t], 8);
    for (int v = 0; v < W; ++v) {
      for (int q = 0; q < kProg; ++q) set(it, v, q, 0);
      for (int q = 0; q < kEnt; ++q) set(it, v, q, zero << 15 | (uint32_t)T.t << 9);
      for (int q = 0; q < prog_pf(VL); ++q) set(it, v, kProgF + q, zero | (uint32_t)T.t << 16);
      set(it, v, kProgT, (uint32_t)T.t | T.flags << 8);
      set(it, v, kProgK, pid >= 0 ? (uint32_t)pid : zero);
      set(it, v, kProgN, (uint32_t)bits);
      set(it, v, kProgN + 1, (uint32_t)(bits >> 32));
      set(it, v, kProgS, (T.flags & TF_PF_SELF) && pid >= 0 ? (uint32_t)(pid - L.pf0) : ~0u);
    }
    int pf0 = -1;
    for (int e = 0; e < ne; ++e) {
      const uint32_t x = L.ent[T.ent0 + e], j = x & 63u, r = (x >> 6) & 1023u, pair = x >> 16;
      const uint32_t role = (r & R_SINK ? SR_SINK : 0) | (r & R_SRC ? SR_SRC : 0) | (r & R_SINK_EAGG ? SR_SINK_EAGG : 0) |
                            (r & R_SRC_EAGG ? SR_SRC_EAGG : 0) | (r & R_PC_WA ? SR_PC_WA : 0) | (r & R_PC_RI ? SR_PC_RI : 0) |
                            (r & (R_PF_OWN | R_PF_OTH) ? SR_PF : 0) | (r & R_FIX_OWN ? SR_FIX_OWN : 0) |
                            (r & R_FIX_OTH ? SR_FIX_OTH : 0);
      const int v = (e % VL) / A, at = (e / VL) * A + e % A;
      if (at >= kEnt) return -1;
      set(it, v, at, pair << 15 | j << 9 | role);
      if (!(role & SR_PF)) continue;
      if (pf0 < 0) pf0 = VL >= 16 ? e - e % 4 : e;
      if (e - pf0 >= prog_pf(VL)) return -1;
      for (int u = 0; u < W; ++u) {
        set(it, u, kProgF + e - pf0, pair | j << 16 | (r & R_PF_OWN ? 1u << 30 : 0u) | 1u << 31);
        set(it, u, kProgQ, (pf0 / 4) & 1);
      }
    }
  }
  return nt * W * kProg;
}

}  // namespace

// Slots whose kernels the work space holds: of the cells with hydrometeors,
// and of those without (fewer pairs).  About 200 MB of FP32 kernels each of
// the 26-bin layout.  (Times below: the two lists one after the other.)
constexpr int kSlotsHyd = 1 << 17, kSlotsAero = 1 << 19;

// The fewest cells of a context that steps with one lane per cell.  A
// workgroup here takes as long for its 64 cells as for one, about 0.1 ms for a
// sweep, and the chip is filled from 256 workgroups on; 16 to 64 lanes per
// cell share the work of a few cells.  Measured us, here (both lists side by
// side) / the general kernel on all cells in one launch: level 4 (32 lanes)
// mixed 5 120 cells 183 / 133, 7 680 186 / 183, 10 240 189 / 201, 15 360
// 190 / 266, with drizzle 7 680 202 / 196, 10 240 205 / 226, 15 360 206 / 293, FP64
// 5 120 180 / 144, 7 680 182 / 198, 15 360 184 / 292: the line would pay from 10 240 on,
// it lies where it paid with the lists one after the other (246 / 266).  Level 5
// (16 lanes) with ice in 30 % of the cells mixed 5 120 238 / 210, 10 240
// 243 / 351, FP64 3 840 320 (one after the other) / 194, 5 120 250 / 319; with ice
// everywhere mixed 3 840 228 / 188, 5 120 236 / 211, 10 240 249 / 372, FP64
// 3 840 247 / 200, 5 120 253 / 348: more than one wavefront per SIMD.
int64_t lanes_least(const DevLayout &L) { return L.level == 5 ? 4096 : 15360; }

// Whether the lane kernels take a context of ncells cells with this layout.
bool lanes_fit(const DevLayout &L, int kt, int64_t ncells) {
  if (ncells < lanes_least(L)) return false;
  const int NV = lanes_volumes(L);
  if (NV < 2 || NV > 4 || (NV == 4 && L.level != 5) || (NV == 2 && L.level == 5) || L.nt > 63 || L.npair < 1 || L.npair > 65535) return false;
  const int VL = NV == 2 ? kPart2 : kPart4, bins = VL * (NV == 2 ? kBins2 : kBins4);
  const bool fits = L.nt - L.in2a <= bins && L.nb[0] - L.in2a <= kPartA * kBinsA && pairs_lds(L.nt, kt, 32) <= kMaxLds &&
                    pairs_lds(L.nb[0], kt, kL) <= kMaxLds && sweep_lds(L.nt, NV, NV == 2 ? kWaves2 : kWaves4, L.ncc, L.nb[3]) <= kMaxLds;
  return fits && L.lscoag && !L.lsdistupdate && !L.autoconv2 && !L.lsactiv && lanes_program(L, kt, nullptr) > 0;
}

// The sweep programs with and then without hydrometeors; returns their words,
// -1 where the layout does not fit.
int lanes_program(const DevLayout &L, int kt, uint32_t *prog) {
  const int n = sweep_program(L, kt, true, prog);
  if (n < 0) return -1;
  const int m = sweep_program(L, kt, false, prog ? prog + n : nullptr);
  return m < 0 ? -1 : n + m;
}

// Work space of a context with ncells cells: byte offsets and the total; where the
// second sweep program begins.
size_t lanes_work(const DevLayout &L, int kt, int64_t ncells, LanesArgs &w) {
  auto slots = [&](int most) { const int64_t n = (ncells + kL - 1) / kL * kL; return (int64_t)(n < most ? n : most); };
  const int64_t sh = slots(kSlotsHyd), sa = slots(kSlotsAero);
  w.gn_hyd = (int)(sh / kL);
  w.gn_aero = (int)(sa / kL);
  size_t o = 0;
  auto take = [&](size_t n) { const size_t at = o; o += (n + 255) / 256 * 256; return at; };
  take((size_t)sh * (L.npair + 1) * kt);
  w.o_Ka = take((size_t)sa * (L.npair_aa + 1) * kt);
  w.o_pf = take((size_t)sh * (L.ncc > 0 ? L.ncc : 1));
  w.o_dwa = take((size_t)sh * L.nb[0] * 8);
  w.o_dwaa = take((size_t)sa * L.nb[0] * 8);
  w.o_rows = take((size_t)L.nt * (1 + lanes_volumes(L)) * sizeof(LaneRow));
  w.prog_aero = sweep_program(L, kt, true, nullptr);
  return o;
}

int launch_lanes_class(const DevLayout &L, const DevLayout *d, const StepArgs &a, const LanesArgs &w, hipStream_t s) {
  hipLaunchKernelGGL(k_lanes_start, dim3(1), dim3(256), 0, s, d, a, w, 1 + lanes_volumes(L));
  hipLaunchKernelGGL(k_lanes_class, dim3((unsigned)((a.ncells + kClassThreads - 1) / kClassThreads)), dim3(kClassThreads),
                     0, s, d, a, w);
  return (int)hipGetLastError();
}

// The cells with or without hydrometeors.
int launch_lanes(const DevLayout &L, int precision, bool hyd, const DevLayout *d, const StepArgs &a, const LanesArgs &w0,
                 hipStream_t s) {
  LanesArgs w = w0;
  const int NV = lanes_volumes(L);
  if (!hyd) {
    w.prog += w.prog_aero;
    w.K = w.Ka;
    w.dwa = w.dwaa;
  }
#define SALSA_LANES(KT, NV_, L5, WP, W, VL, NR)                                                        \
  return hyd ? launch_pair_sweep<KT, NV_, L5, WP, 32, W, VL, NR, true>(L, d, a, w, s)                  \
             : launch_pair_sweep<KT, NV_, L5, 4, kL, kWavesA, kPartA, kBinsA, false>(L, d, a, w, s)
  const bool l5 = L.level == 5;
  if (precision == SALSA_FP64) {
    if (NV == 2) SALSA_LANES(double, 2, false, 8, kWaves2, kPart2, kBins2);
    if (NV == 3 && !l5) SALSA_LANES(double, 3, false, 8, kWaves4, kPart4, kBins4);
    if (NV == 3) SALSA_LANES(double, 3, true, 8, kWaves4, kPart5d, kBins5d);
    SALSA_LANES(double, 4, true, 8, kWaves4, kPart5d, kBins5d);
  }
  if (NV == 2) SALSA_LANES(float, 2, false, 4, kWaves2, kPart2, kBins2);
  if (NV == 3 && !l5) SALSA_LANES(float, 3, false, 4, kWaves4, kPart4, kBins4);
  if (NV == 3) SALSA_LANES(float, 3, true, 4, kWaves4, kPart4, kBins4);
  SALSA_LANES(float, 4, true, 4, kWaves4, kPart4, kBins4);
#undef SALSA_LANES
}

}  // namespace salsa
