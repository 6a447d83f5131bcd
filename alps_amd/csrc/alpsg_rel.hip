// Relativistic species (relativistic = T) of disp(om), for a batch of omegas.
//
// The reference treats a relativistic species in two ways per harmonic n,
// chosen by determine_resonances (ALPS_fns.f90:680-701), which asks whether
// the resonance p_res = (Gamma m om - n q)/kpar of some point of the
// (pperp, ppar) grid falls into that point's own ppar cell:
//
//  * no such point: integrate() over the (pperp, ppar) grid with the point's
//    Gamma in resU (ALPS_fns.f90:799-864, 1560-1596).  Gamma couples pperp and
//    ppar, so the pperp moments of the non-relativistic sweep do not apply;
//    k_rel_nonres sums the 2-D trapezoid directly.
//  * otherwise: integrate_res_rel and landau_integrate_rel along the
//    resonance curve on the (Gamma, pparbar) grid (ALPS_fns_rel.f90:460-1092):
//    k_rel_res, the trapezoid of resU_rel * int_T_rel around the
//    principal-value window of each Gamma row, plus principal_integral_rel;
//    int_T_rel reads J_n from a per-k table on the same grid (k_rel_bessel).
//    k_rel_landau, the Landau term, evaluates int_T_res_rel with the 21-term
//    series CBESSJ.
//
// k_rel_flags decides the flags of a batch first.  The kernels write their
// partial chi into slots of chiR (rel_slots) and the n = -1, 0, 1 terms into
// slots of lowR (rel_low_slots), read by k_assemble for relativistic species
// only.  The root server takes the served form of the sums (launch_rel_ord).
// Decision-critical arithmetic (resonance flags, window limits, the
// principal-value ladder positions) is evaluated without FMA contraction in
// the reference's operation order.
#include <type_traits>

#include "alpsg_device.h"
#include "alpsg_fit.h"

namespace {

constexpr double PI_R = 3.141592653589793238462643383279502884;

__device__ __forceinline__ cd cdivr(cd a, double d) { return cd{a.re / d, a.im / d}; }
__device__ __forceinline__ double m1p(int n) { return (n % 2 == 0) ? 1.0 : -1.0; }

// mode order k: 0 xx, 1 yy, 2 zz, 3 xy, 4 xz, 5 yz; the mode's product among
// {a1, p a1, p^2 a1, a2, a3, p a3}
__device__ __forceinline__ int acc_of_mode(int k) {
  return k == 0 ? 0 : k == 1 ? 3 : k == 2 ? 2 : k == 3 ? 4 : k == 4 ? 1 : 5;
}

// T-tensor constant C_k(n) of int_T (ALPS_fns.f90:1659-1703) for the
// (pperp, ppar) grid; z = kperp/q or 1/q.
__device__ __forceinline__ cd tconst_r(const ProbDev &Pd, const SpecDev &S, int n, int k) {
  const double kp = Pd.kperp, z = S.z;
  const bool kn = Pd.kperp_norm != 0;
  switch (k) {
    case 0: return mk(1.0 * (n * n) / (z * z), 0.0);
    case 1: return mk(kn ? 1.0 : kp * kp, 0.0);
    case 2: return mk(kn ? 1.0 : kp * kp, 0.0);
    case 3: return mk(0.0, (kn ? 1.0 : kp) * (1.0 * n) / z);
    case 4: return mk((kn ? 1.0 : kp) * (1.0 * n) / z, 0.0);
    default: return mk(0.0, kn ? -1.0 : -(kp * kp));
  }
}

// ---------------------------------------------------------------------------
// k_rel_flags: determine_resonances of the harmonics +-n, grid (omega, species,
// nmaxR + 1), 256 threads over the ppar columns.  A launch of its own: every
// harmonic's flags in parallel (they are a chain of nine dependent loads per
// column, which the trapezoid pass had in front of each of its harmonics).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_rel_flags(const ProbDev *__restrict__ probp, int nom,
                                                   const double2 *__restrict__ om_in,
                                                   const int *__restrict__ active,
                                                   int *__restrict__ flags,
                                                   const int *__restrict__ pidx, int nstride) {
  const int iom = blockIdx.x, s = blockIdx.y, an = blockIdx.z;
  const ProbDev &Pd = pidx != nullptr ? probp[pidx[iom]] : *probp;
  if (s >= Pd.nspec) return;
  const SpecDev &S = Pd.sp[s];
  if (!S.rel || an > S.nmax_rel) return;
  if (!(active == nullptr || active[iom] != 0)) return;
  const int nspec = Pd.nspec, nperp = S.nperp, npar = S.npar;
  const double omr = om_in[iom].x;
  const double m = S.m, q = S.q, kpar = Pd.kpar;
  // the Gamma range of the (pperp, ppar) points (from the host's table):
  // p_res(Gamma) = (Gamma m Re w - n q)/kpar is linear in Gamma, so a harmonic
  // whose p_res over [gmin, gmax] stays clear of [ppar(0), ppar(npar)] (with a
  // margin far above rounding) has no point in a resonant cell and skips the
  // scan below
  const double gmin = S.rel_gmin, gmax = S.rel_gmax;
  auto clear_of = [&](int n) {
#pragma clang fp contract(off)
    const double nq = 1.0 * n * q;
    const double pa = (gmin * m * omr - nq) / kpar, pb = (gmax * m * omr - nq) / kpar;
    const double lo = S.ppar[0], hi = S.ppar[npar];
    const double tol = 1e-9 * (fabs(pa) + fabs(pb) + fabs(lo) + fabs(hi));
    return fmax(pa, pb) < lo - tol || fmin(pa, pb) > hi + tol;
  };
  const bool scan0 = !clear_of(an), scan1 = an > 0 && !clear_of(-an);
  int hit0 = 0, hit1 = 0;
  if ((scan0 || scan1) && S.rel_gmono) {
    // Along a ppar column, Gamma does not decrease with iperp, and the
    // reference's pr = (Gamma m Re w - n q)/kpar (each operation rounded,
    // hence monotone in Gamma) is monotone along it: the column has a point
    // with ppar(ia) <= pr < ppar(ia+1) iff the first point past the cell's
    // near end (found by bisection on that same pr) is short of its far end
    for (int ia = threadIdx.x; ia < npar; ia += 256) {
      const double lo = S.ppar[ia], hi = S.ppar[ia + 1];
      const double *gc = S.gam_pp + ia;
      for (int h = 0; h < 2; ++h) {
        if (h == 0 ? !scan0 : !scan1) continue;
        const double nq = 1.0 * (h == 0 ? an : -an) * q;
        auto pr = [&](int ip) {
#pragma clang fp contract(off)
          return (gc[(size_t)ip * (npar + 1)] * m * omr - nq) / kpar;
        };
        const bool up = pr(0) <= pr(nperp);
        // the first ip whose pr is past the near end: pr >= lo (rising) or
        // pr < hi (falling); nperp + 1 if none
        int a0 = 0, a1 = nperp + 1;
        while (a0 < a1) {
          const int mid = (a0 + a1) >> 1;
          const double v = pr(mid);
          if (up ? (v >= lo) : (v < hi))
            a1 = mid;
          else
            a0 = mid + 1;
        }
        if (a0 <= nperp) {
          const double v = pr(a0);
          if (lo <= v && hi > v) (h == 0 ? hit0 : hit1) = 1;
        }
      }
    }
  } else if (scan0 || scan1) {
#pragma clang fp contract(off)
    const double nq0 = 1.0 * an * q, nq1 = 1.0 * -an * q;
    const double ik = 1.0 / kpar;
    // point pt = ip npar + ia, (ip, ia) stepped without a division per point.
    // The test takes the reference's quotient pr = (g m Re w - n q)/kpar;
    // the product by 1/kpar is within 4 ulp of it, so where that product is
    // farther than 1e-14 (relative) from both cell ends the test's answer
    // is the same, and only the other points take the division
    int ip = (int)threadIdx.x / npar, ia = (int)threadIdx.x % npar;
    for (int pt = threadIdx.x; pt < (nperp + 1) * npar; pt += 256) {
      const double g = S.gam_pp[ip * (npar + 1) + ia];
      const double lo = S.ppar[ia], hi = S.ppar[ia + 1];
      const double gm = g * m * omr;
      if (scan0) {
        const double num = gm - nq0;
        double pr = num * ik;
        const double tol = 1e-14 * fabs(pr);
        if (fabs(pr - lo) <= tol || fabs(pr - hi) <= tol) pr = num / kpar;
        if (lo <= pr && hi > pr) hit0 = 1;
      }
      if (scan1) {
        const double num = gm - nq1;
        double pr = num * ik;
        const double tol = 1e-14 * fabs(pr);
        if (fabs(pr - lo) <= tol || fabs(pr - hi) <= tol) pr = num / kpar;
        if (lo <= pr && hi > pr) hit1 = 1;
      }
      for (ia += 256; ia >= npar; ia -= npar) ++ip;
    }
  }
  const int found0 = __syncthreads_or(hit0);
  const int found1 = __syncthreads_or(hit1);
  if (threadIdx.x == 0) {
    int *f = flags + ((size_t)iom * nspec + s) * nstride + Pd.nmaxR;
    f[an] = found0;
    if (an > 0) f[-an] = found1;
  }
}

// ---------------------------------------------------------------------------
// k_rel_nonres: the integrate() terms of the non-resonant harmonics among
// {+-2g, +-(2g + 1)}; grid (omega, species, B (nmaxR/2 + 1)), harmonic group
// g = blockIdx.z / B, part blockIdx.z % B of its grid points.
//
// FP64-VALU bound.  A lane owns one ppar column and walks down the pperp rows,
// so that the row's moment factors a_j(n) are wave-uniform scalars and the
// powers of ppar are applied once at the end: a point costs, per harmonic, its
// reciprocal and three complex multiply-adds a_j r.  The four harmonics of a
// workgroup share each point's loads and numerator, and one reciprocal of the
// product of their |den|^2 (two Newton steps for the four of them).  The
// wavefronts of the B workgroups of a group take (column tile, row chunk)
// items: B = 8 keeps a single omega's solve short, B = 1 writes the fewest
// partial slots.  48 omegas of a 200 x 400 grid, nmax 30: 1035 us with one
// point per lane and two harmonics per pass, 338 us in this form with one
// 1024-thread workgroup per group and a reciprocal per harmonic, 251 us now.
// ---------------------------------------------------------------------------
constexpr int NRW = 4;  // wavefronts of a k_rel_nonres workgroup

// The 24 values v of every lane summed over the wavefront, a half of the
// values handed over per step instead of all of them at each of six steps:
// lane l then holds the totals of values sum24_at(l) + {0, 1, 2}
template <int N, int D>
__device__ __forceinline__ void wave_halve(double *v, int lane) {
  const bool up = (lane & D) != 0;
#pragma unroll
  for (int i = 0; i < N / 2; ++i) {
    const double send = up ? v[i] : v[i + N / 2], keep = up ? v[i + N / 2] : v[i];
    v[i] = keep + __shfl_xor(send, D, 64);
  }
}
__device__ __forceinline__ void wave_sum24(double *v, int lane) {
  wave_halve<24, 32>(v, lane);
  wave_halve<12, 16>(v, lane);
  wave_halve<6, 8>(v, lane);
#pragma unroll
  for (int d = 4; d > 0; d >>= 1)
#pragma unroll
    for (int k = 0; k < 3; ++k) v[k] += __shfl_xor(v[k], d, 64);
}
__device__ __forceinline__ int sum24_at(int lane) {
  return ((lane >> 5) & 1) * 12 + ((lane >> 4) & 1) * 6 + ((lane >> 3) & 1) * 3;
}

__global__ __launch_bounds__(64 * NRW) __attribute__((amdgpu_waves_per_eu(4))) void k_rel_nonres(
    const ProbDev *__restrict__ probp, int nom, const double2 *__restrict__ om_in,
    const int *__restrict__ active, double2 *__restrict__ chiR, double2 *__restrict__ lowR,
    const int *__restrict__ flags, int nstride, int B) {
  __shared__ double red[NRW][48];
  const int iom = blockIdx.x, s = blockIdx.y, g = blockIdx.z / B, part = blockIdx.z % B;
  const ProbDev &Pd = *probp;
  if (s >= Pd.nspec) return;
  const SpecDev &S = Pd.sp[s];
  if (!S.rel) return;
  if (!(active == nullptr || active[iom] != 0)) return;
  const int nspec = Pd.nspec, nperp = S.nperp, npar = S.npar, nmax = S.nmax_rel;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int na = 2 * g, nb = 2 * g + 1;
  double2 *out = chiR + ((size_t)((int)blockIdx.z * nspec + s) * 6) * nom + iom;
  // harmonic h: +na, -na, +nb, -nb
  const int *fl = flags + ((size_t)iom * nspec + s) * nstride + Pd.nmaxR;
  bool use[4];
  use[0] = na <= nmax && fl[na] == 0;
  use[1] = na <= nmax && na > 0 && fl[-na] == 0;
  use[2] = nb <= nmax && fl[nb] == 0;
  use[3] = nb <= nmax && fl[-nb] == 0;
  double2 *low = (lowR != nullptr && g == 0)
                     ? lowR + (((size_t)part * nom + iom) * nspec + s) * 18
                     : nullptr;
  if (!use[0] && !use[1] && !use[2] && !use[3]) {
    if (threadIdx.x < 6) out[(size_t)threadIdx.x * nom] = make_double2(0.0, 0.0);
    if (low && threadIdx.x < 18) low[threadIdx.x] = make_double2(0.0, 0.0);
    return;
  }
  const double2 ov = om_in[iom];
  const double omr = ov.x, omi = ov.y;
  const double m = S.m, q = S.q, kpar = Pd.kpar;
  const double nqa = (1.0 * na) * q, nqb = (1.0 * nb) * q;
  // the one reciprocal needs the product of four |den|^2 to be a double: |den|
  // below 1e38, of which an omega beyond about 1e37 is short (its sums are finite)
  const double dmax = S.rel_gmax * m * (fabs(omr) + fabs(omi)) + fabs(nqb) +
                      fabs(kpar) * fmax(fabs(S.ppar[0]), fabs(S.ppar[npar]));
  const bool all4 = use[0] && use[1] && use[2] && use[3] && dmax < 1e38;
  typedef const __attribute__((address_space(4))) double *cptr;
  // (a pair past nmax is never used; its table pointer stays in range)
  const cptr ata = (cptr)(S.atab + (size_t)(na <= nmax ? na : 0) * (nperp + 1) * ATAB_STRIDE);
  const cptr atb = (cptr)(S.atab + (size_t)(nb <= nmax ? nb : 0) * (nperp + 1) * ATAB_STRIDE);
  const cptr pperp = (cptr)S.pperp;
  const int NT = (npar - 1 + 63) / 64;                      // column tiles
  const int C = max(1, min(NRW * B / NT, nperp - 1));      // row chunks
  const int rows = (nperp - 1 + C - 1) / C;
  double tot[4][3];  // this lane's totals: products 6 l5 + 3 l4 + {0, 1, 2} of each harmonic
#pragma unroll
  for (int h = 0; h < 4; ++h) tot[h][0] = tot[h][1] = tot[h][2] = 0.0;
#pragma unroll 1
  for (int it = part * NRW + wv; it < NT * C; it += NRW * B) {
    const int tile = it % NT, ch = it / NT;
    const int ia = 1 + tile * 64 + lane;
    const bool in = ia <= npar - 1;
    const int ic = in ? ia : npar - 1;
    const double p2 = S.ppar[ic];
    const double wa = in ? ((ia == 1 || ia == npar - 1) ? 1.0 : 2.0) : 0.0;
    const int r0 = 1 + ch * rows, r1 = min(r0 + rows - 1, nperp - 1);
    if (r0 > r1) continue;  // (the last chunk of a short grid)
    cd acc[4][3];
#pragma unroll
    for (int h = 0; h < 4; ++h)
#pragma unroll
      for (int j = 0; j < 3; ++j) acc[h][j] = mk(0.0, 0.0);
    const double kp2 = kpar * p2;
    auto add = [&](double inv, cd num, double dre, double dim, double a1, double a2, double a3,
                   cd *ac) {
      // num / den as num conj(den) / |den|^2 (|den| is O(1) here: no scaling needed)
      const cd r = mk((num.re * dre + num.im * dim) * inv, (num.im * dre - num.re * dim) * inv);
      ac[0].re = __builtin_fma(a1, r.re, ac[0].re);
      ac[0].im = __builtin_fma(a1, r.im, ac[0].im);
      ac[1].re = __builtin_fma(a2, r.re, ac[1].re);
      ac[1].im = __builtin_fma(a2, r.im, ac[1].im);
      ac[2].re = __builtin_fma(a3, r.re, ac[2].re);
      ac[2].im = __builtin_fma(a3, r.im, ac[2].im);
    };
    auto column = [&](auto all4_c) {
      size_t o = (size_t)r0 * (npar + 1) + ic;
      // the next row's table values are loaded while the current row is summed
      double gn = S.gam_pp[o], d1n = S.df1[o], d2n = S.df2[o];
#pragma unroll 1
      for (int ip = r0; ip <= r1; ++ip) {
        const double gg = gn, d1 = d1n, d2 = d2n;
        if (ip < r1) {
          o += npar + 1;
          gn = S.gam_pp[o];
          d1n = S.df1[o];
          d2n = S.df2[o];
        }
        const double w = (ip == nperp - 1 ? wa : 2.0 * wa) * q;
        const double gm = gg * m;
        const double A = (kpar * rcp_d(gm)) * (pperp[ip] * d2 - p2 * d1);
        const cd num = mk(w * (omr * d1 + A), w * (omi * d1));
        const double base = gm * omr - kp2, dim = gm * omi, dim2 = dim * dim;
        const double a1 = ata[ip * ATAB_STRIDE], a2 = ata[ip * ATAB_STRIDE + 1],
                     a3 = ata[ip * ATAB_STRIDE + 2];
        const double b1 = atb[ip * ATAB_STRIDE], b2 = atb[ip * ATAB_STRIDE + 1],
                     b3 = atb[ip * ATAB_STRIDE + 2];
        const double d0 = base - nqa, e0 = base + nqa, f0 = base - nqb, g0 = base + nqb;
        if constexpr (decltype(all4_c)::value) {
          const double x0 = __builtin_fma(d0, d0, dim2), x1 = __builtin_fma(e0, e0, dim2);
          const double x2 = __builtin_fma(f0, f0, dim2), x3 = __builtin_fma(g0, g0, dim2);
          const double x01 = x0 * x1, x23 = x2 * x3;
          const double iv = rcp_d(x01 * x23);
          const double i01 = iv * x23, i23 = iv * x01;
          add(i01 * x1, num, d0, dim, a1, a2, a3, acc[0]);
          add(i01 * x0, num, e0, dim, a1, a2, a3, acc[1]);
          add(i23 * x3, num, f0, dim, b1, b2, b3, acc[2]);
          add(i23 * x2, num, g0, dim, b1, b2, b3, acc[3]);
        } else {
          if (use[0]) add(rcp_d(__builtin_fma(d0, d0, dim2)), num, d0, dim, a1, a2, a3, acc[0]);
          if (use[1]) add(rcp_d(__builtin_fma(e0, e0, dim2)), num, e0, dim, a1, a2, a3, acc[1]);
          if (use[2]) add(rcp_d(__builtin_fma(f0, f0, dim2)), num, f0, dim, b1, b2, b3, acc[2]);
          if (use[3]) add(rcp_d(__builtin_fma(g0, g0, dim2)), num, g0, dim, b1, b2, b3, acc[3]);
        }
      }
    };
    if (all4)
      column(std::true_type{});
    else
      column(std::false_type{});
    // the column's powers of ppar, then the lanes summed, a harmonic at a time
    // (its registers only)
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      const cd c1 = acc[h][0], c2 = acc[h][1], c3 = acc[h][2];
      const double pq = p2 * p2;
      double v[12] = {c1.re,      c1.im,      p2 * c1.re, p2 * c1.im, pq * c1.re, pq * c1.im,
                      c2.re,      c2.im,      c3.re,      c3.im,      p2 * c3.re, p2 * c3.im};
      wave_halve<12, 32>(v, lane);
      wave_halve<6, 16>(v, lane);
#pragma unroll
      for (int d = 8; d > 0; d >>= 1)
#pragma unroll
        for (int k = 0; k < 3; ++k) v[k] += __shfl_xor(v[k], d, 64);
#pragma unroll
      for (int k = 0; k < 3; ++k) tot[h][k] += v[k];
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if ((lane & 15) == 0) {
    const int o = ((lane >> 5) & 1) * 6 + ((lane >> 4) & 1) * 3;
#pragma unroll
    for (int h = 0; h < 4; ++h)
#pragma unroll
      for (int k = 0; k < 3; ++k) red[wv][12 * h + o + k] = tot[h][k];
  }
  __syncthreads();
  // the wavefronts summed in order, times the T constants, then the harmonics
  const double scale = 2.0 * PI_R * S.dpperp * S.dppar_abs * 0.25;
  if (threadIdx.x < 6) {
    const int k = threadIdx.x;
    const int ak = acc_of_mode(k);
    cd res = mk(0.0, 0.0);
    for (int h = 0; h < 4; ++h) {
      const int n = h == 0 ? na : h == 1 ? -na : h == 2 ? nb : -nb;
      cd v = mk(0.0, 0.0);
      if (use[h] && !(n == 0 && (k == 0 || k == 3 || k == 4))) {
        cd t = mk(0.0, 0.0);
        for (int w = 0; w < NRW; ++w)
          t = t + mk(red[w][12 * h + 2 * ak], red[w][12 * h + 2 * ak + 1]);
        v = (scale * t) * tconst_r(Pd, S, n, k);
      }
      res = res + v;
      if (low && !(h == 1)) low[6 * (n + 1) + k] = make_double2(v.re, v.im);  // (h = 1 is -0)
    }
    out[(size_t)k * nom] = make_double2(res.re, res.im);
  }
}

// ---------------------------------------------------------------------------
// the (Gamma, pparbar) grid: integrate_res_rel
// ---------------------------------------------------------------------------
struct RelCtx {
  const SpecDev *S;
  cd om;
  int n, npb;
  double vA, kpar, kperp;
  bool kn;
  // per-call factors of the integrand (not of any decision), so that a grid
  // point costs one reciprocal: vA/kpar, n q vA/(kpar m), 1/zbar, 1/dpparbar
  double vak, nterm, izbar, idpb;
};

// funct_g_rel's interpolation cell (ALPS_fns_rel.f90:918-999) from the raw
// cell k holding x (pb[k] <= x < pb[k+1], -2 if none): the index close whose
// neighbours close-1, close+1 it interpolates
__device__ __forceinline__ int rel_close_of(const double *f0, int npb, int k) {
  int close = k;
  if (close + 1 >= 0 && close + 1 <= npb && f0[close + 1] <= -1.0) close = close - 1;
  if (close - 1 >= 0 && close - 1 <= npb && f0[close - 1] <= -1.0) close = close + 1;
  if (close >= npb - 1) close = npb - 2;
  if (close <= 1) close = 2;
  return close;
}

// the same at real x of row ig, with the search for its raw cell
__device__ int rel_close(const SpecDev &S, int ig, double x) {
  const int npb = S.npb, row = ig * (npb + 1);
  const double *pb = S.pbrel + row;
  int raw = -2;
  {
#pragma clang fp contract(off)
    // the last ip in [0, npb-1] with pb[ip] <= x < pb[ip+1] (increasing row)
    int k = (int)floor((x - pb[0]) / S.rel_dpb);
    if (k >= -1 && k <= npb) {
      k = max(0, min(k, npb - 1));
      while (k > 0 && pb[k] > x) --k;
      while (k < npb - 1 && pb[k + 1] <= x) ++k;
      if (pb[k + 1] > x && pb[k] <= x) raw = k;
    }
  }
  if (x == pb[npb]) return npb - 2;
  return rel_close_of(S.f0rel + row, npb, raw);
}

// The moment products of int_T_rel and resU_rel / funct_g_rel at grid point pt
// for +-an: a1 = J^2, a2 = J'^2 pperpbar^2, a3 = J J' pperpbar (even in the
// sign of n) and num = pref (om df/dGamma + (kpar/vA) df/dpparbar)
struct RelNode {
  double a1, a2, a3, pb;
  cd num;
};
__device__ __forceinline__ RelNode rel_node(const SpecDev &S, int an, size_t np, int pt, cd om,
                                            double kv) {
  RelNode N;
  const double g = S.grel[pt], pb = S.pbrel[pt];
  const double2 d = S.dfrel[pt];
  const double b = S.relbes[(size_t)an * np + pt];
  const double bn = S.relbes[(size_t)(an + 1) * np + pt];
  const double bP = an > 0 ? 0.5 * (S.relbes[(size_t)(an - 1) * np + pt] - bn) : -bn;
  double pp2;
  {
#pragma clang fp contract(off)
    pp2 = g * g - 1.0 - pb * pb;
  }
  N.a1 = b * b;
  N.a2 = (bP * bP) * pp2;
  N.a3 = (b * bP) * sqrt(pp2);
  N.pb = pb;
  N.num = mk(S.rel_pref * (om.re * d.x + kv * d.y), S.rel_pref * (om.im * d.x));
  return N;
}
// acc += c times the node's mode products {a1, pb a1, pb^2 a1, a2, a3, pb a3} num
__device__ __forceinline__ void rel_node_add(const RelNode &N, cd c, cd acc[6]) {
  const cd v = c * N.num;
  const cd u1 = N.a1 * v, u3 = N.a3 * v;
  acc[0] = acc[0] + u1;
  acc[1] = acc[1] + N.pb * u1;
  acc[2] = acc[2] + (N.pb * N.pb) * u1;
  acc[3] = acc[3] + N.a2 * v;
  acc[4] = acc[4] + u3;
  acc[5] = acc[5] + N.pb * u3;
}

// One row of one harmonic as integrate_resU_rel (ALPS_fns_rel.f90:516-719)
// lays it out: trapezoid ranges [a1, b1] and [a2, b2] (none where a > b), and
// the principal-value window around ipres (pv) with its ladder
struct RelRow {
  int a1, b1, a2, b2, ipres, pv, bad, nt;  // pv 2: ladder points outside the window's cells
  double dR, dI, cap;          // the resonance and the half width of its ladder
  double sm, ism, corr, ct;    // its step, the step's reciprocal, the tiny rest's correction and step
};
// The ladder points of principal_integral_rel: x_j = dR + t_j up to dR + cap,
// their mirror images 2 dR - x_j, and the tiny rest above dR + cap, each
// rounded as the reference rounds it
struct RelLadder {
  double dR, cap, sm, ct, corr;
  int nri, nt;
  __device__ __forceinline__ double up(int j) const {
#pragma clang fp contract(off)
    return j == 0 ? dR : (j == nri ? dR + cap : dR + sm * j);
  }
  __device__ __forceinline__ double dn(int j) const {
#pragma clang fp contract(off)
    return 2.0 * dR - up(j);
  }
  __device__ __forceinline__ double tiny(int k) const {
#pragma clang fp contract(off)
    return k == 0 ? dR + cap : dR + cap + ct * k;
  }
};
__device__ __forceinline__ RelRow rel_row(const SpecDev &S, cd om, int n, double vA, double kpar,
                                          int pos, int nri, int ig) {
#pragma clang fp contract(off)
  RelRow R;
  const int npb = S.npb;
  const double dpb = S.rel_dpb;
  const double *pb2 = S.pbrel + 2 * (npb + 1);  // row 2 of pparbar_rel
  int ipres = 0;
  bool found = false;
  double pr;
  const double g1 = S.grel[ig * (npb + 1) + 1];
  const double tr = g1 * om.re - (1.0 * n) * S.q / S.m;
  pr = tr * vA / kpar;
  if ((pr * pr) <= (g1 * g1 - 1.0)) {
    // the unique ip in [1, npb-2] with pb2[ip] <= pr < pb2[ip+1]
    if (pb2[1] <= pr && pr < pb2[npb - 1]) {
      int k = 1 + (int)((pr - pb2[1]) / dpb);
      k = max(1, min(k, npb - 2));
      while (k > 1 && pb2[k] > pr) --k;
      while (k < npb - 2 && pb2[k + 1] <= pr) ++k;
      ipres = k;
      found = true;
    }
  }
  for (int ip = 0; ip <= pos; ++ip) {
    if (pr >= (pb2[0] - dpb * ip) && pr < (pb2[0] - dpb * (ip - 1))) {
      ipres = -ip;
      found = true;
    }
    if (pr >= (pb2[npb - 1] + dpb * ip) && pr < (pb2[npb - 1] + dpb * (ip + 1))) {
      ipres = npb - 1 + ip;
      found = true;
    }
  }
  const int2 lim = S.rowlim[ig];
  const int lower = lim.x, upper = lim.y;
  int int_start, int_end, lowerlimit, upperlimit;
  R.bad = R.ipres = R.pv = R.nt = 0;
  R.dR = R.dI = R.cap = R.sm = R.ism = R.corr = R.ct = 0.0;
  if (found) {
    int_start = lower;
    int_end = upper;
    lowerlimit = ipres - pos;
    upperlimit = ipres + pos + 1;
    if (ipres >= 0 && ipres <= npb)
      if (fabs(pr - pb2[ipres]) > (0.5 * dpb)) upperlimit = upperlimit + 1;
    if (lowerlimit < lower && upperlimit > upper) {
      R.bad = 1;
      R.a1 = R.a2 = 1;
      R.b1 = R.b2 = 0;
      return R;
    }
    if (lowerlimit <= lower) {
      int_start = 1;
      lowerlimit = 0;
      upperlimit = lower;
    } else if (upperlimit >= upper) {
      lowerlimit = upper;
      upperlimit = npb;
      int_end = npb - 1;
    }
  } else {
    int_start = lower;
    lowerlimit = upper;
    int_end = npb - 1;
    upperlimit = npb;
  }
  R.a1 = int_start;
  R.b1 = lowerlimit;
  R.a2 = upperlimit;
  R.b2 = int_end;
  R.ipres = ipres;
  R.pv = (found && lowerlimit >= int_start && upperlimit <= int_end) ? 1 : 0;
  if (R.pv) {
    // principal_integral_rel (ALPS_fns_rel.f90:724-913)
    const double G = S.grel[ig * (npb + 1) + ipres];
    const double gr = G * om.re * vA / kpar, gi = G * om.im * vA / kpar;
    R.dR = gr - (1.0 * n) * (S.q / S.m) * vA / kpar;
    R.dI = gi;
    R.cap = R.dR - S.pbrel[1 * (npb + 1) + ipres - pos];
    R.sm = R.cap / (1.0 * nri);
    R.ism = 1.0 / R.sm;
    const double *pbr = S.pbrel + ig * (npb + 1);
    const double base = pbr[upperlimit] - R.dR - R.cap;
    R.nt = R.sm > 0.0 ? (int)(base / R.sm) : 0;
    R.corr = R.nt > 0 ? (base / (1.0 * R.nt)) / R.sm : 0.0;
    R.ct = R.corr * R.sm;
    // the cells ipres-P-2 .. ipres+P+3 hold every ladder point of a row of the
    // usual table (each row the same uniform pparbar grid); a row with points
    // outside them adds its points one by one
    const RelLadder L{R.dR, R.cap, R.sm, R.ct, R.corr, nri, R.nt};
    const int k0 = max(ipres - pos - 2, 0), k1 = min(ipres + pos + 3, npb - 1);
    const double xl = L.dn(nri), xt = L.tiny(max(R.nt, 0));
    const double lo = pbr[k0], hi = pbr[k1 + 1];
    if (!(R.sm > 0.0 && xl >= lo && xt < hi && R.dR - dpb >= lo && R.dR + dpb < hi)) R.pv = 2;
  }
  return R;
}

// the first j in [0, top + 1] at which the monotone test past(j) holds, from a
// guess (top + 1: none)
template <typename F>
__device__ __forceinline__ int first_past(double guess, int top, F past) {
  int j = guess > 0.0 ? (guess < (double)top ? (int)guess : top) : 0;
  while (j > 0 && past(j - 1)) --j;
  while (j <= top && !past(j)) ++j;
  return j;
}

// ---------------------------------------------------------------------------
// k_rel_res: integrate_res_rel of the resonant harmonics +-n; grid (omega,
// species, RS (nmaxR + 1)), n = blockIdx.z / RS, part blockIdx.z % RS of its
// Gamma rows.
//
// A row's sum is sum_i c_i (num T)(i) over its pparbar nodes: the trapezoid
// weight over the denominator outside the principal-value window, and inside
// it the ladder's weights times funct_g_rel's interpolation weights (linear in
// the node values).  A wavefront:
//  * decides 32 of its rows at once, a lane per (row, sign);
//  * takes the ladders of two rows: a lane per (row, sign, raw pparbar cell)
//    finds the ladder points of its cell by the comparisons a search would
//    make and sums their weights.  Since t r = w + i dI r for a weight r =
//    w/(t - i dI), the cell's interpolation sum follows from the sums of r and
//    w (S, W), as in the non-relativistic ladder;
//  * sums the nodes of the two rows: a lane per node, every table read
//    coalesced, +n and -n sharing the node's table products.
// One lane per Gamma row, walking its nodes and ladder (k_rel_res_ord), reads 64
// different cache lines per load: 803 us for 48 omegas (200 x 400, 100 x 200
// grids), against 188 us for this form with a row at a time and 154 us with two.
// RS = 4 parts keep a single
// omega's solve short; RS = 1 writes the fewest partial slots.
// ---------------------------------------------------------------------------
constexpr int RSW = 4;         // wavefronts of a k_rel_res workgroup
constexpr int RCELL_MAX = 38;  // raw cells ipres-P-2 .. ipres+P+3, P <= 16

__device__ __forceinline__ int rl_i(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ double rl_d(double v, int l) {
  union {
    double d;
    int i[2];
  } u;
  u.d = v;
  u.i[0] = __builtin_amdgcn_readlane(u.i[0], l);
  u.i[1] = __builtin_amdgcn_readlane(u.i[1], l);
  return u.d;
}
__device__ __forceinline__ void rel_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// two rows' cells: per (row, sign) slot and cell c0 (re, im), cp (re, im) and
// the cell's interpolation index
struct RelCells {
  double c[4][RCELL_MAX][4];
  int close[4][RCELL_MAX];
};

__global__ __launch_bounds__(64 * RSW) __attribute__((amdgpu_waves_per_eu(2))) void k_rel_res(
    const ProbDev *__restrict__ probp, int nom, const double2 *__restrict__ om_in,
    const int *__restrict__ active, double2 *__restrict__ chiR, double2 *__restrict__ lowR,
    const int *__restrict__ flags, int slot0, int low0, int *__restrict__ err, int nstride,
    int RS) {
  __shared__ RelCells cells[RSW];
  __shared__ double red[RSW][24];
  const int iom = blockIdx.x, s = blockIdx.y, an = blockIdx.z / RS, part = blockIdx.z % RS;
  const ProbDev &Pd = *probp;
  if (s >= Pd.nspec) return;
  const SpecDev &S = Pd.sp[s];
  if (!S.rel) return;
  if (!(active == nullptr || active[iom] != 0)) return;
  const int nspec = Pd.nspec;
  double2 *out = chiR + ((size_t)((slot0 + (int)blockIdx.z) * nspec + s) * 6) * nom + iom;
  double2 *low = (lowR != nullptr && an <= 1)
                     ? lowR + (((size_t)(low0 + part) * nom + iom) * nspec + s) * 18
                     : nullptr;
  const int *fl = flags + ((size_t)iom * nspec + s) * nstride + Pd.nmaxR;
  const bool inr = an <= S.nmax_rel;
  const bool fP = inr && fl[an] != 0, fM = inr && an > 0 && fl[-an] != 0;
  if (!fP && !fM) {
    if (threadIdx.x < 6) {
      out[(size_t)threadIdx.x * nom] = make_double2(0.0, 0.0);
      if (low) low[6 * (1 + an) + threadIdx.x] = low[6 * (1 - an) + threadIdx.x] = make_double2(0.0, 0.0);
    }
    return;
  }
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  RelCells &Cw = cells[wv];
  const double2 ov = om_in[iom];
  const cd om = mk(ov.x, ov.y);
  const int npb = S.npb, ng = S.ng, pos = Pd.P, nri = Pd.NRI;
  const double vA = Pd.vA, kpar = Pd.kpar, Tlim = Pd.Tlim;
  const double vak = vA / kpar, kv = kpar / vA;
  const double nterm = (1.0 * an) * S.q * vA / (kpar * S.m);
  const double dpb = S.rel_dpb, hinv = 0.5 / dpb;
  const size_t np = (size_t)(ng + 1) * (npb + 1);
  const int NC = 2 * pos + 6;
  const int step = RSW * RS;  // the wavefront's rows: 1 + part RSW + wv, and every step-th after
  cd acc[2][6];
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int k = 0; k < 6; ++k) acc[g][k] = mk(0.0, 0.0);
  int bad = 0;
  for (int b0 = 1 + part * RSW + wv; b0 <= ng - 1; b0 += 32 * step) {
    // lane 2r + sign decides row b0 + r step of that sign
    RelRow R;
    R.a1 = R.a2 = 1;
    R.b1 = R.b2 = 0;
    R.ipres = R.pv = R.bad = R.nt = 0;
    R.dR = R.dI = R.cap = R.sm = R.ism = R.corr = R.ct = 0.0;
    const int igl = b0 + (lane >> 1) * step;
    if (igl <= ng - 1 && ((lane & 1) ? fM : fP))
      R = rel_row(S, om, (lane & 1) ? -an : an, vA, kpar, pos, nri, igl);
    bad |= R.bad;
    for (int r = 0; r < 32; r += 2) {
      if (b0 + r * step > ng - 1) break;
      // the ladders of rows r, r + 1: slots 2 (row) + sign
      bool plain = true;  // every cell interpolates around itself
      if (rl_i(R.pv, 2 * r) | rl_i(R.pv, 2 * r + 1) | rl_i(R.pv, 2 * r + 2) | rl_i(R.pv, 2 * r + 3)) {
        // the Lorentz sum of the analytic form (|dI| <= Tlim), lanes over its points
        double sph[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const double dI = rl_d(R.dI, 2 * r + g);
          if (rl_i(R.pv, 2 * r + g) != 1 || fabs(dI) > Tlim) continue;
          const RelLadder L{rl_d(R.dR, 2 * r + g), rl_d(R.cap, 2 * r + g), rl_d(R.sm, 2 * r + g),
                            0.0, 0.0, nri, 0};
          double v = 0.0;
          for (int j = 1 + lane; j <= nri; j += 64) {
            const double t = L.up(j) - L.dR, t2 = t * t;
            v += (j == nri ? 2.0 : 4.0) * (t2 / (t2 + dI * dI));
          }
#pragma unroll
          for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d, 64);
          sph[g] = v;
        }
        bool off = false;
        for (int it0 = 0; it0 < 4 * NC; it0 += 64) {
          const int it = min(it0 + lane, 4 * NC - 1);
          const int g = it / NC, ci = it - g * NC, src = 2 * r + g;
          // (every lane takes part in the shuffles, also those past the last item:
          // the rows they hold are other lanes' sources)
          const int pvs = __shfl(R.pv, src, 64);
          const bool on = it0 + lane < 4 * NC && pvs == 1;
          RelLadder L;
          L.dR = __shfl(R.dR, src, 64);
          L.cap = __shfl(R.cap, src, 64);
          L.sm = __shfl(R.sm, src, 64);
          L.ct = __shfl(R.ct, src, 64);
          L.corr = __shfl(R.corr, src, 64);
          L.nri = nri;
          L.nt = __shfl(R.nt, src, 64);
          const double dR = L.dR, dI = __shfl(R.dI, src, 64), ism = __shfl(R.ism, src, 64);
          const int k = __shfl(R.ipres, src, 64) - pos - 2 + ci;
          double c0r = 0.0, c0i = 0.0, cpr = 0.0, cpi = 0.0;
          int close = 0;
          if (on && k >= 0 && k <= npb - 1) {
            const int row = (b0 + (r + (g >> 1)) * step) * (npb + 1);
            const double lo = S.pbrel[row + k], hi = S.pbrel[row + k + 1];
            close = rel_close_of(S.f0rel + row, npb, k);
            const double pc = S.pbrel[row + close];
            const double dI2 = dI * dI;
            double Sr = 0.0, Si = 0.0, W = 0.0, Mr = 0.0, V = 0.0, Mi = 0.0;
            if (fabs(dI) > Tlim) {
              // the points in the cell of the ladder and of its mirror image
              const int ja = first_past((lo - dR) * ism, nri, [&](int j) { return L.up(j) >= lo; });
              const int jb = first_past((hi - dR) * ism, nri, [&](int j) { return L.up(j) >= hi; });
              const int ma = first_past((dR - hi) * ism, nri, [&](int j) { return L.dn(j) < hi; });
              const int mb = first_past((dR - lo) * ism, nri, [&](int j) { return L.dn(j) < lo; });
              for (int j = ja; j < jb; ++j) {
                const double t = L.up(j) - dR, w = (j == 0 || j == nri) ? 1.0 : 2.0;
                const double inv = w * rcp_d(__builtin_fma(t, t, dI2));
                Sr = __builtin_fma(t, inv, Sr);
                Si += inv;
                W += w;
              }
              for (int j = ma; j < mb; ++j) {
                const double t = L.up(j) - dR, w = (j == 0 || j == nri) ? 1.0 : 2.0;
                const double inv = w * rcp_d(__builtin_fma(t, t, dI2));
                Mr = __builtin_fma(t, inv, Mr);
                Mi += inv;
                V += w;
              }
            } else {
              // 2 sum gprimetr t^2/(t^2 + dI^2), gprimetr the difference of g
              // at dR +- dpparbar, and the residue at dR (times 1/smdelta)
              const double f =
                  (g == 0 ? sph[0] : g == 1 ? sph[1] : g == 2 ? sph[2] : sph[3]) / (2.0 * dpb);
              auto point = [&](double x, cd wt) {
                if (!(lo <= x && x < hi)) return;
                const double fr = (x - pc) * hinv;
                c0r += wt.re;
                c0i += wt.im;
                cpr += fr * wt.re;
                cpi += fr * wt.im;
              };
              point(dR + dpb, mk(f, 0.0));
              point(dR - dpb, mk(-f, 0.0));
              if (dI != 0.0) point(dR, mk(0.0, (dI > 0.0 ? 2.0 : -2.0) * PI_R * ism));
            }
            if (L.nt > 0 && L.tiny(L.nt) >= lo && L.tiny(0) < hi) {
              const double xe = dR + L.cap;
              const double ict = rcp_d(L.ct);
              const int ja = first_past((lo - xe) * ict, L.nt, [&](int j) { return L.tiny(j) >= lo; });
              const int jb = first_past((hi - xe) * ict, L.nt, [&](int j) { return L.tiny(j) >= hi; });
              for (int j = ja; j < jb; ++j) {
                const double t = L.tiny(j) - dR,
                             w = ((j == 0 || j == L.nt) ? 1.0 : 2.0) * L.corr;
                const double inv = w * rcp_d(__builtin_fma(t, t, dI2));
                Sr = __builtin_fma(t, inv, Sr);
                Si += inv;
                W += w;
              }
            }
            const cd z = mk(dR - pc, dI), Sc = mk(Sr, dI * Si), Mc = mk(Mr, -dI * Mi);
            const cd zS = z * Sc, zM = z * Mc;
            c0r += Sc.re - Mc.re;
            c0i += Sc.im - Mc.im;
            cpr += hinv * ((W + zS.re) + (V - zM.re));
            cpi += hinv * (zS.im - zM.im);
            off = off || (close != k && (c0r != 0.0 || c0i != 0.0 || cpr != 0.0 || cpi != 0.0));
          }
          if (it0 + lane < 4 * NC) {
            Cw.c[g][ci][0] = c0r;
            Cw.c[g][ci][1] = c0i;
            Cw.c[g][ci][2] = cpr;
            Cw.c[g][ci][3] = cpi;
            Cw.close[g][ci] = close;
          }
        }
        plain = !__any(off);
        rel_wave_sync();
      }
      // the rows' nodes
#pragma unroll 1
      for (int rr = r; rr < r + 2; ++rr) {
        const int ig = b0 + rr * step;
        if (ig > ng - 1) break;
        const int row = ig * (npb + 1);
        const double wr = ig <= ng - 2 ? 2.0 : 1.0;
        int a1[2], e1[2], a2[2], e2[2], kb[2], pv[2];
        double fw[2];  // the window's factor wr smdelta
        int lo = npb + 1, hi = -1;
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          a1[g] = rl_i(R.a1, 2 * rr + g);
          e1[g] = rl_i(R.b1, 2 * rr + g);
          a2[g] = rl_i(R.a2, 2 * rr + g);
          e2[g] = rl_i(R.b2, 2 * rr + g);
          kb[g] = rl_i(R.ipres, 2 * rr + g) - pos - 2;
          pv[g] = rl_i(R.pv, 2 * rr + g);
          fw[g] = wr * rl_d(R.sm, 2 * rr + g);
          if (a1[g] <= e1[g]) lo = min(lo, a1[g]), hi = max(hi, e1[g]);
          if (a2[g] <= e2[g]) lo = min(lo, a2[g]), hi = max(hi, e2[g]);
          if (pv[g] == 1) lo = min(lo, max(kb[g] - 1, 0)), hi = max(hi, min(kb[g] + NC, npb));
        }
        for (int i = lo + lane; i <= hi; i += 64) {
          const RelNode N = rel_node(S, an, np, row + i, om, kv);
          const double G = S.grel[row + i];
          const double gre = G * om.re * vak, gim = G * om.im * vak;
          const double wt = wr * dpb;
#pragma unroll
          for (int g = 0; g < 2; ++g) {
            cd c = mk(0.0, 0.0);
            bool in = false;
            const bool r1 = i >= a1[g] && i <= e1[g], r2 = i >= a2[g] && i <= e2[g];
            if (r1 || r2) {
              const int ra = r1 ? a1[g] : a2[g], rb = r1 ? e1[g] : e2[g];
              const double w = (i == ra || i == rb) ? wt : 2.0 * wt;
              const double dre = (N.pb - gre) + (g ? -nterm : nterm), dim = -gim;
              const double inv = w * rcp_d(dre * dre + dim * dim);
              c = mk(-(dre * inv), dim * inv);
              in = true;
            }
            const int d = i - kb[g];
            if (pv[g] == 1 && d >= -1 && d <= NC) {
              const int sl = 2 * (rr - r) + g;
              cd w = mk(0.0, 0.0);
              if (plain) {
                if (d >= 0 && d < NC) w = w + mk(Cw.c[sl][d][0], Cw.c[sl][d][1]);
                if (d >= 1) w = w + mk(Cw.c[sl][d - 1][2], Cw.c[sl][d - 1][3]);
                if (d + 1 < NC) w = w - mk(Cw.c[sl][d + 1][2], Cw.c[sl][d + 1][3]);
              } else {
                for (int ci = 0; ci < NC; ++ci) {
                  const int e = i - Cw.close[sl][ci];
                  if (e == 0) w = w + mk(Cw.c[sl][ci][0], Cw.c[sl][ci][1]);
                  if (e == 1) w = w + mk(Cw.c[sl][ci][2], Cw.c[sl][ci][3]);
                  if (e == -1) w = w - mk(Cw.c[sl][ci][2], Cw.c[sl][ci][3]);
                }
              }
              if (w.re != 0.0 || w.im != 0.0) {
                c = c - fw[g] * w;
                in = true;
              }
            }
            // (a node without a weight may lie outside the cone, where the
            // products are not numbers)
            if (in) rel_node_add(N, c, acc[g]);
          }
        }
        // ladder points outside the cells: each by its own search
#pragma unroll 1
        for (int g = 0; g < 2; ++g) {
          if ((g ? pv[1] : pv[0]) != 2) continue;
          const int src = 2 * rr + g;
          const RelLadder L{rl_d(R.dR, src), rl_d(R.cap, src), rl_d(R.sm, src), rl_d(R.ct, src),
                            rl_d(R.corr, src), nri, rl_i(R.nt, src)};
          const double dR = L.dR, dI = rl_d(R.dI, src);
          const double f = wr * L.sm;
          cd e[6];
          for (int k = 0; k < 6; ++k) e[k] = mk(0.0, 0.0);
          auto point = [&](double x, cd wt) {
            const int close = rel_close(S, ig, x);
            const double fr = (x - S.pbrel[row + close]) * hinv;
            const cd c = -f * wt;
            rel_node_add(rel_node(S, an, np, row + close, om, kv), c, e);
            rel_node_add(rel_node(S, an, np, row + close + 1, om, kv), fr * c, e);
            rel_node_add(rel_node(S, an, np, row + close - 1, om, kv), -fr * c, e);
          };
          double sph = 0.0;
          for (int j = lane; j <= nri; j += 64) {
            const double x = L.up(j), t = x - dR, w = (j == 0 || j == nri) ? 1.0 : 2.0;
            if (fabs(dI) > Tlim) {
              const double inv = w * rcp_d(t * t + dI * dI);
              point(x, mk(t * inv, dI * inv));
              point(L.dn(j), mk(-t * inv, dI * inv));
            } else if (j >= 1) {
              sph += 2.0 * w * ((t * t) / (t * t + dI * dI));
            }
          }
          if (fabs(dI) <= Tlim) {
            for (int d = 32; d > 0; d >>= 1) sph += __shfl_xor(sph, d, 64);
            if (lane == 0) {
              point(dR + dpb, mk(sph / (2.0 * dpb), 0.0));
              point(dR - dpb, mk(-sph / (2.0 * dpb), 0.0));
              if (dI != 0.0) point(dR, mk(0.0, (dI > 0.0 ? 2.0 : -2.0) * PI_R / L.sm));
            }
          }
          for (int k = lane; k <= L.nt && L.nt > 0; k += 64) {
            const double x = L.tiny(k), t = x - dR,
                         w = ((k == 0 || k == L.nt) ? 1.0 : 2.0) * L.corr;
            const double inv = w * rcp_d(t * t + dI * dI);
            point(x, mk(t * inv, dI * inv));
          }
          for (int k = 0; k < 6; ++k) {
            if (g)
              acc[1][k] = acc[1][k] + e[k];
            else
              acc[0][k] = acc[0][k] + e[k];
          }
        }
      }
      rel_wave_sync();  // the next rows write the cells again
    }
  }
  if (bad) err[0] = 8;
  double tot[24];
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      tot[12 * g + 2 * k] = acc[g][k].re;
      tot[12 * g + 2 * k + 1] = acc[g][k].im;
    }
  wave_sum24(tot, lane);
  if ((lane & 7) == 0) {
    const int o = sum24_at(lane);
#pragma unroll
    for (int k = 0; k < 3; ++k) red[wv][o + k] = tot[k];
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    const int k = threadIdx.x;
    const int ak = acc_of_mode(k);
    const double iz = 1.0 / S.rel_zbar, kp = Pd.kperp_norm != 0 ? 1.0 : Pd.kperp;
    cd res = mk(0.0, 0.0);
    for (int g = 0; g < (an > 0 ? 2 : 1); ++g) {
      const int n = g ? -an : an;
      cd v = mk(0.0, 0.0);
      if ((g ? fM : fP) && !(n == 0 && (k == 0 || k == 3 || k == 4))) {
        cd t = mk(0.0, 0.0);
        for (int w = 0; w < RSW; ++w)
          t = t + mk(red[w][12 * g + 2 * ak], red[w][12 * g + 2 * ak + 1]);
        // int_T_rel's constants (ALPS_fns_rel.f90:1340-1366)
        const double nn = 1.0 * n;
        cd C;
        switch (k) {
          case 0: C = mk((1.0 * (n * n)) * (iz * iz), 0.0); break;
          case 1: C = mk(kp * kp, 0.0); break;
          case 2: C = mk(kp * kp, 0.0); break;
          case 3: C = mk(0.0, nn * kp * iz); break;
          case 4: C = mk(nn * kp * iz, 0.0); break;
          default: C = mk(0.0, -(kp * kp)); break;
        }
        v = ((t * C) * S.rel_dg) * 0.25;
      }
      res = res + v;
      if (low) low[6 * (n + 1) + k] = make_double2(v.re, v.im);
    }
    out[(size_t)k * nom] = make_double2(res.re, res.im);
  }
}

// workgroup sum of a complex value (blockDim.x = 256 or 64), result to all
template <int NT>
__device__ __forceinline__ cd block_sum(cd v, double *lds) {
  for (int o = 32; o > 0; o >>= 1) {
    v.re += __shfl_xor(v.re, o, 64);
    v.im += __shfl_xor(v.im, o, 64);
  }
  if constexpr (NT == 64) return v;
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) {
    lds[2 * w] = v.re;
    lds[2 * w + 1] = v.im;
  }
  __syncthreads();
  cd t = mk(0.0, 0.0);
  for (int i = 0; i < NT / 64; ++i) t = t + mk(lds[2 * i], lds[2 * i + 1]);
  return t;
}

// ---------------------------------------------------------------------------
// The served form of the relativistic sums (the root server): each sum is
// taken in one fixed order, whatever the batch, and a solve's end point depends
// on that order.  Where a ladder's end falls on a pparbar node, funct_g_rel's
// cell is decided by the last bit of omega and D steps by 1e-11 or so; a solve
// that is rounded differently there stops elsewhere in the |D| < D_threshold set
// (1e-8 to 1e-7 of the root), or not at all.  k_rel_nonres / k_rel_res above
// order their sums by their split, so the server keeps these.
//
// k_rel_nonres_ord: the integrate() terms of two neighbouring harmonics, grid
// (omega, species, nmaxR + 1), 256 threads over the points, each harmonic in a
// partial slot of its own (k_assemble adds them in groups of every fourth
// harmonic).  One workgroup per pair, not per sixteen harmonics: a pass of one
// to some tens of omegas is the length of one workgroup.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_rel_nonres_ord(
    const ProbDev *__restrict__ probp, int nom, const double2 *__restrict__ om_in,
    double2 *__restrict__ chiR, const int *__restrict__ flags, const int *__restrict__ pidx,
    int nstride) {
  __shared__ double lds[16];
  const int iom = blockIdx.x, s = blockIdx.y;
  const ProbDev &Pd = probp[pidx[iom]];
  if (s >= Pd.nspec) return;
  const SpecDev &S = Pd.sp[s];
  if (!S.rel) return;
  const int nspec = Pd.nspec, nperp = S.nperp, npar = S.npar, nmax = S.nmax_rel;
  const int z0 = 2 * blockIdx.z, z1 = z0 + 1;  // slots of the harmonics n0, n1
  const int n0 = z0 - Pd.nmaxR, n1 = n0 + 1;
  const int *fl = flags + ((size_t)iom * nspec + s) * nstride;
  const bool do0 = n0 >= -nmax && n0 <= nmax && fl[z0] == 0;
  const bool do1 = n1 >= -nmax && n1 <= nmax && fl[z1] == 0;
  for (int h = 0; h < 2; ++h)
    if (z0 + h < nstride && !(h == 0 ? do0 : do1) && threadIdx.x < 6)
      chiR[((size_t)((z0 + h) * nspec + s) * 6 + threadIdx.x) * nom + iom] = make_double2(0.0, 0.0);
  if (!do0 && !do1) return;
  const double2 ov = om_in[iom];
  const cd om = mk(ov.x, ov.y);
  const double m = S.m, q = S.q, kpar = Pd.kpar;
  const double scale = 2.0 * PI_R * S.dpperp * S.dppar_abs * 0.25;
  const double *at0 = S.atab + (size_t)(n0 < 0 ? -n0 : n0) * (nperp + 1) * ATAB_STRIDE;
  const double *at1 = S.atab + (size_t)(n1 < 0 ? -n1 : n1) * (nperp + 1) * ATAB_STRIDE;
  cd acc0[6], acc1[6];
  for (int k = 0; k < 6; ++k) acc0[k] = acc1[k] = mk(0.0, 0.0);
  // one harmonic's terms of the point: resU (ALPS_fns.f90:1587-1592) with the
  // point's Gamma, num / den as num conj(den) / |den|^2 with one reciprocal
  // (|den| is O(1) here: no scaling needed), times the int_T moments
  auto add = [&](const double *at, int ip, double w, cd num, double dre, double dim, double p2,
                 cd acc[6]) {
    const double inv = w * rcp1_d(dre * dre + dim * dim);
    const cd r = mk((num.re * dre + num.im * dim) * inv, (num.im * dre - num.re * dim) * inv);
    const double a1 = at[ip * ATAB_STRIDE + 0], a2 = at[ip * ATAB_STRIDE + 1],
                 a3 = at[ip * ATAB_STRIDE + 2];
    const cd u1 = a1 * r, u3 = a3 * r;
    acc[0] = acc[0] + u1;
    acc[1] = acc[1] + p2 * u1;
    acc[2] = acc[2] + (p2 * p2) * u1;
    acc[3] = acc[3] + a2 * r;
    acc[4] = acc[4] + u3;
    acc[5] = acc[5] + p2 * u3;
  };
  // point pt = (ip - 1)(npar - 1) + ia - 1, stepped as above
  int ip = 1 + (int)threadIdx.x / (npar - 1), ia = 1 + (int)threadIdx.x % (npar - 1);
  for (int pt = threadIdx.x; pt < (nperp - 1) * (npar - 1); pt += 256) {
    const double w = (ip == nperp - 1 ? 1.0 : 2.0) * ((ia == 1 || ia == npar - 1) ? 1.0 : 2.0);
    const size_t o = (size_t)ip * (npar + 1) + ia;
    const double g = S.gam_pp[o], d1 = S.df1[o], d2 = S.df2[o];
    const double p1 = S.pperp[ip], p2 = S.ppar[ia];
    const double A = (kpar * rcp_d(g * m)) * (p1 * d2 - p2 * d1);
    const cd num = mk(q * (om.re * d1 + A), q * (om.im * d1));
    const double base = (g * m) * om.re - kpar * p2, dim = (g * m) * om.im;
    if (do0) add(at0, ip, w, num, base - (1.0 * n0) * q, dim, p2, acc0);
    if (do1) add(at1, ip, w, num, base - (1.0 * n1) * q, dim, p2, acc1);
    for (ia += 256; ia > npar - 1; ia -= npar - 1) ++ip;
  }
  for (int h = 0; h < 2; ++h) {
    const int n = h == 0 ? n0 : n1;
    if (h == 0 ? !do0 : !do1) continue;
    const cd *acc = h == 0 ? acc0 : acc1;
    cd v[6];
    for (int k = 0; k < 6; ++k) {
      const cd t = block_sum<256>(acc[acc_of_mode(k)], lds);
      v[k] = (scale * t) * tconst_r(Pd, S, n, k);
    }
    if (n == 0) v[0] = v[3] = v[4] = mk(0.0, 0.0);
    if (threadIdx.x == 0) {
      double2 *o = chiR + ((size_t)((z0 + h) * nspec + s) * 6) * nom + iom;
      for (int k = 0; k < 6; ++k) o[(size_t)k * nom] = make_double2(v[k].re, v[k].im);
    }
  }
}

// a / b for complex b of moderate size: a conj(b) / |b|^2 with one reciprocal
__device__ __forceinline__ cd cdiv_r(cd a, cd b) {
  const double inv = rcp_d(b.re * b.re + b.im * b.im);
  return mk((a.re * b.re + a.im * b.im) * inv, (a.im * b.re - a.re * b.im) * inv);
}

// bessel and besselP of int_T_rel (ALPS_fns_rel.f90:1324-1338) from the J table
__device__ __forceinline__ void rel_bessel(const RelCtx &C, int pt, double &b, double &bP) {
  const SpecDev &S = *C.S;
  const int n = C.n;
  const size_t np = (size_t)(S.ng + 1) * (S.npb + 1);
  auto J = [&](int k) { return S.relbes[(size_t)k * np + pt]; };
  b = n < 0 ? m1p(n) * J(-n) : J(n);
  if (n >= 1)
    bP = 0.5 * (J(n - 1) - J(n + 1));
  else if (n < -1)
    bP = 0.5 * ((m1p(n - 1) * J(-(n - 1))) - (m1p(n + 1) * J(-(n + 1))));
  else if (n == 0)
    bP = -J(1);
  else
    bP = 0.5 * (J(2) - J(0));
}

// int_T_rel for the six modes at grid point pt (ALPS_fns_rel.f90:1340-1366)
__device__ __forceinline__ void int_T_rel6(const RelCtx &C, int pt, cd T[6]) {
  const SpecDev &S = *C.S;
  const double g = S.grel[pt], pb = S.pbrel[pt];
  double pperpbar;
  {
#pragma clang fp contract(off)
    pperpbar = sqrt(g * g - 1.0 - pb * pb);
  }
  double b, bP;
  rel_bessel(C, pt, b, bP);
  const double iz = C.izbar, kp = C.kperp, nn = 1.0 * C.n;
  if (C.kn) {
    T[0] = mk(1.0 * (C.n * C.n) * b * b * (iz * iz), 0.0);
    T[1] = mk(bP * bP * pperpbar * pperpbar, 0.0);
    T[2] = mk(b * b * (pb * pb), 0.0);
    T[3] = mk(0.0, nn * b * bP * pperpbar * iz);
    T[4] = mk(nn * b * b * pb * iz, 0.0);
    T[5] = mk(0.0, -(b * bP * pb * pperpbar));
  } else {
    T[0] = mk(1.0 * (C.n * C.n) * b * b * (iz * iz), 0.0);
    T[1] = mk(kp * kp * bP * bP * pperpbar * pperpbar, 0.0);
    T[2] = mk(kp * kp * b * b * (pb * pb), 0.0);
    T[3] = mk(0.0, nn * kp * b * bP * pperpbar * iz);
    T[4] = mk(nn * kp * b * b * pb * iz, 0.0);
    T[5] = mk(0.0, -(kp * kp * b * bP * pb * pperpbar));
  }
}

// the numerator of resU_rel and funct_g_rel: pref * (om df/dGamma + (kpar/vA) df/dpparbar)
__device__ __forceinline__ cd rel_num(const RelCtx &C, int pt) {
  const double2 d = C.S->dfrel[pt];
  const cd t = mk(C.om.re * d.x + (C.kpar / C.vA) * d.y, C.om.im * d.x);
  return C.S->rel_pref * t;
}

// funct_g_rel's interpolation cell (ALPS_fns_rel.f90:918-999): the index
// close of row ig whose neighbours close-1, close+1 it interpolates at real x
// (*lo, *hi): the bounds pb[k] <= x < pb[k+1] of the cell the search found,
// or (+inf, -inf) if none: any x' in [lo, hi) gives the same index
__device__ int rel_close_in(const RelCtx &C, int ig, double x, double *lo = nullptr,
                            double *hi = nullptr) {
  const SpecDev &S = *C.S;
  const int npb = C.npb, row = ig * (npb + 1);
  const double *pb = S.pbrel + row;
  int close = -2;
  double cl = 1.0 / 0.0, ch = -1.0 / 0.0;
  {
#pragma clang fp contract(off)
    // the last ip in [0, npb-1] with pb[ip] <= x < pb[ip+1] (increasing row)
    int k = (int)floor((x - pb[0]) / S.rel_dpb);
    if (k >= -1 && k <= npb) {
      k = max(0, min(k, npb - 1));
      while (k > 0 && pb[k] > x) --k;
      while (k < npb - 1 && pb[k + 1] <= x) ++k;
      if (pb[k + 1] > x && pb[k] <= x) {
        close = k;
        cl = pb[k];
        ch = pb[k + 1];
      }
    }
  }
  if (lo) {
    *lo = cl;
    *hi = ch;
  }
  const double *f0 = S.f0rel + row;
  if (close + 1 >= 0 && close + 1 <= npb && f0[close + 1] <= -1.0) close = close - 1;
  if (close - 1 >= 0 && close - 1 <= npb && f0[close - 1] <= -1.0) close = close + 1;
  if (x == pb[npb]) close = npb - 2;
  if (close >= npb - 1) close = npb - 2;
  if (close <= 1) close = 2;
  return close;
}

// funct_g_rel (ALPS_fns_rel.f90:918-999) for the six modes at real pparbar x
// of row ig: g(close) + (x - pparbar(close)) (g(close+1) - g(close-1)) /
// (2 dpparbar), g = -(rel_num T), with one node's T values live at a time
__device__ void funct_g_rel6(const RelCtx &C, int ig, double x, cd g[6]) {
  const SpecDev &S = *C.S;
  const int npb = C.npb, row = ig * (npb + 1);
  const double *pb = S.pbrel + row;
  const int close = rel_close_in(C, ig, x);
  const double f = 0.5 * ((x - pb[close]) * C.idpb);
  cd T[6];
  int_T_rel6(C, row + close, T);
  const cd nc = rel_num(C, row + close);
  for (int k = 0; k < 6; ++k) g[k] = -1.0 * (nc * T[k]);
  int_T_rel6(C, row + close + 1, T);
  const cd np_ = -f * rel_num(C, row + close + 1);
  for (int k = 0; k < 6; ++k) g[k] = g[k] + np_ * T[k];
  int_T_rel6(C, row + close - 1, T);
  const cd nm = f * rel_num(C, row + close - 1);
  for (int k = 0; k < 6; ++k) g[k] = g[k] + nm * T[k];
}

// the resU_rel * int_T_rel terms of point ip of row ig, weight w, into acc
__device__ __forceinline__ void rel_point(const RelCtx &C, int ig, int ip, double w, cd acc[6]) {
  const SpecDev &S = *C.S;
  const int pt = ig * (C.npb + 1) + ip;
  const double G = S.grel[pt], PB = S.pbrel[pt];
  const cd gom = mk(G * C.om.re * C.vak, G * C.om.im * C.vak);
  const cd den = mk((PB - gom.re) + C.nterm, -gom.im);
  const cd U = -1.0 * cdiv_r(rel_num(C, pt), den);
  cd T[6];
  int_T_rel6(C, pt, T);
  for (int k = 0; k < 6; ++k) acc[k] = acc[k] + w * (U * T[k]);
}

// funct_g_rel is linear in the values g_k(node) = -(rel_num T_k) at the three
// nodes of its cell (close - 1, close, close + 1): g(x) = g(close) +
// f (g(close+1) - g(close-1)), f = 0.5 (x - pparbar(close)) / dpparbar.  A
// weighted sum of g over a monotone ladder of x is therefore the sum over the
// cells it passes of three coefficients times the node values: RelCell holds
// the open cell's coefficients, and the node values are evaluated once per
// cell, when the ladder leaves it.
struct RelCell {
  int close;  // -1: empty
  cd cm, c0, cp;
  // the last cell search of this ladder: any x in [klo, khi) has index kc,
  // whose pparbar is kp (klo > khi: none yet)
  double klo, khi, kp;
  int kc;
};

__device__ __forceinline__ void rel_node_g(const RelCtx &C, int pt, cd g[6]) {
  cd T[6];
  int_T_rel6(C, pt, T);
  const cd nm = rel_num(C, pt);
  for (int k = 0; k < 6; ++k) g[k] = -1.0 * (nm * T[k]);
}

// Cells that a row's ladders have left, in the order they were left: the lanes
// (rows) leave theirs at different points of the ladder, and evaluating three
// nodes there ran that code for almost every point of the wavefront's ladder;
// the queued cells are evaluated together (rel_drain), in the same order (a
// served stream of 96 solves: 1285 us a launch, 757 us with the queue)
constexpr int RELQ = 16;
struct RelQueue {
  int n;
  int close[RELQ];
  cd cm[RELQ], c0[RELQ], cp[RELQ];
};

// one cell's three coefficients, times f, into acc
__device__ __forceinline__ void rel_cell_eval(const RelCtx &C, int ig, int close, cd m, cd z, cd p,
                                              cd acc[6], double f) {
  const int pt = ig * (C.npb + 1) + close;
  cd g[6];
  rel_node_g(C, pt, g);
  const cd c0 = f * z, cp = f * p, cm = f * m;
  for (int k = 0; k < 6; ++k) acc[k] = acc[k] + c0 * g[k];
  rel_node_g(C, pt + 1, g);
  for (int k = 0; k < 6; ++k) acc[k] = acc[k] + cp * g[k];
  rel_node_g(C, pt - 1, g);
  for (int k = 0; k < 6; ++k) acc[k] = acc[k] + cm * g[k];
}

__device__ __forceinline__ void rel_drain(const RelCtx &C, int ig, RelQueue &q, cd acc[6],
                                          double f) {
#pragma unroll 1
  for (int i = 0; i < q.n; ++i)
    rel_cell_eval(C, ig, q.close[i], q.cm[i], q.c0[i], q.cp[i], acc, f);
  q.n = 0;
}

// the open cell to the queue
__device__ __forceinline__ void rel_cell_flush(const RelCtx &C, int ig, RelCell &cc, RelQueue &q,
                                               cd acc[6], double f) {
  if (cc.close < 0) return;
  if (q.n == RELQ) rel_drain(C, ig, q, acc, f);
  q.close[q.n] = cc.close;
  q.cm[q.n] = cc.cm;
  q.c0[q.n] = cc.c0;
  q.cp[q.n] = cc.cp;
  q.n += 1;
  cc.close = -1;
  cc.cm = cc.c0 = cc.cp = mk(0.0, 0.0);
}

// add wt g(x) through the cell cache (a cell leaving it goes into acc, times
// fac).  The ladder's x rise (or fall) monotonically: while x stays in the
// raw cell of the last search, the index is that search's.
__device__ __forceinline__ void rel_cell_add(const RelCtx &C, int ig, RelCell &cc, RelQueue &q,
                                             double x, cd wt, cd acc[6], double fac) {
  if (!(cc.klo <= x && x < cc.khi)) {
    cc.kc = rel_close_in(C, ig, x, &cc.klo, &cc.khi);
    cc.kp = C.S->pbrel[ig * (C.npb + 1) + cc.kc];
  }
  const int close = cc.kc;
  if (close != cc.close) {
    rel_cell_flush(C, ig, cc, q, acc, fac);
    cc.close = close;
  }
  const double f = 0.5 * ((x - cc.kp) * C.idpb);
  cc.c0 = cc.c0 + wt;
  cc.cp = cc.cp + f * wt;
  cc.cm = cc.cm - f * wt;
}

// principal_integral_rel (ALPS_fns_rel.f90:724-913), six modes, times smdelta
// and the row's trapezoid weight wr, added to acc (each term carries the
// factor, so that no partial sum of the row is held beside acc).  The ladder
// sums go through cell coefficients (RelCell), with the ladder's points
// visited in increasing x (the far end of each ladder after its inner
// points), so that each cell is opened once.
__device__ void principal_rel6(const RelCtx &C, int ig, int ipres, int upperlimit, double Tlim,
                               int pos, int nri, double wr, cd acc[6]) {
  const SpecDev &S = *C.S;
  const int row = ig * (C.npb + 1);
  double denomR, denomI, capDelta, smdelta;
  {
#pragma clang fp contract(off)
    const double G = S.grel[row + ipres];
    const double gr = G * C.om.re * C.vA / C.kpar, gi = G * C.om.im * C.vA / C.kpar;
    denomR = gr - (1.0 * C.n) * (S.q / S.m) * C.vA / C.kpar;
    denomI = gi;
    capDelta = denomR - S.pbrel[1 * (C.npb + 1) + ipres - pos];
    smdelta = capDelta / (1.0 * nri);
  }
  const double f = wr * smdelta;
  cd g[6], g2[6];
  RelQueue q;
  q.n = 0;
  RelCell up, dn;  // x = denomR + t (increasing) and its mirror 2 denomR - x (decreasing)
  up.close = dn.close = -1;
  up.cm = up.c0 = up.cp = dn.cm = dn.c0 = dn.cp = mk(0.0, 0.0);
  up.klo = dn.klo = 1.0 / 0.0;
  up.khi = dn.khi = -1.0 / 0.0;
  up.kc = dn.kc = 0;
  up.kp = dn.kp = 0.0;
  auto pv_pair = [&](double x, double wgt) {
    // wgt / (t - i denomI) and wgt / (t + i denomI), t = x - denomR: one
    // reciprocal, the second the conjugate of the first
    const double t = x - denomR;
    const double inv = wgt * rcp_d(t * t + denomI * denomI);
    const cd r = mk(t * inv, denomI * inv);
    rel_cell_add(C, ig, up, q, x, r, acc, f);
    rel_cell_add(C, ig, dn, q, 2.0 * denomR - x, mk(-r.re, r.im), acc, f);
  };
  if (fabs(denomI) > Tlim) {
    pv_pair(denomR, 1.0);
    for (int ip = 1; ip <= nri - 1; ++ip) {
      double x;
      {
#pragma clang fp contract(off)
        x = denomR + smdelta * ip;
      }
      pv_pair(x, 2.0);
    }
    pv_pair(denomR + capDelta, 1.0);
    rel_cell_flush(C, ig, up, q, acc, f);
    rel_cell_flush(C, ig, dn, q, acc, f);
  } else {
    funct_g_rel6(C, ig, denomR + S.rel_dpb, g);
    funct_g_rel6(C, ig, denomR - S.rel_dpb, g2);
    cd gp[6];
    for (int k = 0; k < 6; ++k) gp[k] = cdivr(g[k] - g2[k], 2.0 * S.rel_dpb);
    auto lorentz = [&](double x) {
      const double d = x - denomR;
      return (d * d) / (d * d + denomI * denomI);
    };
    {
      const double l = lorentz(denomR + capDelta);
      for (int k = 0; k < 6; ++k) acc[k] = acc[k] + (f * (2.0 * l)) * gp[k];
    }
    for (int ip = 1; ip <= nri - 1; ++ip) {
      double x;
      {
#pragma clang fp contract(off)
        x = denomR + smdelta * ip;
      }
      const double l = lorentz(x);
      for (int k = 0; k < 6; ++k) acc[k] = acc[k] + (f * ((2.0 * 2.0) * l)) * gp[k];
    }
    if (denomI != 0.0) {
      funct_g_rel6(C, ig, denomR, g);
      const double sg = denomI > 0.0 ? 1.0 : -1.0;
      for (int k = 0; k < 6; ++k)
        acc[k] = acc[k] + wr * timesI((sg * 2.0 * PI_R) * g[k]);  // (2 pi i g / smdelta) f
    }
  }
  int ntiny;
  double base;
  {
#pragma clang fp contract(off)
    base = S.pbrel[row + upperlimit] - denomR - capDelta;
    ntiny = (int)(base / smdelta);
  }
  if (ntiny > 0) {
    double correction;
    {
#pragma clang fp contract(off)
      correction = (base / (1.0 * ntiny)) / smdelta;
    }
    auto tiny = [&](double x, double wgt) {
      const double t = x - denomR;
      const double inv = (wgt * correction) * rcp_d(t * t + denomI * denomI);
      rel_cell_add(C, ig, up, q, x, mk(t * inv, denomI * inv), acc, f);
    };
    double x0, x1;
    {
#pragma clang fp contract(off)
      x0 = denomR + capDelta;
      x1 = denomR + capDelta + correction * smdelta * ntiny;
    }
    tiny(x0, 1.0);
    for (int ip = 1; ip <= ntiny - 1; ++ip) {
      double x;
      {
#pragma clang fp contract(off)
        x = denomR + capDelta + correction * smdelta * ip;
      }
      tiny(x, 2.0);
    }
    tiny(x1, 1.0);
    rel_cell_flush(C, ig, up, q, acc, f);
  }
  rel_drain(C, ig, q, acc, f);
}

// integrate_resU_rel (ALPS_fns_rel.f90:516-719) of row ig, six modes, times
// the row's trapezoid weight wr, added to acc (term by term); returns false,
// before adding anything, where the reference calls alps_error(8)
__device__ bool resU_row6(const RelCtx &C, int ig, int pos, int nri, double Tlim, double wr,
                          cd acc[6]) {
  const SpecDev &S = *C.S;
  const int npb = C.npb;
  const double dpb = S.rel_dpb;
  const double *pb2 = S.pbrel + 2 * (npb + 1);  // row 2 of pparbar_rel
  int ipres = 0;
  bool found = false;
  double pr;
  {
#pragma clang fp contract(off)
    const double g1 = S.grel[ig * (npb + 1) + 1];
    const double tr = g1 * C.om.re - (1.0 * C.n) * S.q / S.m;
    pr = tr * C.vA / C.kpar;
    if ((pr * pr) <= (g1 * g1 - 1.0)) {
      // the unique ip in [1, npb-2] with pb2[ip] <= pr < pb2[ip+1]
      if (pb2[1] <= pr && pr < pb2[npb - 1]) {
        int k = 1 + (int)((pr - pb2[1]) / dpb);
        k = max(1, min(k, npb - 2));
        while (k > 1 && pb2[k] > pr) --k;
        while (k < npb - 2 && pb2[k + 1] <= pr) ++k;
        ipres = k;
        found = true;
      }
    }
    for (int ip = 0; ip <= pos; ++ip) {
      if (pr >= (pb2[0] - dpb * ip) && pr < (pb2[0] - dpb * (ip - 1))) {
        ipres = -ip;
        found = true;
      }
      if (pr >= (pb2[npb - 1] + dpb * ip) && pr < (pb2[npb - 1] + dpb * (ip + 1))) {
        ipres = npb - 1 + ip;
        found = true;
      }
    }
  }
  const int2 lim = S.rowlim[ig];
  const int lower = lim.x, upper = lim.y;
  int int_start, int_end, lowerlimit, upperlimit;
  if (found) {
    int_start = lower;
    int_end = upper;
    lowerlimit = ipres - pos;
    upperlimit = ipres + pos + 1;
    if (ipres >= 0 && ipres <= npb) {
#pragma clang fp contract(off)
      if (fabs(pr - pb2[ipres]) > (0.5 * dpb)) upperlimit = upperlimit + 1;
    }
    if (lowerlimit < lower && upperlimit > upper) return false;
    if (lowerlimit <= lower) {
      int_start = 1;
      lowerlimit = 0;
      upperlimit = lower;
    } else if (upperlimit >= upper) {
      lowerlimit = upper;
      upperlimit = npb;
      int_end = npb - 1;
    }
  } else {
    int_start = lower;
    lowerlimit = upper;
    int_end = npb - 1;
    upperlimit = npb;
  }
  const double w1 = wr * dpb, w2 = 2.0 * w1;  // trapezoid weights times dpparbar and wr
  if (int_start <= lowerlimit) rel_point(C, ig, int_start, w1, acc);
  for (int ip = int_start + 1; ip <= lowerlimit - 1; ++ip) rel_point(C, ig, ip, w2, acc);
  if (int_start < lowerlimit) rel_point(C, ig, lowerlimit, w1, acc);
  if (upperlimit <= int_end) rel_point(C, ig, upperlimit, w1, acc);
  for (int ip = upperlimit + 1; ip <= int_end - 1; ++ip) rel_point(C, ig, ip, w2, acc);
  if (upperlimit < int_end) rel_point(C, ig, int_end, w1, acc);
  if (found && lowerlimit >= int_start && upperlimit <= int_end)
    principal_rel6(C, ig, ipres, upperlimit, Tlim, pos, nri, wr, acc);
  return true;
}

// complex ** integer by repeated squaring
__device__ __forceinline__ cd cpowi_d(cd a, int n) {
  cd pw = mk(1.0, 0.0), x = a;
  unsigned u = (unsigned)n;
  if (n == 0) return pw;
  for (;;) {
    if (u & 1u) pw = pw * x;
    u >>= 1;
    if (u)
      x = x * x;
    else
      break;
  }
  return pw;
}

// CBESSJ (ALPS_fns_rel.f90:1502-1553), 21 terms of the power series, for
// J_nu0, J_nu0+1, J_nu0+2 of the same z: the three
// orders share the powers (-z^2/4)^k, built by one product per term, and
// take the coefficients 1/(k! Gamma(nu+k+1)) from the table (requires
// nu0 + 2 < RFG_NU)
__device__ void cbessj3_d(const double *gtab, cd z, int nu0, cd J[3]) {
  const double *rf = gtab + GTAB_N + 21 + (size_t)nu0 * 21;
  const cd w = cdivr(-1.0 * (z * z), 4.0);
  cd t = mk(1.0, 0.0), s0 = mk(0.0, 0.0), s1 = s0, s2 = s0;
  for (int k = 0; k <= 20; ++k) {
    if (k > 0) t = t * w;
    s0 = s0 + t * rf[k];
    s1 = s1 + t * rf[21 + k];
    s2 = s2 + t * rf[42 + k];
  }
  const cd h = cdivr(z, 2.0);
  cd pw = cpowi_d(h, nu0);
  J[0] = pw * s0;
  pw = pw * h;
  J[1] = pw * s1;
  pw = pw * h;
  J[2] = pw * s2;
}

// int_T_res_rel (ALPS_fns_rel.f90:1374-1495), six modes, at complex pparbar p of row ig
__device__ void int_T_res_rel6(const RelCtx &C, const double *gtab, int ig, cd p, cd T[6]) {
  const SpecDev &S = *C.S;
  const double g = S.grel[ig * (C.npb + 1) + 1];
  const cd pp2 = p * p;
  const cd pperpbar = csqrtd(mk((g * g - 1.0) - pp2.re, -pp2.im));
  const cd z = S.rel_zfac * pperpbar;
  const int n = C.n;
  const int an = n < 0 ? -n : n;
  // the orders |n| - 1, |n|, |n| + 1 (0, 1, 2 for |n| <= 1)
  cd J[3];
  cbessj3_d(gtab, z, an >= 1 ? an - 1 : 0, J);
  cd b, bP;
  if (n >= 1) {
    b = J[1];
    bP = 0.5 * (J[0] - J[2]);
  } else if (n < -1) {
    b = m1p(n) * J[1];
    bP = 0.5 * ((m1p(n - 1) * J[2]) - (m1p(n + 1) * J[0]));
  } else if (n == 0) {
    b = J[0];
    bP = -1.0 * J[1];
  } else {  // n == -1
    b = m1p(n) * J[1];
    bP = 0.5 * (J[2] - J[0]);
  }
  const double zbar = S.rel_zbar, kp = C.kperp, nn = 1.0 * n;
  const double f = C.kn ? 1.0 : kp, f2 = C.kn ? 1.0 : kp * kp;
  T[0] = cdivr(1.0 * (n * n) * (b * b), zbar * zbar);
  T[1] = f2 * (((bP * bP) * pperpbar) * pperpbar);
  T[2] = f2 * ((b * b) * pp2);
  T[3] = cdivr(timesI((nn * f) * ((b * bP) * pperpbar)), zbar);
  T[4] = cdivr((nn * f) * ((b * b) * p), zbar);
  T[5] = -1.0 * timesI(f2 * (((b * bP) * p) * pperpbar));
}

// ---------------------------------------------------------------------------
// k_rel_res_ord / k_rel_landau: one resonant harmonic, grid (omega, species,
// 2 nmaxR + 1), 64 threads over the Gamma rows.  k_rel_res_ord (LANDAU = false):
// integrate_res_rel in the served form's order; k_rel_landau (LANDAU = true,
// served or not): landau_integrate_rel for Im om <= 0.  Two launches rather
// than one body: the Landau rows' Bessel series and continuation need registers
// that would hold the whole pass to one wavefront per SIMD.
// ---------------------------------------------------------------------------
template <bool LANDAU>
__device__ __forceinline__ void rel_res_body(const ProbDev *__restrict__ probp, int nom,
                                             const double2 *__restrict__ om_in,
                                             const int *__restrict__ active,
                                             double2 *__restrict__ chiR,
                                             double2 *__restrict__ lowR,
                                             const int *__restrict__ flags, int slot0, int low0,
                                             int *__restrict__ err,
                                             const int *__restrict__ pidx, int nstride) {
  const int iom = blockIdx.x, s = blockIdx.y;
  const ProbDev &Pd = pidx != nullptr ? probp[pidx[iom]] : *probp;
  if (s >= Pd.nspec) return;
  const SpecDev &S = Pd.sp[s];
  if (!S.rel) return;
  if (!(active == nullptr || active[iom] != 0)) return;
  const int nspec = Pd.nspec;
  const int n = (int)blockIdx.z - Pd.nmaxR;
  const int slot = slot0 + (int)blockIdx.z;
  double2 *low = (lowR != nullptr && n >= -1 && n <= 1)
                     ? lowR + (((size_t)low0 * nom + iom) * nspec + s) * 18 + 6 * (n + 1)
                     : nullptr;
  double2 *o = chiR + ((size_t)(slot * nspec + s) * 6) * nom + iom;
  const bool inr = (n >= -S.nmax_rel && n <= S.nmax_rel);
  const bool found = inr && flags[((size_t)iom * nspec + s) * nstride + blockIdx.z] != 0;
  if (!found) {
    if (threadIdx.x == 0)
      for (int k = 0; k < 6; ++k) {
        o[(size_t)k * nom] = make_double2(0.0, 0.0);
        if (low) low[k] = make_double2(0.0, 0.0);
      }
    return;
  }
  const double2 ov = om_in[iom];
  RelCtx C;
  C.S = &S;
  C.om = mk(ov.x, ov.y);
  C.n = n;
  C.npb = S.npb;
  C.vA = Pd.vA;
  C.kpar = Pd.kpar;
  C.kperp = Pd.kperp;
  C.kn = Pd.kperp_norm != 0;
  C.vak = C.vA / C.kpar;
  C.nterm = (1.0 * C.n) * S.q * C.vA / (C.kpar * S.m);
  C.izbar = 1.0 / S.rel_zbar;
  C.idpb = 1.0 / S.rel_dpb;
  const int ng = S.ng;
  cd acc[6];
  for (int k = 0; k < 6; ++k) acc[k] = mk(0.0, 0.0);
  int bad = 0;
  for (int ig = 1 + threadIdx.x; ig <= ng - 1; ig += 64) {
    if constexpr (!LANDAU) {
      const double wr = ig <= ng - 2 ? 2.0 : 1.0;
      if (!resU_row6(C, ig, Pd.P, Pd.NRI, Pd.Tlim, wr, acc)) bad = 1;
    } else if (C.om.im <= 0.0) {
      // landau_integrate_rel row (ALPS_fns_rel.f90:1065-1083)
      const double g1 = S.grel[ig * (S.npb + 1) + 1];
      cd pres;
      bool in;
      {
#pragma clang fp contract(off)
        const double a = g1 * C.om.re * C.vA / C.kpar, b = g1 * C.om.im * C.vA / C.kpar;
        pres = mk(a - (1.0 * n) * S.q * C.vA / (C.kpar * S.m), b);
        in = (pres.re * pres.re) <= (g1 * g1 - 1.0);
      }
      if (in) {
        const double h = (ig == ng - 1) ? 0.5 : 1.0;
        cd dfg;
        // (a relativistic species' fits are stored in the Maxwell form)
        if (ig == 1)
          dfg = cdivr(eval_fit_maxwell(S, ig + 1, pres) - eval_fit_maxwell(S, ig, pres), S.rel_dg);
        else
          dfg = cdivr(eval_fit_maxwell(S, ig + 1, pres) - eval_fit_maxwell(S, ig - 1, pres),
                      2.0 * S.rel_dg);
        const cd dfp = cdivr(eval_fit_maxwell(S, ig, mk(pres.re + S.rel_dpb, pres.im)) -
                                 eval_fit_maxwell(S, ig, mk(pres.re - S.rel_dpb, pres.im)),
                             2.0 * S.rel_dpb);
        const cd fac = h * (C.om * dfg + (C.kpar / C.vA) * dfp);
        cd T[6];
        int_T_res_rel6(C, Pd.gtab, ig, pres, T);
        for (int k = 0; k < 6; ++k) acc[k] = acc[k] - fac * T[k];
      }
    }
  }
  if (bad) err[pidx != nullptr ? iom : 0] = 8;  // with problem indices: one flag per omega
  cd v[6];
  for (int k = 0; k < 6; ++k) {
    const cd r = block_sum<64>(acc[k], nullptr);
    if constexpr (!LANDAU) {
      v[k] = (r * S.rel_dg) * 0.25;
    } else if (C.om.im <= 0.0) {
      const cd Lf = (((timesI(r) * S.rel_dg) * PI_R) * 2.0) * PI_R *
                    ((S.q * C.vA / (C.kpar * S.m)) * ((S.m / C.vA) * (S.m / C.vA) * (S.m / C.vA)));
      v[k] = (C.om.im < 0.0 ? 2.0 : 1.0) * Lf;
    } else {
      v[k] = mk(0.0, 0.0);
    }
  }
  if (n == 0) v[0] = v[3] = v[4] = mk(0.0, 0.0);
  if (threadIdx.x == 0) {
    for (int k = 0; k < 6; ++k) o[(size_t)k * nom] = make_double2(v[k].re, v[k].im);
    if (low)
      for (int k = 0; k < 6; ++k) low[k] = make_double2(v[k].re, v[k].im);
  }
}

// three wavefronts per SIMD (a few spilled registers; two by its register count)
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3))) void k_rel_res_ord(
    const ProbDev *__restrict__ probp, int nom, const double2 *__restrict__ om_in,
    double2 *__restrict__ chiR, const int *__restrict__ flags, int slot0, int *__restrict__ err,
    const int *__restrict__ pidx, int nstride) {
  rel_res_body<false>(probp, nom, om_in, nullptr, chiR, nullptr, flags, slot0, 0, err, pidx,
                      nstride);
}

__global__ __launch_bounds__(64) void k_rel_landau(
    const ProbDev *__restrict__ probp, int nom, const double2 *__restrict__ om_in,
    const int *__restrict__ active, double2 *__restrict__ chiR, double2 *__restrict__ lowR,
    const int *__restrict__ flags, int slot0, int low0, const int *__restrict__ pidx,
    int nstride) {
  rel_res_body<true>(probp, nom, om_in, active, chiR, lowR, flags, slot0, low0, nullptr, pidx,
                     nstride);
}

}  // namespace

// How the harmonics are split: B workgroups per harmonic group of
// k_rel_nonres, RS per harmonic of k_rel_res
RelSplit rel_split(int nom) {
  // A few omegas (secant steps) need the parts to fill the chip: one omega is
  // 16 x 8 + 31 x 4 workgroups at nmax 30.  A large batch fills it without, and
  // the parts would only add partial slots to write and sum.  Whole calls with
  // tensors at {8, 4}, {4, 2}, {1, 1}, us: 200 x 400 grid 1 omega 260, 291, 457;
  // 64: 658, 664, 820; 96: 892, 872, 935; 192: 1448, 1475, 1509; 256: 1896, 1885,
  // 1820; 512: 3484, 3310, 3210.  100 x 200: 1: 223, 222, 275; 64: 454, 393, 437;
  // 192: 822, 693, 729; 256: 1011, 952, 883.  The lines lie where the larger table
  // breaks even.
  if (nom <= 64) return {8, 4};
  if (nom <= 256) return {4, 2};
  return {1, 1};
}

// partial slots of chiR: B (nmaxR/2 + 1) of k_rel_nonres, then RS (nmaxR + 1)
// of k_rel_res and 2 nmaxR + 1 of k_rel_landau; slots of lowR: B + RS + 1
int rel_slots(RelSplit sp, int nmaxR) {
  return sp.B * (nmaxR / 2 + 1) + sp.RS * (nmaxR + 1) + 2 * nmaxR + 1;
}
int rel_low_slots(RelSplit sp) { return sp.B + sp.RS + 1; }

// nmaxR: the problem's largest relativistic nmax; flags [nom][nspec]
// [2 nmaxR + 1]; err [1]
hipError_t launch_rel(hipStream_t st, const ProbDev *prob, int nspec, int nmaxR, RelSplit sp,
                      int nom, const double2 *om, const int *active, double2 *chiR, double2 *lowR,
                      int *flags, int *err) {
  if (nom <= 0) return hipSuccess;
  const int nstride = 2 * nmaxR + 1, ng = sp.B * (nmaxR / 2 + 1), nh = nmaxR + 1;
  hipLaunchKernelGGL(k_rel_flags, dim3(nom, nspec, nh), dim3(256), 0, st, prob, nom, om, active,
                     flags, nullptr, nstride);
  hipLaunchKernelGGL(k_rel_nonres, dim3(nom, nspec, ng), dim3(64 * NRW), 0, st, prob, nom, om,
                     active, chiR, lowR, flags, nstride, sp.B);
  hipLaunchKernelGGL(k_rel_res, dim3(nom, nspec, sp.RS * nh), dim3(64 * RSW), 0, st, prob, nom, om,
                     active, chiR, lowR, flags, ng, sp.B, err, nstride, sp.RS);
  hipLaunchKernelGGL(k_rel_landau, dim3(nom, nspec, nstride), dim3(64), 0, st, prob, nom, om,
                     active, chiR, lowR, flags, ng + sp.RS * nh, sp.B + sp.RS, nullptr, nstride);
  return hipGetLastError();
}

// The served form: partial slots of chiR 2 nmaxR + 1 each (slot n + the
// problem's nmaxR) of k_rel_nonres_ord, k_rel_res_ord and k_rel_landau
int rel_ord_slots(int nmaxR) { return 3 * (2 * nmaxR + 1); }

// nmaxR: the largest of the batch's problems (each descriptor's own nmaxR
// offsets its flags and slots, so it may be smaller); flags [nom][nspec]
// [2 nmaxR + 1]; err [nom]
hipError_t launch_rel_ord(hipStream_t st, const ProbDev *prob, int nspec, int nmaxR, int nom,
                          const double2 *om, double2 *chiR, int *flags, int *err,
                          const int *pidx) {
  if (nom <= 0) return hipSuccess;
  const int nstride = 2 * nmaxR + 1;
  hipLaunchKernelGGL(k_rel_flags, dim3(nom, nspec, nmaxR + 1), dim3(256), 0, st, prob, nom, om,
                     nullptr, flags, pidx, nstride);
  hipLaunchKernelGGL(k_rel_nonres_ord, dim3(nom, nspec, nmaxR + 1), dim3(256), 0, st, prob, nom, om,
                     chiR, flags, pidx, nstride);
  hipLaunchKernelGGL(k_rel_res_ord, dim3(nom, nspec, nstride), dim3(64), 0, st, prob, nom, om, chiR,
                     flags, nstride, err, pidx, nstride);
  hipLaunchKernelGGL(k_rel_landau, dim3(nom, nspec, nstride), dim3(64), 0, st, prob, nom, om,
                     nullptr, chiR, nullptr, flags, 2 * nstride, 0, pidx, nstride);
  return hipGetLastError();
}
