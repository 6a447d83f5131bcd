// Landau tables of a batch: the pperp sums of landau_integrate
// (ALPS_fns.f90:1327-1452) as Taylor series in the complex resonant momentum.
//
// With om = (kpar p + n q)/m the row integrand of landau_integrate at p = p_res,
//   (q/|kpar|) [ (pperp dfpar - p dfperp) kpar/m + om dfperp ]
//   = (q/|kpar|) [ (kpar/m) pperp dfpar(p) + (n q/m) dfperp(p) ],
// depends on p alone, so its sum over the pperp rows with the weights
// h {J^2, pperp^2 J'^2, pperp J J'} is A_a(p) + n B_a(p), six analytic functions
// per |n|.  A batch of many omegas asks for them at many points of the same part
// of the p plane: every resonance lies within positions_principal steps of the
// ppar grid, at Im p = m Im om / kpar.  That part is covered by square tiles,
// and each tile gets the Taylor coefficients about its centre from the
// functions' values at LT_N points of the circle through its corners (their
// discrete Fourier transform).  A row then costs LT_J complex multiply-adds
// instead of three evaluations of the fit on every pperp row.
//
// A tile is used only where its series is as good as the sums: the last
// coefficients must have fallen to the rounding of the sums (a singularity of
// the continuation close by keeps them up), and no value may underflow or
// overflow near the circle.  Every other tile, and momenta outside the tiles,
// take the row sums.
//
// A tile whose series does not converge is cut into LT_SUB^2 smaller ones (the
// first LT_MAXP such tiles), which are closer to their centres.
//
// The tables are rebuilt by every batch that uses them: on 256 pperp rows a
// tile costs what about 60 row sums cost.
#include "alpsg_device.h"
#include "alpsg_fit.h"

namespace {

constexpr int LT_CH = 16;   // pperp rows evaluated at a time
constexpr int LT_TAIL = 4;  // coefficients past the last used one that are checked with it

// f of row ip at p, and in bad whether the value is too small or too large to be
// part of a series
__device__ __forceinline__ cd land_f(const SpecDev &S, int ip, cd p, bool &bad) {
  const cd f = eval_fit_kappa(S, ip, p);
  // (also NaN: a comparison with it is false)
  if (!(fabs(f.re) + fabs(f.im) > 1e-280) || !(fabs(f.re) + fabs(f.im) < 1e280)) bad = true;
  return f;
}

// grid (tiles, species), 256 threads; dynamic LDS, Q = 6 (nr + 1): the function
// values [Q][LT_N] complex, their rounding scales [Q][LT_N], the rows' weights
// [Q][LT_CH]
template <bool SUB>
__global__ __launch_bounds__(256) void k_land_build(const ProbDev *__restrict__ probp, LandTabs T) {
  extern __shared__ double2 Fq[];
  __shared__ double2 f0[LT_CH][LT_N], fd[LT_CH][LT_N];
  __shared__ double2 tw[LT_N];
  __shared__ int bad_s;
  const int s = blockIdx.y;
  const LandTab &L = T.sp[s];
  const ProbDev &Pd = *probp;
  const SpecDev &S = Pd.sp[s];
  if (L.c == nullptr) return;
  // SUB: block LT_SUB^2 i + j is small tile j of the i-th tile cut
  int par = blockIdx.x, tile = blockIdx.x;
  if constexpr (SUB) {
    par = L.cut[blockIdx.x / (LT_SUB * LT_SUB)];
    tile = LT_NX * L.ny + (int)blockIdx.x;
    if (par < 0) return;
  } else {
    if (tile >= LT_NX * L.ny) return;
  }
  const int t = threadIdx.x, smp = t & (LT_N - 1), grp = t / LT_N;
  const int nperp = S.nperp, nr = L.nr, Q = 6 * (nr + 1);
  const double d = S.dppar_abs, dpp = S.dpperp;
  double xc = (par % LT_NX) + 0.5, yc = (par / LT_NX) + 0.5;
  if constexpr (SUB) {
    const int j = blockIdx.x % (LT_SUB * LT_SUB);
    xc = (par % LT_NX) + ((j % LT_SUB) + 0.5) / LT_SUB;
    yc = (par / LT_NX) + ((j / LT_SUB) + 0.5) / LT_SUB;
  }
  const cd z0 = mk(__builtin_fma(xc, L.t, L.x0), -(yc * L.t));
  if (t < LT_N) {
    double sn, cs;
    sincospi(2.0 * t / LT_N, &sn, &cs);
    tw[t] = make_double2(cs, sn);
  }
  double *Nq = reinterpret_cast<double *>(Fq + Q * LT_N), *Wq = Nq + Q * LT_N;
  if (t == 0) bad_s = 0;
  for (int i = t; i < Q * LT_N; i += 256) {
    Fq[i] = make_double2(0.0, 0.0);
    Nq[i] = 0.0;
  }
  __syncthreads();
  const double r = (SUB ? 1.0 / LT_SUB : 1.0) / L.ir;
  const cd p = mk(z0.re + r * tw[smp].x, z0.im + r * tw[smp].y);
  const double qk = S.q / fabs(Pd.kpar);
  const double fA = qk * (Pd.kpar / S.m) / (2.0 * d), fB = qk * (S.q / S.m);
  const double i2p = 1.0 / (2.0 * dpp), i1p = 1.0 / dpp;
  bool bad = false;
  for (int c0 = 0; c0 <= nperp; c0 += LT_CH) {
#pragma unroll 1
    for (int u = grp; u < LT_CH; u += 256 / LT_N) {
      const int ip = min(c0 + u, nperp);  // (rows past the last get no weight)
      const cd a = land_f(S, ip, p, bad);
      const cd b = land_f(S, ip, mk(p.re + d, p.im), bad);
      const cd e = land_f(S, ip, mk(p.re - d, p.im), bad);
      f0[u][smp] = make_double2(a.re, a.im);
      fd[u][smp] = make_double2(b.re - e.re, b.im - e.im);
    }
    // row ip's weight in function q
    for (int i = t; i < Q * LT_CH; i += 256) {
      const int q = i / LT_CH, ip = c0 + i % LT_CH;
      const double *at = S.atab + (size_t)(q / 6) * (nperp + 1) * ATAB_STRIDE + q % 3;
      // h a of row ip for the interior rows of dfperp
      auto ha = [&](int r_) {
        if (r_ < 1 || r_ > nperp - 1) return 0.0;
        return (r_ == nperp - 1 ? 0.5 : 1.0) * at[(size_t)r_ * ATAB_STRIDE];
      };
      double w = 0.0;
      if (ip <= nperp) {
        if ((q % 6) < 3) {
          const double h = (ip == 0 || ip >= nperp - 1) ? 0.5 : 1.0;
          w = (h * at[(size_t)ip * ATAB_STRIDE]) * S.pperp[ip] * fA;
        } else {
          // the coefficient of f(ip, p) in sum h a dfperp: central differences
          // inside, one-sided at the first and last row
          w = (ha(ip - 1) - ha(ip + 1)) * i2p;
          if (ip <= 1) w += (ip == 1 ? 0.5 : -0.5) * at[0] * i1p;
          if (ip >= nperp - 1)
            w += (ip == nperp ? 0.5 : -0.5) * at[(size_t)nperp * ATAB_STRIDE] * i1p;
          w *= fB;
        }
      }
      Wq[i] = w;
    }
    __syncthreads();
    for (int q = grp; q < Q; q += 256 / LT_N) {
      const bool isB = (q % 6) >= 3;
      const double2(*fv)[LT_N] = isB ? f0 : fd;
      const double *w = Wq + q * LT_CH;
      cd acc = mk(0.0, 0.0);  // (chunk sums first: a shorter chain of roundings)
      double sc = 0.0;
#pragma unroll 4
      for (int u = 0; u < LT_CH; ++u) {
        const double2 v = fv[u][smp], z = f0[u][smp];
        acc.re = __builtin_fma(w[u], v.x, acc.re);
        acc.im = __builtin_fma(w[u], v.y, acc.im);
        sc = __builtin_fma(fabs(w[u]), fabs(z.x) + fabs(z.y), sc);
      }
      Fq[q * LT_N + smp].x += acc.re;
      Fq[q * LT_N + smp].y += acc.im;
      Nq[q * LT_N + smp] += isB ? sc : 2.0 * sc;  // (|f(p + d)| + |f(p - d)| for A)
    }
    __syncthreads();
  }
  // the j-th coefficient (times r^j) of function q
  auto coef = [&](int q, int j) {
    cd c = mk(0.0, 0.0);
#pragma unroll 4
    for (int i = 0; i < LT_N; ++i) {
      const double2 v = Fq[q * LT_N + i], w = tw[(i * j) & (LT_N - 1)];
      c.re += v.x * w.x + v.y * w.y;
      c.im += v.y * w.x - v.x * w.y;
    }
    return c * (1.0 / LT_N);
  };
#pragma unroll 1
  for (int q = t; q < Q; q += 256) {
    double sc = 0.0, tail = 0.0;
#pragma unroll 4
    for (int i = 0; i < LT_N; ++i) sc = fmax(sc, Nq[q * LT_N + i]);
#pragma unroll 1
    for (int j = LT_J - 2; j < LT_J + LT_TAIL; ++j) {
      const cd c = coef(q, j);
      tail = fmax(tail, fabs(c.re) + fabs(c.im));
    }
    // (the roundings of the fit's values, which the row sums carry too, are larger)
    if (!(tail <= 0x1p-51 * sc)) bad = true;
  }
  if (bad) bad_s = 1;
  __syncthreads();
  if (t == 0) L.ok[tile] = bad_s ? 0 : 1;
  if (bad_s) return;
  for (int i = t; i < Q * LT_J; i += 256) {
    const int q = i / LT_J, j = i % LT_J;
    const cd c = coef(q, j);
    double *o = L.c + ((((size_t)tile * (nr + 1) + q / 6) * 3 + q % 3) * LT_J + j) * 4 +
                ((q % 6) >= 3 ? 2 : 0);
    o[0] = c.re;
    o[1] = c.im;
  }
}

// the tiles to cut, in order: the unusable ones (ok 0); one workgroup per species
__global__ __launch_bounds__(256) void k_land_cut(LandTabs T) {
  __shared__ int sc[256];
  const LandTab &L = T.sp[blockIdx.x];
  if (L.c == nullptr) return;
  const int t = threadIdx.x, tiles = LT_NX * L.ny, per = (tiles + 255) / 256;
  int cnt = 0;
  for (int i = t * per; i < min((t + 1) * per, tiles); ++i) cnt += L.ok[i] == 0;
  sc[t] = cnt;
  if (t < LT_MAXP) L.cut[t] = -1;
  __syncthreads();
  for (int o = 1; o < 256; o <<= 1) {
    const int v = t >= o ? sc[t - o] : 0;
    __syncthreads();
    sc[t] += v;
    __syncthreads();
  }
  int k = sc[t] - cnt;
  for (int i = t * per; i < min((t + 1) * per, tiles); ++i)
    if (L.ok[i] == 0) {
      if (k < LT_MAXP) {
        L.cut[k] = i;
        L.ok[i] = (unsigned char)(2 + k);
      }
      ++k;
    }
}

}  // namespace

// the tables of every species with T.sp[s].c set, kappa species all (ny: the
// largest of their tile rows, nr: of their harmonics)
hipError_t launch_land_build(hipStream_t st, const ProbDev *prob, int nspec, int ny, int nr,
                             const LandTabs &T) {
  const size_t lds = (size_t)6 * (nr + 1) * (LT_N * sizeof(double2) + (LT_N + LT_CH) * sizeof(double));
  if (nr > LT_NR || ny > LT_NY) return hipErrorInvalidValue;
  const dim3 g0(LT_NX * ny, nspec), g1(LT_MAXP * LT_SUB * LT_SUB, nspec), blk(256);
  hipLaunchKernelGGL(k_land_build<false>, g0, blk, lds, st, prob, T);
  hipLaunchKernelGGL(k_land_cut, dim3(nspec), blk, 0, st, T);
  hipLaunchKernelGGL(k_land_build<true>, g1, blk, lds, st, prob, T);
  return hipGetLastError();
}
