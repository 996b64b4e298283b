// ape.hip -- 3D APE smearing of the gauge field with SU(3) projection, stout
// smearing (3d or 4d), and the plaquette.
//
// One step (lib/src/qcd_smearing.c:205-273), for the spatial directions
// mu = 1, 2, 3 (temporal links are copied unchanged):
//   U'_mu(x) = P_SU3[ U_mu(x) + alpha sum_{nu = 1..3, nu != mu}
//                 ( U_nu(x) U_mu(x+nu) U_nu(x+mu)^+ + U_nu(x-nu)^+ U_mu(x-nu) U_nu(x-nu+mu) ) ]
// P_SU3(M) is the unitary polar factor of M, M (M^+ M)^-1/2, times
// exp(-i arg(det M) / 3) (lib/src/qcd_blas.c:940-1364, which diagonalises
// M^+ M by Cardano's formula).  The polar factor is unique for non-singular
// M; it is computed here by Newton's iteration X <- (g X + X^-+ / g) / 2 with
// Frobenius-norm scaling g, which converges quadratically from X = M.
// One lane per (site, direction); FP64 throughout.  The gauge field is read
// in the device layout (one array per direction of [tile][9][64] links).
#include "blas_common.h"

namespace qcdhip {

using C = Cx<double>;

__device__ __forceinline__ C cm(C a, C b) { return C{fma(a.re, b.re, -(a.im * b.im)), fma(a.re, b.im, a.im * b.re)}; }
__device__ __forceinline__ C cj(C a) { return C{a.re, -a.im}; }

// c (+)= a b (DA: a^+, DB: b^+; ADD: added to c): a chain of fused
// multiply-adds per element, 108 instructions.  An element's product is summed
// from zero and then added: a chain that starts from c rounds each of its terms
// at the size of a whole staple sum.
template <bool DA, bool DB, bool ADD = false>
__device__ __forceinline__ void mm3(C c[9], const C a[9], const C b[9]) {
#pragma unroll
  for (int i = 0; i < 3; i++)
#pragma unroll
    for (int j = 0; j < 3; j++) {
      double re, im;
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const C x = DA ? cj(a[3 * k + i]) : a[3 * i + k];
        const C y = DB ? cj(b[3 * j + k]) : b[3 * k + j];
        re = k == 0 ? x.re * y.re : fma(x.re, y.re, re);
        im = k == 0 ? x.re * y.im : fma(x.re, y.im, im);
        re = fma(-x.im, y.im, re);
        im = fma(x.im, y.re, im);
      }
      c[3 * i + j] = ADD ? C{c[3 * i + j].re + re, c[3 * i + j].im + im} : C{re, im};
    }
}

// 1 / x for normal x > 0: the hardware's approximation and two Newton steps.
// Zero, infinity and NaN give NaN.
__device__ __forceinline__ double recip(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(fma(-x, r, 1.0), r, r);
  return fma(fma(-x, r, 1.0), r, r);
}

// cofactor of element (r, c) of a 3x3 matrix
__device__ __forceinline__ C cof3(const C x[9], int r, int c) {
  const int r1 = (r + 1) % 3, r2 = (r + 2) % 3, c1 = (c + 1) % 3, c2 = (c + 2) % 3;
  const C p = x[3 * r1 + c1], q = x[3 * r2 + c2], u = x[3 * r1 + c2], v = x[3 * r2 + c1];
  return C{fma(p.re, q.re, fma(-p.im, q.im, fma(-u.re, v.re, u.im * v.im))),
           fma(p.re, q.im, fma(p.im, q.re, fma(-u.re, v.im, -(u.im * v.re))))};
}

// SU(3) projection in place: Newton's iteration X <- (g X + X^-+ / g) / 2.
//
// The FP64 arithmetic of this loop and of the staples bounds the smearing
// kernels, so a step spends nothing that the result does not need:
//  * any positive factors in place of g and 1/g leave the polar factor as it
//    is, so the Frobenius scaling (|X^-1| / |X|)^1/2 is a single-precision
//    fourth root with the exponents split off (it cannot over- or underflow),
//    taken while the last change was above 1e-2 per unit;
//  * an unscaled step that changed X by D leaves an error of |D|^2 / 2, so
//    the loop ends at |D|^2 <= 1e-17 without a step that confirms it;
//  * the phase exp(-i arg(det M) / 3) starts from single precision and takes two
//    Newton steps z <- z + z (1 - z^3 det X) / 3 on the determinant of the X
//    reached, not of M: every step's rounding turns X by a common phase too, and
//    leaves a common factor, which z takes out.
// 24^3x48: an APE step 446-468 -> 322 us with these and the fused products.  Error
// of a step on generated fields (eps 0.1, 0.3, 1.0), rms over the links: 4.0, 5.3,
// 10.1e-17; with the phase of det M, the last factor as z (4 - t) / 3 and the
// products added into the staple sum term by term 7.3, 8.7, 15.6e-17; with sin, cos
// and atan2 and a confirming step 5.6, 6.9, 12.3e-17.
__device__ __forceinline__ void project_su3(C m[9]) {
  C x[9];
#pragma unroll
  for (int k = 0; k < 9; k++) x[k] = m[k];
  C w{0.0, 0.0};   // det M, normalised for the range of FP32
  double diff = 1.0;
  for (int it = 0; it < 100; it++) {
    // y = (x^-1)^+ = conj(cofactor(x)) / conj(det x)
    C y[9];
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
      for (int c = 0; c < 3; c++) y[3 * r + c] = cof3(x, r, c);
    C d = cm(x[0], y[0]);
#pragma unroll
    for (int c = 1; c < 3; c++)
      d = C{fma(x[c].re, y[c].re, fma(-x[c].im, y[c].im, d.re)), fma(x[c].re, y[c].im, fma(x[c].im, y[c].re, d.im))};
    const double dd = fma(d.re, d.re, d.im * d.im);
    if (it == 0) {
      const double rd = __builtin_amdgcn_rsq(dd);
      w = C{d.re * rd, d.im * rd};
    }
    const double rdd = recip(dd);
    double g = 0.5, rg = 0.5;
    const bool scale = !(diff <= 1e-4);
    if (scale) {
      double nx = 0.0, ny = 0.0;
#pragma unroll
      for (int k = 0; k < 9; k++) {
        nx = fma(x[k].re, x[k].re, fma(x[k].im, x[k].im, nx));
        ny = fma(y[k].re, y[k].re, fma(y[k].im, y[k].im, ny));
      }
      ny *= rdd;   // |X^-1|^2
      // ny / nx = 2^(4 q) f with f in (1/2, 16): g = 2^q f^1/4
      const int e = __builtin_amdgcn_frexp_exp(ny) - __builtin_amdgcn_frexp_exp(nx), q = e >> 2;
      const float f = ldexpf((float)__builtin_amdgcn_frexp_mant(ny) *
                                 __builtin_amdgcn_rcpf((float)__builtin_amdgcn_frexp_mant(nx)),
                             e - 4 * q);
      const float h = __builtin_amdgcn_sqrtf(__builtin_amdgcn_sqrtf(f));
      g = ldexp((double)h, q - 1);
      rg = ldexp((double)__builtin_amdgcn_rcpf(h), -q - 1);
    }
    // conj(cof / d) rg = conj(cof) d rdd rg
    const C s{d.re * rdd * rg, d.im * rdd * rg};
    diff = 0.0;
#pragma unroll
    for (int k = 0; k < 9; k++) {
      const C q = cm(cj(y[k]), s);
      const C n{fma(g, x[k].re, q.re), fma(g, x[k].im, q.im)};
      const double dr = n.re - x[k].re, di = n.im - x[k].im;
      diff = fma(dr, dr, fma(di, di, diff));
      x[k] = n;
    }
    if (!scale && diff <= 1e-17) break;
  }
  C d{0.0, 0.0};   // det X
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const C y = cof3(x, 0, c);
    d = C{fma(x[c].re, y.re, fma(-x[c].im, y.im, d.re)), fma(x[c].re, y.im, fma(x[c].im, y.re, d.im))};
  }
  const float ph = -atan2f((float)w.im, (float)w.re) / 3.0f;
  C z{(double)__cosf(ph), (double)__sinf(ph)};
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const C t = cm(cm(cm(z, z), z), d);
    const C e{(1.0 - t.re) * (1.0 / 3.0), t.im * (-1.0 / 3.0)};
    z = C{fma(z.re, e.re, fma(-z.im, e.im, z.re)), fma(z.re, e.im, fma(z.im, e.re, z.im))};
  }
#pragma unroll
  for (int k = 0; k < 9; k++) m[k] = cm(x[k], z);
}

// Plaquette sum of one site over the 6 planes mu < nu (qcd_observables.c:15-36):
// Re tr[U_mu(x) U_nu(x+mu) U_mu(x+nu)^+ U_nu(x)^+], one workgroup partial each.
__global__ void __launch_bounds__(kBlock) k_plaquette(DslashArgs a, GaugeIn<QCD_HIP_F64> U, double *partials) {
  const unsigned s = xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  double sum = 0.0;
  if (s < a.V) {
    const Site st = site_coords(s, a);
    unsigned fwd[4];
    fwd[0] = neighbour<0, +1>(st, a);
    fwd[1] = neighbour<1, +1>(st, a);
    fwd[2] = neighbour<2, +1>(st, a);
    fwd[3] = neighbour<3, +1>(st, a);
    for (int mu = 0; mu < 3; mu++)
      for (int nu = mu + 1; nu < 4; nu++) {
        C A[9], B[9], T[9], P[9];
        U.load(mu, s, A);
        U.load(nu, fwd[mu], B);
        mm3<false, false>(T, A, B);
        U.load(mu, fwd[nu], A);
        mm3<false, true>(P, T, A);
        U.load(nu, s, A);
        // Re tr(P A^+) = sum_ij Re(P_ij conj(A_ij))
#pragma unroll
        for (int k = 0; k < 9; k++) sum += P[k].re * A[k].re + P[k].im * A[k].im;
      }
  }
  block_reduce_store(sum, partials, blockIdx.x);
}

// ------------------------------------------------------------ stout
// sin(w)/w, with the reference's series below |w| = 0.05 (qcd_smearing.c:279-290)
__device__ __forceinline__ double stout_xi0(double w) {
  if (fabs(w) < 0.05) {
    const double t = 1.0 - w * w / 42.0;
    const double t1 = 1.0 - w * w / 20.0 * t;
    return 1.0 - w * w / 6.0 * t1;
  }
  return sin(w) / w;
}

// m <- exp(i m) for Hermitian traceless m: f0 + f1 Q + f2 Q^2 with the
// Cayley-Hamilton coefficients of Peardon & Morningstar (hep-lat/0311018
// eqs. 19, 29-34; qcd_smearing.c:293-370).  Where rounding puts the argument
// of acos above 1 (two equal eigenvalues) it is clamped to 1; at Q = 0 the
// reference divides 0 by 0.  It returns NaN in both cases.
//
// For tr Q^2 / 2 <= 3/4 the eigenvalues are at most 1 in size and the
// coefficients come from the exponential series instead: Q^3 = c1 Q + c0 gives
// Q^n = a_n + b_n Q + d_n Q^2 with a' = c0 d, b' = a + c1 d, d' = b (real), and
// 21 orders reach 1/21! = 2e-20.  No trigonometric functions, no division by
// 9 u^2 - w^2 (which is small for nearly equal eigenvalues).  A step of
// rho = 0.1 stays below it on any SU(3) field (|Q| <= 0.6).
__device__ __forceinline__ void stout_exp(C m[9]) {
  // Q^2, Hermitian
  C m2[9];
#pragma unroll
  for (int i = 0; i < 3; i++) {
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < 3; k++) t = fma(m[3 * i + k].re, m[3 * i + k].re, fma(m[3 * i + k].im, m[3 * i + k].im, t));
    m2[4 * i] = C{t, 0.0};
#pragma unroll
    for (int j = i + 1; j < 3; j++) {
      C q = cm(m[3 * i], m[j]);
#pragma unroll
      for (int k = 1; k < 3; k++) {
        const C x = m[3 * i + k], y = m[3 * k + j];
        q = C{fma(x.re, y.re, fma(-x.im, y.im, q.re)), fma(x.re, y.im, fma(x.im, y.re, q.im))};
      }
      m2[3 * i + j] = q;
      m2[3 * j + i] = cj(q);
    }
  }
  // c0 = tr Q^3 / 3, c1 = tr Q^2 / 2
  double c0 = 0.0;
#pragma unroll
  for (int i = 0; i < 3; i++)
#pragma unroll
    for (int j = 0; j < 3; j++)
      c0 = fma(m2[3 * i + j].re, m[3 * j + i].re, fma(-m2[3 * i + j].im, m[3 * j + i].im, c0));
  c0 *= 1.0 / 3.0;
  const double c1 = (m2[0].re + m2[4].re + m2[8].re) / 2.0;
  C f0, f1, f2;
  if (c1 <= 0.75) {
    // scaled by 1/n!: a, b, d hold a_n / n!
    double a = 1.0, b = 0.0, d = 0.0;
    f0 = C{1.0, 0.0};
    f1 = f2 = C{0.0, 0.0};
#pragma unroll
    for (int n = 1; n <= 21; n++) {
      const double r = 1.0 / n, na = c0 * d * r, nb = fma(c1, d, a) * r, nd = b * r;
      a = na;
      b = nb;
      d = nd;
      if (n % 2 == 0) {   // i^n real
        const double sg = n % 4 == 0 ? 1.0 : -1.0;
        f0.re = fma(sg, a, f0.re);
        f1.re = fma(sg, b, f1.re);
        f2.re = fma(sg, d, f2.re);
      } else {
        const double sg = n % 4 == 1 ? 1.0 : -1.0;
        f0.im = fma(sg, a, f0.im);
        f1.im = fma(sg, b, f1.im);
        f2.im = fma(sg, d, f2.im);
      }
    }
  } else {
    const bool neg = c0 < 0.0;
    if (neg) c0 = -c0;
    const double c0max = 2.0 * pow(c1 / 3.0, 1.5);
    const double theta = acos(c0 < c0max ? c0 / c0max : 1.0);   // degenerate spectra: rounding can exceed 1
    const double u = sqrt(c1 / 3.0) * cos(theta / 3.0);
    const double w = sqrt(c1) * sin(theta / 3.0);
    const double xi = stout_xi0(w), cw = cos(w);
    const C e2iu{cos(2 * u), sin(2 * u)}, emiu{cos(u), -sin(u)};
    const C h0 = [&] {
      const C a = cm(C{u * u - w * w, 0.0}, e2iu), b = cm(emiu, C{8 * u * u * cw, 2 * u * (3 * u * u + w * w) * xi});
      return C{a.re + b.re, a.im + b.im};
    }();
    const C h1 = [&] {
      const C a = cm(C{2 * u, 0.0}, e2iu), b = cm(emiu, C{2 * u * cw, -(3 * u * u - w * w) * xi});
      return C{a.re - b.re, a.im - b.im};
    }();
    const C h2 = [&] {
      const C b = cm(emiu, C{cw, 3 * u * xi});
      return C{e2iu.re - b.re, e2iu.im - b.im};
    }();
    const double fac = 9 * u * u - w * w;
    // eq. (34): f_j(-c0) = (-1)^j conj(f_j(c0))
    f0 = neg ? C{h0.re / fac, -h0.im / fac} : C{h0.re / fac, h0.im / fac};
    f1 = neg ? C{-h1.re / fac, h1.im / fac} : C{h1.re / fac, h1.im / fac};
    f2 = neg ? C{h2.re / fac, -h2.im / fac} : C{h2.re / fac, h2.im / fac};
  }
#pragma unroll
  for (int k = 0; k < 9; k++) {
    const C p = m[k], q = m2[k];
    C r = k % 4 == 0 ? f0 : C{0.0, 0.0};
    r = C{fma(f1.re, p.re, fma(-f1.im, p.im, r.re)), fma(f1.re, p.im, fma(f1.im, p.re, r.im))};
    m[k] = C{fma(f2.re, q.re, fma(-f2.im, q.im, r.re)), fma(f2.re, q.im, fma(f2.im, q.re, r.im))};
  }
}

template <int MU>
__device__ __forceinline__ unsigned fwd_of(const Site &st, const DslashArgs &a) {
  return neighbour<MU, +1>(st, a);
}
__device__ __forceinline__ unsigned fwd_dir(unsigned mu, const Site &st, const DslashArgs &a) {
  return mu == 0 ? fwd_of<0>(st, a) : mu == 1 ? fwd_of<1>(st, a) : mu == 2 ? fwd_of<2>(st, a) : fwd_of<3>(st, a);
}
__device__ __forceinline__ unsigned bwd_dir(unsigned mu, const Site &st, const DslashArgs &a) {
  return mu == 0 ? neighbour<0, -1>(st, a) : mu == 1 ? neighbour<1, -1>(st, a)
                                           : mu == 2 ? neighbour<2, -1>(st, a) : neighbour<3, -1>(st, a);
}

// Site order of the smearing kernels.  Lane j of the launch takes the sites of
// one y slab after another, each slab swept along z in (t, x, y) order, and the
// directions of a block of sites are the fastest block index: an XCD then
// holds the planes z - 1, z, z + 1 of its slab and the links that the
// directions share in its L2.  24^3x48, against site order with the directions
// as separate passes and the same arithmetic (us a step): APE 322 -> 286,
// stout 440 -> 415.  What bounds APE now is traffic between L2 and the fabric
// (1.6 GB read for 0.29 GB of spatial links a step, 6.3 TB/s with the writes)
// together with the FP64 pipes, busy 48% of the time; a 4d stout step reads 1.5 GB
// for 0.38 at 4.0 TB/s, pipes 44%, with two wavefronts per SIMD (224 VGPRs).  Tried and slower: rows of the products
// formed one at a time (fewer registers, 3-4 wavefronts per SIMD), separate
// loops over backward and forward stout staples (3 wavefronts).
struct SlabOrder {
  unsigned by;     // y rows per slab
  unsigned full;   // sites of a full slab, T X by Z
};
__device__ __forceinline__ Site slab_site(unsigned j, const SlabOrder &o, const DslashArgs &a) {
  const unsigned P = a.L[0] * a.L[1];
  const unsigned k = j / o.full, y0 = k * o.by, ny = min(o.by, a.L[2] - y0);
  unsigned r = j - k * o.full;
  Site st;
  st.z = r / (P * ny);
  r -= st.z * P * ny;
  const unsigned yy = r / P;
  r -= yy * P;
  st.y = y0 + yy;
  st.x = r / a.L[0];
  st.t = r - st.x * a.L[0];
  st.s = r + P * (st.y + a.L[2] * st.z);
  st.valid = true;
  return st;
}

// One APE step for the spatial directions, one lane per (site, direction)
// with the direction uniform over the workgroup, so the staple loops do not
// diverge.  Each staple's three links are loaded as its
// products need them, which bounds the live matrices to the staple sum and
// two factors.  The temporal links are copied by the caller.
__global__ void __launch_bounds__(kBlock) k_ape3d(DslashArgs a, GaugeIn<QCD_HIP_F64> U, double2 *__restrict__ out,
                                                  size_t stride, double alpha, SlabOrder ord) {
  const unsigned lb = xcd_block(blockIdx.x, gridDim.x);
  const unsigned j = lb / 3 * kBlock + threadIdx.x, mu = 1 + lb % 3;   // mu is uniform over the workgroup
  if (j >= a.V) return;
  const Site st = slab_site(j, ord, a);
  const unsigned s = st.s;
  C S[9];
#pragma unroll
  for (int k = 0; k < 9; k++) S[k] = C{0.0, 0.0};
  // forward staples U_nu(x) U_mu(x+nu) U_nu(x+mu)^+, then backward ones
  // U_nu(x-nu)^+ U_mu(x-nu) U_nu(x-nu+mu) (the reference's order)
  const unsigned sf = fwd_dir(mu, st, a);
#pragma unroll 1
  for (unsigned nu = 1; nu < 4; nu++) {
    if (nu == mu) continue;
    C T[9];
    {
      C A[9], B[9];
      U.load(nu, s, A);
      U.load(mu, fwd_dir(nu, st, a), B);
      mm3<false, false>(T, A, B);
    }
    C W[9];
    U.load(nu, sf, W);
    mm3<false, true, true>(S, T, W);
  }
#pragma unroll 1
  for (unsigned nu = 1; nu < 4; nu++) {
    if (nu == mu) continue;
    const unsigned sn = bwd_dir(nu, st, a);
    C T[9];
    {
      C B[9], W[9];
      U.load(mu, sn, B);
      U.load(nu, fwd_dir(mu, site_coords(sn, a), a), W);
      mm3<false, false>(T, B, W);
    }
    C A[9];
    U.load(nu, sn, A);
    mm3<true, false, true>(S, A, T);
  }
  C m[9];
  U.load(mu, s, m);
#pragma unroll
  for (int k = 0; k < 9; k++) m[k] = C{m[k].re + alpha * S[k].re, m[k].im + alpha * S[k].im};
  project_su3(m);
  double2 *o = out + (size_t)mu * 9 * stride + (size_t)(s / kTile) * 9 * kTile + s % kTile;
#pragma unroll
  for (int k = 0; k < 9; k++) o[(size_t)k * kTile] = make_double2(m[k].re, m[k].im);
}

// One stout step (qcd_smearing.c:374-476), one lane per (site, direction):
// C = sum over nu != mu (nu from START) of the backward staple then the
// forward one, W = C U^+, A = W - W^+ minus tr(A)/3, Q = -i rho/2 A,
// U' = exp(iQ) U.  The direction is uniform over the workgroup; directions below START (the temporal one for 3d stout) are
// copied by the caller.
template <unsigned START>
__global__ void __launch_bounds__(kBlock) k_stout(DslashArgs a, GaugeIn<QCD_HIP_F64> U, double2 *__restrict__ out,
                                                  size_t stride, double rho, SlabOrder ord) {
  const unsigned lb = xcd_block(blockIdx.x, gridDim.x);
  const unsigned j = lb / (4 - START) * kBlock + threadIdx.x;
  const unsigned mu = START + lb % (4 - START);   // uniform over the workgroup
  if (j >= a.V) return;
  const Site st = slab_site(j, ord, a);
  const unsigned s = st.s;
  C S[9];
#pragma unroll
  for (int k = 0; k < 9; k++) S[k] = C{0.0, 0.0};
  const unsigned sf = fwd_dir(mu, st, a);
#pragma unroll 1
  for (unsigned nu = START; nu < 4; nu++) {
    if (nu == mu) continue;
    // backward: U_nu(x-nu)^+ [U_mu(x-nu) U_nu(x-nu+mu)]
    const unsigned sb = bwd_dir(nu, st, a);
    {
      C T[9];
      {
        C B[9], W[9];
        U.load(mu, sb, B);
        U.load(nu, fwd_dir(mu, site_coords(sb, a), a), W);
        mm3<false, false>(T, B, W);
      }
      C A[9];
      U.load(nu, sb, A);
      mm3<true, false, true>(S, A, T);
    }
    // forward: [U_nu(x) U_mu(x+nu)] U_nu(x+mu)^+
    {
      C T[9];
      {
        C A[9], B[9];
        U.load(nu, s, A);
        U.load(mu, fwd_dir(nu, st, a), B);
        mm3<false, false>(T, A, B);
      }
      C W[9];
      U.load(nu, sf, W);
      mm3<false, true, true>(S, T, W);
    }
  }
  C m[9], W[9];
  U.load(mu, s, m);
  mm3<false, true>(W, S, m);   // W = C U^+
  C q[9];
#pragma unroll
  for (int r = 0; r < 3; r++)
#pragma unroll
    for (int c = 0; c < 3; c++) q[3 * r + c] = C{W[3 * r + c].re - W[3 * c + r].re, W[3 * r + c].im + W[3 * c + r].im};
  const C tr{(q[0].re + q[4].re + q[8].re) / 3.0, (q[0].im + q[4].im + q[8].im) / 3.0};
#pragma unroll
  for (int r = 0; r < 3; r++) q[4 * r] = C{q[4 * r].re - tr.re, q[4 * r].im - tr.im};
#pragma unroll
  for (int k = 0; k < 9; k++) q[k] = C{0.5 * rho * q[k].im, -0.5 * rho * q[k].re};   // Q = -i rho/2 A
  stout_exp(q);
  mm3<false, false>(W, q, m);
  double2 *o = out + (size_t)mu * 9 * stride + (size_t)(s / kTile) * 9 * kTile + s % kTile;
#pragma unroll
  for (int k = 0; k < 9; k++) o[(size_t)k * kTile] = make_double2(W[k].re, W[k].im);
}

// One slab per XCD while its plane of links fits L2 (2.4 MB): 24^3x48 takes 3
// rows (APE 10 steps 2.92 ms; 2 rows 3.01, 6 rows 3.08, site order 3.27),
// 32^3x64 2 rows (2 steps 2.34 ms; 4 rows 2.41, site order 2.43), 48^3x96
// single rows.
static SlabOrder slab_order(qcd_hip_lattice lat) {
  const unsigned Y = (unsigned)lat->L[2], row = (unsigned)lat->L[0] * (unsigned)lat->L[1];
  const unsigned fit = std::max(1u, 2400000u / (row * 576u));
  const unsigned by = std::min((Y + kNumXcd - 1) / kNumXcd, fit);
  return SlabOrder{by, row * by * (unsigned)lat->L[3]};
}

// temporal links of in copied to out: direction 0 is the first 9 stride
// links of the layout
static int copy_temporal(qcd_hip_field out, qcd_hip_field in, hipStream_t st) {
  QH_CHECK(hipMemcpyAsync(out->data, in->data, (size_t)9 * in->lat->stride * sizeof(double2),
                          hipMemcpyDeviceToDevice, st));
  return 0;
}

// keep: out holds the temporal links already (the second and later steps
// that write one of the two ping-pong fields)
int stout_step(qcd_hip_field out, qcd_hip_field in, double rho, int ndim, bool keep, hipStream_t st) {
  const DslashArgs a = make_args(in->lat, 0.0, 0.0);
  const int grid = grid_for(in->lat->V);
  if (ndim == 3) {
    if (!keep) QH_TRY(copy_temporal(out, in, st));
    k_stout<1><<<3 * grid, kBlock, 0, st>>>(a, GaugeIn<QCD_HIP_F64>::of(in), (double2 *)out->data,
                                                 (size_t)in->lat->stride, rho, slab_order(in->lat));
  } else {
    k_stout<0><<<4 * grid, kBlock, 0, st>>>(a, GaugeIn<QCD_HIP_F64>::of(in), (double2 *)out->data,
                                                 (size_t)in->lat->stride, rho, slab_order(in->lat));
  }
  QH_CHECK(hipGetLastError());
  return 0;
}

int ape_step(qcd_hip_field out, qcd_hip_field in, double alpha, bool keep, hipStream_t st) {
  const DslashArgs a = make_args(in->lat, 0.0, 0.0);
  if (!keep) QH_TRY(copy_temporal(out, in, st));
  k_ape3d<<<3 * grid_for(in->lat->V), kBlock, 0, st>>>(a, GaugeIn<QCD_HIP_F64>::of(in), (double2 *)out->data,
                                                           (size_t)in->lat->stride, alpha, slab_order(in->lat));
  QH_CHECK(hipGetLastError());
  return 0;
}

// every link (all four directions) projected onto SU(3) in place
// (lib/src/qcd_blas.c:541-939): one lane per (site, direction)
__global__ void __launch_bounds__(kBlock) k_project_links(GaugeIn<QCD_HIP_F64> U, double2 *__restrict__ data,
                                                          unsigned V, size_t stride) {
  const unsigned s = xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  if (s >= V) return;
  const unsigned mu = blockIdx.y;
  C m[9];
  U.load(mu, s, m);
  project_su3(m);
  double2 *o = data + (size_t)mu * 9 * stride + (size_t)(s / kTile) * 9 * kTile + s % kTile;
#pragma unroll
  for (int k = 0; k < 9; k++) o[(size_t)k * kTile] = make_double2(m[k].re, m[k].im);
}
}  // namespace qcdhip

using namespace qcdhip;

extern "C" {

int qcd_hip_project_su3(qcd_hip_field g) {
  QH_TRY(ensure_init());
  if (!g || g->kind != QCD_HIP_GAUGE || g->prec != QCD_HIP_F64) {
    set_error("project_su3: expected an FP64 gauge field");
    return 1;
  }
  std::lock_guard<std::recursive_mutex> lock(state_mutex());
  hipStream_t st = ctx()->stream;
  gauge_written(g);
  k_project_links<<<dim3(grid_for(g->lat->V), 4), kBlock, 0, st>>>(GaugeIn<QCD_HIP_F64>::of(g), (double2 *)g->data,
                                                                   (unsigned)g->lat->V, (size_t)g->lat->stride);
  QH_CHECK(hipGetLastError());
  QH_CHECK(hipStreamSynchronize(st));
  return 0;
}

int qcd_hip_ape_smear(qcd_hip_field out, qcd_hip_field in, double alpha, int nsteps) {
  QH_TRY(ensure_init());
  if (!out || !in || out == in || out->kind != QCD_HIP_GAUGE || in->kind != QCD_HIP_GAUGE ||
      out->prec != QCD_HIP_F64 || in->prec != QCD_HIP_F64 || out->lat->V != in->lat->V || nsteps < 0) {
    set_error("ape_smear: expected two distinct FP64 gauge fields on one lattice and nsteps >= 0");
    return 1;
  }
  for (int d = 0; d < 4; d++)
    if (out->lat->L[d] != in->lat->L[d]) {
      set_error("ape_smear: lattice extents differ");
      return 1;
    }
  std::lock_guard<std::recursive_mutex> lock(state_mutex());
  gauge_written(out);
  hipStream_t st = ctx()->stream;
  if (nsteps == 0) {
    QH_CHECK(hipMemcpyAsync(out->data, in->data, out->bytes, hipMemcpyDeviceToDevice, st));
    QH_CHECK(hipStreamSynchronize(st));
    return 0;
  }
  qcd_hip_field tmp = nullptr;
  if (nsteps > 1) QH_TRY(gauge_create_unfilled(&tmp, in->lat));
  // ping-pong so that the last step writes out
  qcd_hip_field src = in;
  int rc = 0;
  for (int k = 0; k < nsteps && !rc; k++) {
    qcd_hip_field dst = ((nsteps - 1 - k) % 2 == 0) ? out : tmp;
    rc = ape_step(dst, src, alpha, k >= 2, st);
    src = dst;
  }
  if (!rc && hipStreamSynchronize(st) != hipSuccess) {
    set_error("ape_smear: %s", hipGetErrorString(hipGetLastError()));
    rc = 2;
  }
  qcd_hip_field_destroy(tmp);
  return rc;
}

int qcd_hip_stout_smear(qcd_hip_field out, qcd_hip_field in, double rho, int ndim, int nsteps) {
  QH_TRY(ensure_init());
  if (!out || !in || out == in || out->kind != QCD_HIP_GAUGE || in->kind != QCD_HIP_GAUGE ||
      out->prec != QCD_HIP_F64 || in->prec != QCD_HIP_F64 || out->lat->V != in->lat->V || nsteps < 0) {
    set_error("stout_smear: expected two distinct FP64 gauge fields on one lattice and nsteps >= 0");
    return 1;
  }
  if (ndim != 3 && ndim != 4) {
    set_error("stout_smear: ndim should be either 3 or 4");
    return 1;
  }
  for (int d = 0; d < 4; d++)
    if (out->lat->L[d] != in->lat->L[d]) {
      set_error("stout_smear: lattice extents differ");
      return 1;
    }
  std::lock_guard<std::recursive_mutex> lock(state_mutex());
  gauge_written(out);
  hipStream_t st = ctx()->stream;
  if (nsteps == 0) {
    QH_CHECK(hipMemcpyAsync(out->data, in->data, out->bytes, hipMemcpyDeviceToDevice, st));
    QH_CHECK(hipStreamSynchronize(st));
    return 0;
  }
  qcd_hip_field tmp = nullptr;
  if (nsteps > 1) QH_TRY(gauge_create_unfilled(&tmp, in->lat));
  qcd_hip_field src = in;
  int rc = 0;
  for (int k = 0; k < nsteps && !rc; k++) {
    qcd_hip_field dst = ((nsteps - 1 - k) % 2 == 0) ? out : tmp;
    rc = stout_step(dst, src, rho, ndim, k >= 2, st);
    src = dst;
  }
  if (!rc && hipStreamSynchronize(st) != hipSuccess) {
    set_error("stout_smear: %s", hipGetErrorString(hipGetLastError()));
    rc = 2;
  }
  qcd_hip_field_destroy(tmp);
  return rc;
}

int qcd_hip_plaquette(qcd_hip_field gauge, double *plaq) {
  QH_TRY(ensure_init());
  if (!gauge || !plaq || gauge->kind != QCD_HIP_GAUGE || gauge->prec != QCD_HIP_F64) {
    set_error("plaquette: expected an FP64 gauge field");
    return 1;
  }
  std::lock_guard<std::recursive_mutex> lock(state_mutex());
  hipStream_t st = ctx()->stream;
  const DslashArgs a = make_args(gauge->lat, 0.0, 0.0);
  const int grid = grid_for(gauge->lat->V);
  double *part = nullptr;
  QH_TRY(dev_alloc((void **)&part, sizeof(double) * (size_t)grid));
  k_plaquette<<<grid, kBlock, 0, st>>>(a, GaugeIn<QCD_HIP_F64>::of(gauge), part);
  int rc = hipGetLastError() == hipSuccess ? 0 : 2;
  if (!rc) rc = finalize(part, grid, 1, ctx()->scalars, st);
  double sum = 0.0;
  if (!rc) rc = hipMemcpyAsync(&sum, ctx()->scalars, sizeof(double), hipMemcpyDeviceToHost, st) ? 2 : 0;
  if (!rc) rc = hipStreamSynchronize(st) ? 2 : 0;
  dev_free(part, sizeof(double) * (size_t)grid);
  if (rc) {
    set_error("plaquette: kernel failed");
    return rc;
  }
  *plaq = sum / ((double)gauge->lat->V * 3.0 * 6.0);
  return 0;
}

}  // extern "C"
