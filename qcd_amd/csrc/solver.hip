// solver.hip -- the propagator solve of invert.c on the GPU.
//
// Outer loop (invert.c:255-294): true residual r = b - A x in FP64, stop when
// ||r|| / ||b|| <= tol, otherwise solve A e = r with GCR(n) and add e to x.
// Inner GCR(n) (invert.c:20-113, algorithm gcr.m:3-48) in the inner precision
// (FP64 for the plain solver, FP32 or FP16 storage for the mixed one) on the
// operator A = Q = i g5 D (as invert.c) or A = D.  For A = Q the system solved
// is Q x = i g5 b, i.e. D x = b, so the residual is ||b - D x|| either way.
//
// GCR's steps are taken in blocks of S = 8 (FP16: 4; then 4, 2 and 1 for the last
// ones of a cycle), from residual res_k: the operator S times, then
//   k_gcr_dots:    the S new vectors with the earlier w_j, j < k, and with each
//                  other (reads k + S + 1 vectors)
//   k_gcr_scal:    coef and alpha of the S steps
//   k_gcr_update:  w_k .. w_{k+S-1}, orthogonal and unnormalised, and res_{k+S}
//                  (reads k + S + 1 vectors, writes S + 1; not needed in the
//                  last block)
// After n steps k_solution forms x = sum_j beta_j d_j over the directions d_j
// that the operator was applied to, beta from coef and alpha (the reference
// updates x every iteration).
// All coefficients live in device memory: a cycle needs no host round trip.
// Right-hand sides are solved in batches of prm.batch that advance in
// lockstep: every kernel takes a second grid dimension over the batch, and
// right-hand sides that have converged drop out of the launches.
// Orthogonalisation is block-classical Gram-Schmidt in one fused pass (the
// reference's modified Gram-Schmidt, invert.c:68-73, is the same projection in
// exact arithmetic); the outer FP64 residual absorbs the difference.
#include "eo_common.h"

#include <chrono>
#include <cmath>
#include <type_traits>

namespace qcdhip {

// eo.hip
int eo_split(qcd_hip_field full, int f0, qcd_hip_field ev, qcd_hip_field od, const int *ids, int count,
             hipStream_t st);
int eo_accumulate(qcd_hip_field x, int f0, qcd_hip_field ev, qcd_hip_field od, const int *ids, int count,
                  hipStream_t st);
int eo_minv(qcd_hip_lattice full, qcd_hip_field in, qcd_hip_field out, double m, double tm, const int *ids, int count,
            hipStream_t st);
int eo_scale64(qcd_hip_lattice full, qcd_hip_field in, qcd_hip_field out, const double *scale, size_t scale_stride,
               const int *ids, int count, hipStream_t st);
qcd_hip_lattice eo_half_lattice(qcd_hip_lattice full);

constexpr int kN = kMaxKrylov;
constexpr int kSteps = 8;   // most GCR steps of one block

// The coefficients of one right-hand side's GCR cycle: w_k = A d_k + sum_j
// coef[k][j] w_j, and the residual after step k is the one before + alpha[k] w_k.
struct GcrScal {
  double2 coef[kN * kN];   // [k][j], j < k
  double2 alpha[kN];
  double2 beta[kN];        // the cycle's solution is sum_j beta_j d_j
  double w2inv[kN];        // 1 / |w_k|^2 of the stored w_k
  double2 step[kSteps];    // what the stored residual takes of the block's w
  double2 undo, take;      // the part of w_{k-1} that the next / this block takes out of it
  double rmin;             // smallest |res_k|^2 so far
  int stop;                // the rest of the cycle's steps are left out
  double rnorm;
  double rscale;
  int bad;
};

__device__ __forceinline__ double2 cmul2(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// Batched kernels: grid row y works on right-hand-side slot ids[y]; the
// Krylov vector j of slot b is vector b*n + j of the Rs / Ws fields; row y
// writes its partial sums at part + y*rowsz.

// ------------------------------------------------------------ chunks
// A vector is an array of 16-byte chunks: tile after tile, kG groups of 64
// chunks each (SpinorIn::offset), kC complex components of one site per chunk.
// A wavefront takes M consecutive groups, lane by lane, so each of its loads
// is one contiguous 1 KB, and the kernels below see one array whatever the
// layout.  M = kG is one site per lane.
typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
template <int P>
struct Chunk {
  using T = typename Prec<P>::T;
  static constexpr int kG = 12 * (int)sizeof(T) / 16, kC = 16 / (int)sizeof(T);
  static __device__ __forceinline__ u32x4 *at(const SpinorSet<P> &v, int j, unsigned q) {
    return (u32x4 *)(v.base + (size_t)j * v.vstride) + q;
  }
  static __device__ __forceinline__ u32x4 load(const SpinorSet<P> &v, int j, unsigned q) {
    return __builtin_nontemporal_load(at(v, j, q));
  }
  static __device__ __forceinline__ float norm(const SpinorSet<P> &v, int j, unsigned s) {
    if constexpr (P == QCD_HIP_F16) return __builtin_nontemporal_load(&v.norm[(size_t)j * v.nstride + s]);
    else return 1.0f;
  }
  // component i of a chunk as stored (FP16: without the site norm)
  static __device__ __forceinline__ Cx<typename Prec<P>::R> get(u32x4 q, int i) {
    using R = typename Prec<P>::R;
    if constexpr (P == QCD_HIP_F64) {
      const f64x2 d = __builtin_bit_cast(f64x2, q);
      return Cx<R>{d.x, d.y};
    } else if constexpr (P == QCD_HIP_F32) {
      const f32x4 f = __builtin_bit_cast(f32x4, q);
      return Cx<R>{f[2 * i], f[2 * i + 1]};
    } else {
      return to_cx<R>(as_half2(q[i]));
    }
  }
  // sum over the chunk of conj(a) b, of stored values, in FP64 from the product on
  // (FP16 with each pair of products added in FP32: 12 rhs on 24^3x48, 406 against
  // 496 us a launch, 96.1 against 98.5 ms a solve)
  static __device__ __forceinline__ void dot(u32x4 a, u32x4 b, double &re, double &im) {
#pragma unroll
    for (int i = 0; i < kC; i++) {
      const auto x = get(a, i), y = get(b, i);
      re = fma((double)x.re, (double)y.re, fma((double)x.im, (double)y.im, re));
      im = fma((double)x.re, (double)y.im, fma(-(double)x.im, (double)y.re, im));
    }
  }
  // |a|^2 of stored values
  static __device__ __forceinline__ void norm2(u32x4 a, double &re) {
#pragma unroll
    for (int i = 0; i < kC; i++) {
      const auto x = get(a, i);
      re = fma((double)x.re, (double)x.re, fma((double)x.im, (double)x.im, re));
    }
  }
  // acc += c a (FP16: c includes the site norm)
  static __device__ __forceinline__ void axpy(Cx<double> acc[kC], double2 c, u32x4 a) {
#pragma unroll
    for (int i = 0; i < kC; i++) {
      const auto x = get(a, i);
      acc[i].re = fma(c.x, (double)x.re, fma(-c.y, (double)x.im, acc[i].re));
      acc[i].im = fma(c.x, (double)x.im, fma(c.y, (double)x.re, acc[i].im));
    }
  }
};

// first group of this wavefront and its lane's site there
template <int P, int M>
struct ChunkLane {
  unsigned q0, tile, lane;   // chunk of group 0, tile of the wavefront, lane
  bool valid;
  // T lanes per workgroup
  static __device__ __forceinline__ ChunkLane of(unsigned V) {
    constexpr unsigned kG = Chunk<P>::kG;
    static_assert(kG % M == 0, "a wavefront stays in one tile");
    ChunkLane l;
    l.lane = threadIdx.x & 63u;
    const unsigned u = blockIdx.x * (blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    l.tile = u / (kG / M);
    l.q0 = u * (M * 64u) + l.lane;
    l.valid = l.tile * 64u + l.lane < V;
    return l;
  }
  __device__ __forceinline__ unsigned site() const { return tile * 64u + lane; }
};

// x of the lane that DPP control CTRL selects (within rows of 16 lanes)
template <int CTRL>
__device__ __forceinline__ double dpp_move(double x) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const unsigned lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)u, CTRL, 0xf, 0xf, true);
  const unsigned hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(u >> 32), CTRL, 0xf, 0xf, true);
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}
constexpr int kRowMirror = 0x140, kHalfMirror = 0x141, kQuadMirror = 0x1B, kQuadSwap = 0xB1;
// Sums of a over lanes l and l ^ W where bit W of the lane is clear, of b
// where it is set (W = 32 or 16): one swap of register halves (rows) and an
// addition
template <int W>
__device__ __forceinline__ double swap_add(double a, double b) {
  const uint64_t x = __builtin_bit_cast(uint64_t, a), y = __builtin_bit_cast(uint64_t, b);
  auto swap = [](unsigned p, unsigned q) {
    if constexpr (W == 32) return __builtin_amdgcn_permlane32_swap(p, q, false, false);
    else return __builtin_amdgcn_permlane16_swap(p, q, false, false);
  };
  const auto lo = swap((unsigned)x, (unsigned)y), hi = swap((unsigned)(x >> 32), (unsigned)(y >> 32));
  return __builtin_bit_cast(double, (uint64_t)hi[0] << 32 | lo[0]) +
         __builtin_bit_cast(double, (uint64_t)hi[1] << 32 | lo[1]);
}
// the same across the mirrored half rows (W = 8) or quads (W = 4)
template <int W>
__device__ __forceinline__ double mirror_add(double a, double b) {
  const bool up = (threadIdx.x & W) != 0;
  const double keep = up ? b : a, send = up ? a : b;
  return keep + dpp_move<W == 8 ? kRowMirror : kHalfMirror>(send);
}

// Sum NV (2, 4, 8 or 16) values over the wavefront; lane l returns value
// l / (64 / NV).  Every exchange halves the values a lane keeps, by register
// swaps between rows and DPP moves within them: 18 exchanges and additions
// for 8 values, no LDS latency.
template <int NV>
__device__ __forceinline__ double wave_sum_scatter(double (&v)[NV]) {
  constexpr int H = NV / 2;
#pragma unroll
  for (int i = 0; i < H; i++) v[i] = swap_add<32>(v[i], v[i + H]);
  constexpr int Q = H > 1 ? H / 2 : 1;
#pragma unroll
  for (int i = 0; i < Q; i++) v[i] = swap_add<16>(v[i], H > 1 ? v[i + Q] : v[i]);
  if constexpr (NV == 16) v[0] = mirror_add<8>(v[0], v[2]), v[1] = mirror_add<8>(v[1], v[3]);
  else if constexpr (NV == 8) v[0] = mirror_add<8>(v[0], v[1]);
  else v[0] += dpp_move<kRowMirror>(v[0]);
  if constexpr (NV == 16) v[0] = mirror_add<4>(v[0], v[1]);
  else v[0] += dpp_move<kHalfMirror>(v[0]);
  v[0] += dpp_move<kQuadMirror>(v[0]);
  v[0] += dpp_move<kQuadSwap>(v[0]);
  return v[0];
}

// out[i] = x[i] summed over the wavefront, i < min(NX, used), NP at a time
template <int NP_, int NX>
__device__ __forceinline__ void wave_reduce(const double (&x)[NX], double *out, int used) {
  constexpr int NP = NP_ < 16 ? NP_ : 16;
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < NX; i += NP) {
    double y[NP];
#pragma unroll
    for (int q = 0; q < NP; q++) y[q] = i + q < NX ? x[i + q < NX ? i + q : 0] : 0.0;
    const double t = wave_sum_scatter<NP>(y);
    const int q = i + lane / (64 / NP);
    if (lane % (64 / NP) == 0 && q < (NX < used ? NX : used)) out[q] = t;
  }
}

// Sum a [nv][nb] partial array (one wave per value, an order fixed by nb)
// into sums.  Each lane keeps four running sums over partials 256 apart, so
// its loads do not wait on one chain of additions (rows of 20 000 partials
// on 48^3x96).
__device__ void wave_sums(const double *part, int nv, unsigned nb, double *sums) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  for (int v = wid; v < nv; v += nw) {
    const double *p = part + (size_t)v * nb;
    double t0 = 0.0, t1 = 0.0, t2 = 0.0, t3 = 0.0;
    unsigned i = lane;
    for (; i + 192 < nb; i += 256) {
      t0 += p[i];
      t1 += p[i + 64];
      t2 += p[i + 128];
      t3 += p[i + 192];
    }
    for (; i < nb; i += 64) t0 += p[i];
    double t = (t0 + t1) + (t2 + t3);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) t += __shfl_xor(t, off, 64);
    if (lane == 0) sums[v] = t;
  }
}

// sums[q] = sum over p < np of part[p nv + q], q < nv, in an order fixed by np,
// nv and BLK: BLK / nv lanes per value, each over every (BLK / nv)th p, then a
// tree over LDS.  The whole workgroup calls it; sums holds BLK values, nv <= BLK.
template <int BLK>
__device__ __forceinline__ void sum_parts(const double *part, unsigned np, unsigned nv, double *sums) {
  constexpr unsigned NL = 8;
  unsigned g = BLK / nv;
  const unsigned t = threadIdx.x, p0 = t / nv, q = t - p0 * nv;
  double x = 0.0;
  if (p0 < g) {
    const double *a = part + q;
    for (unsigned p = p0; p < np; p += NL * g) {   // NL loads in flight, the last ones too (16: no faster)
      double y[NL];
#pragma unroll
      for (unsigned i = 0; i < NL; i++) y[i] = a[(size_t)min(p + i * g, np - 1) * nv];
#pragma unroll
      for (unsigned i = 0; i < NL; i++) y[i] = p + i * g < np ? y[i] : 0.0;
#pragma unroll
      for (unsigned h = NL / 2; h > 0; h /= 2)
#pragma unroll
        for (unsigned i = 0; i < h; i++) y[i] += y[i + h];
      x += y[0];
    }
  }
  sums[t] = x;
  __syncthreads();
  while (g > 1) {
    const unsigned h = (g + 1) / 2;
    if (p0 + h < g) sums[t] += sums[t + h * nv];
    g = h;
    __syncthreads();
  }
}

// ------------------------------------------------------- blocks of GCR steps
// Directions of a block of S steps at k: d_0 = res_k, d_{a+1} = (A - theta) d_a,
// so v_a = A d_a = d_{a+1} + theta d_a.  w_k .. w_{k+S-1} span what S single steps
// would add, so the residual and the solution after the block are those of
// GCR(n).  The S vectors are projected against the w_j, j < k, in one pass over
// them and formed in a second one, where single steps take 2 S passes, and these
// passes are what a cycle spends its time on (bound by the rate of the fabric, 6.0-6.7 TB/s).  Solves with blocks of 1, 2, 4
// and 8, ms: one FP64 rhs, Q, GCR(32) on 16^3x32 204, 126, 87, 69; one FP32 rhs
// 4: 20.8, 8: 17.3; 12 FP16 rhs, GCR(12), 1, 2, 4 steps: on 24^3x48 136, 111, 98, on
// 16^3x32 21.8, 17.5, 15.4.  FP16 stays at 4: its dots are bound by arithmetic, which
// blocks do not save (8 steps, with cheaper dots, 97 against 96 and 16.0 against
// 15.0), and eight steps carry up to twice the rounding of single ones into long
// cycles.
//
// theta is the local term m + 4 of D and of the Schur complement (0 for Q): the
// d_a are then, but for factors, the residuals of Richardson's iteration, about
// as independent of each other as the residuals of single steps, and a long FP16
// cycle reaches the same residual: GCR(32) on 8^3x16, kappa 0.125, 4.0e-4 of the
// one before, single steps 4.9e-4 (d_1 without theta 8.1e-4).  A cycle reaches
// the least residual of its Krylov space to 2% and the rounding of the stored w_j,
// but for Q beyond 27 steps in FP16 and 40 in FP32, where they lose orthogonality.
// Outer steps against the earlier single steps, which took them from the stored
// w_k: 672 solves each, GCR(8) to GCR(64), kappa 0.1 to 0.139, mu 0 to 0.2, D, Q and
// the Schur complement, random and point sources: FP64 the same or fewer; FP32 one
// more in 3, fewer in 57; FP16 more in 33, all Q, fewer in 278.  Most of the 33 are
// restarted cycles at kappa 0.139 that came out shorter with the rounding of those
// single steps (8^3x16, GCR(24): 97; in blocks of 1, 2 and 4 141, as in FP64).
// Heavy quarks on Q leave directions of a block out: FP64, kappa 0.005, GCR(16)
// takes 2 cycles of blocks for one of single steps.

// Smallest |w_{k+a}|^2 / |v_a|^2 that is told from rounding of the stored vectors:
// a v_a with less to itself is left out of the cycle
template <int P>
constexpr double gcr_floor() { return P == QCD_HIP_F64 ? 1e-13 : P == QCD_HIP_F32 ? 1e-12 : 1e-6; }

// sums of a block of S steps at k: <w_j, d_{a+1}>, a < S, at 2 S j + 2 a (re,
// im) for j < k; then at 2 S k: <d_b, d_a> for b < a <= S at a a + 2 b (re,
// im), |d_a|^2 at a a + 2 a; then |w_{k-1-i}|^2, i < kSteps
template <int S>
constexpr unsigned gcr_own = (S + 1) * (S + 1);
template <int S>
__host__ __device__ constexpr unsigned gcr_values(int k) {
  return 2 * S * (unsigned)k + gcr_own<S> + kSteps;
}

__device__ __forceinline__ double2 cadd2(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 conj2(double2 a) { return make_double2(a.x, -a.y); }
__device__ __forceinline__ double2 scale2(double f, double2 a) { return make_double2(f * a.x, f * a.y); }
__device__ __forceinline__ double norm2(double2 a) { return a.x * a.x + a.y * a.y; }

// Coefficients of a block of S steps from its sums (one wavefront, lane j takes
// w_j).  The w_j are orthogonal to each other and to res_k, so with
//   <w_{k+b}, v_a>, |w_{k+a}|^2, <w_{k+a}, res_k>
// from the Gram matrix of the v_a less its part along the w_j (an L D L^H
// factorisation) every step length is known before the w_{k+a} are formed, and
// w_k .. w_{k+S-1} and res_{k+S} come out of one pass.  The solution is formed
// from the same coef and alpha, so it matches the residual whatever alpha is;
// rounding in alpha only makes a step a little shorter or longer than the best
// one.  A v_a in the span of the others (gcr_floor: exhausted spaces) gets alpha =
// 0 and w2inv = 0, so nothing refers to it.  In reduced precision the w_j of a
// long cycle lose their orthogonality and a step can come out far too long
// (FP16, 64 steps on 270 sites): |res_k|^2 above four times the smallest before
// it leaves the last block and the rest of the cycle out (alpha = 0).  That is
// seen one block late, and never for a cycle's last one.  But the steps of a
// block cannot take more off |res_k|^2 than there is (Bessel): sums that claim so
// by more than kExcess of it come from vectors that are not orthogonal, and leave
// their own block and the rest out.  (FP16, Q, mu = 0.04, point source, 8x6x4x6,
// one cycle of 40 steps: 0.36 of the residual without this, 0.016 with it.)  What
// neither sees is a last block that is too long without claiming too much.  A
// residual of exactly 0 (heavy quarks: FP16 vectors of a few steps) ends the
// cycle as well.  prev: steps of the block before.
//
// The next block starts from res_{k+S}, which has to hold something of
// w_{k+S-1} for its vectors to be new.  Q is indefinite and leaves every other
// step nearly empty (point sources: empty): then the stored residual takes
// kKeep |res_{k+S}| of w_{k+S-1} in place of the step alpha, the solution alpha
// itself, and the next block takes the difference (undo) out again.
constexpr double kKeep = 0.5;
constexpr double kExcess = 0.01;   // above the rounding of the sums, of single and half precision vectors too
template <int P, int S>
__device__ __forceinline__ void gcr_coefficients(GcrScal *sc, const double *sums, int k, int prev, double theta,
                                                 double *tot) {
  const int l = threadIdx.x;
  const double *own = sums + 2 * S * k, *wn = own + gcr_own<S>;
  const double2 undo = k > 0 ? sc->undo : make_double2(0.0, 0.0);
  const double r2 = own[0] - (k > 0 ? norm2(undo) * wn[0] : 0.0);
  const bool stop = k > 0 && (sc->stop || r2 > 4.0 * sc->rmin);
  const bool done = r2 <= 0.0;   // (also where an even-odd source has nothing on the odd sites)
  // <w_j, v_a>
  auto wv = [&](int j, int a) {
    const double *x = sums + 2 * (S * j + a);
    double2 d = make_double2(x[0], x[1]);
    if (a > 0) d = cadd2(d, make_double2(theta * x[-2], theta * x[-1]));
    else if (j == k - 1) d = cadd2(d, scale2(-theta * wn[0], undo));   // <w_j, res_k> = 0
    return d;
  };
  // what the w_j take of the v_a's Gram matrix: tot, indexed as the sums are
  {
    double w = 0.0;
    double2 d[S] = {};
    if (l < k) {
      w = sc->w2inv[l];
      if (l >= k - prev && w > 0.0) {   // as stored
        const double x = wn[k - 1 - l];
        w = x > 0.0 ? 1.0 / x : 0.0;
        sc->w2inv[l] = w;
      }
#pragma unroll
      for (int a = 0; a < S; a++) {
        d[a] = wv(l, a);
        sc->coef[(k + a) * kN + l] = scale2(-w, d[a]);
      }
    }
#pragma unroll
    for (int a = 0; a < S; a++) {
      double e[2 * S] = {};
#pragma unroll
      for (int c = 0; c < a; c++) {
        const double2 x = cmul2(conj2(d[c]), d[a]);
        e[2 * c] = w * x.x;
        e[2 * c + 1] = w * x.y;
      }
      e[2 * a] = w * norm2(d[a]);
      wave_reduce<2 * S>(e, tot + a * a, 2 * a + 1);
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  // <x_b, x_a> from a table of the lower triangle
  auto entry = [](const double *x, int b, int a) {
    if (a == b) return make_double2(x[a * a + 2 * a], 0.0);
    return b < a ? make_double2(x[a * a + 2 * b], x[a * a + 2 * b + 1])
                 : make_double2(x[b * b + 2 * a], -x[b * b + 2 * a + 1]);
  };
  // lane l < S S holds G = <v_i, v_j>, and R = <v_j, res_k>
  const int i = l / S % S, j = l % S;
  const double2 full = cadd2(cadd2(entry(own, i + 1, j + 1),
                                   scale2(theta, cadd2(entry(own, i + 1, j), entry(own, i, j + 1)))),
                             scale2(theta * theta, entry(own, i, j)));
  const double2 x = entry(tot, i, j);
  double2 G = make_double2(full.x - x.x, full.y - x.y);
  double2 R = cadd2(entry(own, j + 1, 0), scale2(theta, entry(own, j, 0)));
  if (k > 0) R = cadd2(R, cmul2(undo, conj2(wv(k - 1, j))));   // res_k = d_0 + undo w_{k-1}
  double rest = r2, w = 0.0;
  double2 al = make_double2(0.0, 0.0);
  bool bad = false, cut = false;
#pragma unroll
  for (int a = 0; a < S; a++) {
    const int o = a * S;   // lanes of row a: <w_{k+a}, v_j>
    const double N = __shfl(G.x, o + a, 64), n = __shfl(full.x, o + a, 64);
    const double2 Gj = make_double2(__shfl(G.x, o + j, 64), __shfl(G.y, o + j, 64));
    const double2 Gi = make_double2(__shfl(G.x, o + i, 64), __shfl(G.y, o + i, 64));
    const double2 Ra = make_double2(__shfl(R.x, a, 64), __shfl(R.y, a, 64));
    w = N > gcr_floor<P>() * n ? 1.0 / N : 0.0;
    bad = bad || !(N == N) || isinf(N) || (a == 0 && !(n > 0.0));
    rest -= w * norm2(Ra);
    cut = cut || rest < -kExcess * r2;
    al = scale2(-w, Ra);
    if (l == 0) {
      sc->w2inv[k + a] = w;
      sc->alpha[k + a] = sc->step[a] = stop || done ? make_double2(0.0, 0.0) : al;
    }
    if (j > a) {
      if (l < S) sc->coef[(k + j) * kN + k + a] = scale2(-w, Gj);
      R = cadd2(R, scale2(-w, cmul2(conj2(Gj), Ra)));
      if (i > a) G = cadd2(G, scale2(-w, cmul2(conj2(Gi), Gj)));
    }
  }
  if (l == 0) {
    if (!stop && !done && bad) sc->bad = 1;   // Krylov space is sick (invert.c:75-79)
    if (stop)
      for (int q = 1; q <= prev; q++) sc->alpha[k - q] = make_double2(0.0, 0.0);
    if (cut)
      for (int a = 0; a < S; a++) sc->alpha[k + a] = sc->step[a] = make_double2(0.0, 0.0);
    sc->rmin = k > 0 ? fmin(sc->rmin, r2) : r2;
    sc->stop = stop || cut || done;
    sc->take = undo;
    const double least = kKeep * kKeep * fmax(rest, 0.0) * w, len = norm2(al);
    double2 un = make_double2(0.0, 0.0);
    if (!sc->stop && len < least) {   // (w = 0: never)
      const double f = sqrt(least);
      const double2 y = len > 0.0 ? scale2(f / sqrt(len), al) : make_double2(f, 0.0);
      sc->step[S - 1] = y;
      un = make_double2(al.x - y.x, al.y - y.y);
    }
    sc->undo = un;
  }
}

// vector d_a of a block of S steps at k: the last one where the last w goes,
// the others among the search directions
template <int P, int S>
struct GcrD {
  const SpinorSet<P> &set;
  int slot;
  __device__ __forceinline__ GcrD(const SpinorSet<P> &W, const SpinorSet<P> &Rs, int k, int a)
      : set(a == S ? W : Rs), slot(k + (a == S ? S - 1 : a)) {}
};

// The sums (gcr_values) of a block of S steps at k, one partial per value and
// workgroup, a workgroup's side by side.
//
// Streams k + S + 1 vectors, J of the w_j in flight at a time (the last group
// reads its last vector again where k is no multiple of J); PRE: the next
// group is loaded before the present one is reduced, for launches with few
// wavefronts per SIMD.  A wavefront adds its sums in its LDS row; the workgroup
// adds the rows once.
template <int P, int S, int M, int J, int BLK, bool PRE>
__global__ void __launch_bounds__(BLK) k_gcr_dots(SpinorSet<P> W, SpinorSet<P> Rs, int n, int k, int prev,
                                                  const int *ids, unsigned V, double *part, size_t rowsz) {
  using CH = Chunk<P>;
  constexpr int NW = BLK / 64, D = S + 1, NV = 2 * S * J, NP = NV <= 4 ? 4 : NV <= 8 ? 8 : 16;
  __shared__ double sums[NW][gcr_values<S>(kN - S)];
  const int b = ids[blockIdx.y];
  const ChunkLane<P, M> l = ChunkLane<P, M>::of(V);
  const unsigned wid = threadIdx.x >> 6;
  const int k0 = b * n;
  struct Group {
    u32x4 a[J][M];
    float nj[J];
  };
  auto load = [&](Group &g, int j0) {
    if (!l.valid) return;
#pragma unroll
    for (int i = 0; i < J; i++) {
      const int j = k0 + min(j0 + i, k - 1);
      g.nj[i] = CH::norm(W, j, l.site());
#pragma unroll
      for (int m = 0; m < M; m++) g.a[i][m] = CH::load(W, j, l.q0 + 64 * m);
    }
  };
  u32x4 d[D][M];
  float nd[D] = {};
  Group next;
  double *own = sums[wid] + 2 * S * k;
  if (l.lane < kSteps) own[gcr_own<S> + l.lane] = 0.0;
  {
    if (l.valid)
#pragma unroll
      for (int a = 0; a < D; a++) {
        const GcrD<P, S> v(W, Rs, k0 + k, a);
        nd[a] = CH::norm(v.set, v.slot, l.site());
#pragma unroll
        for (int m = 0; m < M; m++) d[a][m] = CH::load(v.set, v.slot, l.q0 + 64 * m);
      }
    if constexpr (PRE)
      if (k > 0) load(next, 0);
    // the Gram matrix, kRows rows at a time (nine vectors have 81 sums)
    constexpr int kRows = D > 5 ? 1 : D;
#pragma unroll
    for (int a0 = 0; a0 < D; a0 += kRows) {
      constexpr int NX = D > 5 ? 2 * D - 1 : gcr_own<S>;
      double x[NX] = {};
      if (l.valid)
#pragma unroll
        for (int a = a0; a < a0 + kRows; a++) {
          double *y = x + a * a - a0 * a0;
#pragma unroll
          for (int m = 0; m < M; m++) {
#pragma unroll
            for (int c = 0; c < a; c++) CH::dot(d[c][m], d[a][m], y[2 * c], y[2 * c + 1]);
            CH::norm2(d[a][m], y[2 * a]);
          }
          if constexpr (P == QCD_HIP_F16) {
#pragma unroll
            for (int c = 0; c <= 2 * a; c++) y[c] *= (double)nd[a] * (double)nd[c / 2];
          }
        }
      wave_reduce<NP>(x, own + a0 * a0, D > 5 ? 2 * a0 + 1 : NX);
    }
  }
  for (int j0 = 0; j0 < k; j0 += J) {
    Group g;
    if constexpr (PRE) {
      g = next;
      if (j0 + J < k) load(next, j0 + J);
    } else {
      load(g, j0);
    }
    double x[NV] = {};
    if (l.valid)
#pragma unroll
      for (int i = 0; i < J; i++)
#pragma unroll
        for (int a = 0; a < S; a++) {
          double *y = x + 2 * (S * i + a);
#pragma unroll
          for (int m = 0; m < M; m++) CH::dot(g.a[i][m], d[a + 1][m], y[0], y[1]);
          if constexpr (P == QCD_HIP_F16) {
            const double f = (double)g.nj[i] * (double)nd[a + 1];
            y[0] *= f;
            y[1] *= f;
          }
        }
    wave_reduce<NP>(x, sums[wid] + 2 * S * j0, 2 * S * (k - j0));
    if (j0 + J > k - prev)   // the block before: |w_j|^2 as stored
#pragma unroll
      for (int i = 0; i < J; i++)
        if (j0 + i >= k - prev && j0 + i < k) {
          double y[2] = {0.0, 0.0};
          if (l.valid) {
#pragma unroll
            for (int m = 0; m < M; m++) CH::norm2(g.a[i][m], y[0]);
            if constexpr (P == QCD_HIP_F16) y[0] *= (double)g.nj[i] * (double)g.nj[i];
          }
          const double t = wave_sum_scatter<2>(y);
          if (l.lane == 0) own[gcr_own<S> + (k - 1 - (j0 + i))] = t;
        }
  }
  __syncthreads();
  const unsigned nv = gcr_values<S>(k);
  double *pr = part + blockIdx.y * rowsz + (size_t)blockIdx.x * nv;
  for (unsigned q = threadIdx.x; q < nv; q += BLK) {
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < NW; w++) t += sums[w][q];
    pr[q] = t;
  }
}

// The coefficients of a block from the sums of k_gcr_dots (np workgroups), one
// workgroup per rhs
template <int P, int S>
__global__ void __launch_bounds__(1024) k_gcr_scal(GcrScal *scs, const double *part, size_t rowsz, unsigned np, int k,
                                                   int prev, double theta, const int *ids) {
  __shared__ double sums[1024], tot[S * S];
  static_assert(gcr_values<S>(kN - S) <= 1024, "one value per lane");
  sum_parts<1024>(part + blockIdx.x * rowsz, np, gcr_values<S>(k), sums);
  if (threadIdx.x < 64) gcr_coefficients<P, S>(scs + ids[blockIdx.x], sums, k, prev, theta, tot);
}

// The sums of c workgroups of k_gcr_dots each, added up behind the partial sums
// of all np: the one workgroup of k_gcr_scal reads 0.1 TB/s.  Solves of one rhs
// on 16^3x32, Q, GCR(32), without and with it, ms: FP64 (512 workgroups, up to
// 253 values) 90.2, 89.1; FP32 (1024) 22.3, 20.8 (in blocks of 4).
__global__ void __launch_bounds__(256) k_gcr_sum(double *part, size_t rowsz, unsigned np, unsigned nv, unsigned c) {
  double *row = part + blockIdx.y * rowsz;
  const unsigned p0 = blockIdx.x * c, p1 = min(p0 + c, np);
  for (unsigned q = threadIdx.x; q < nv; q += 256) {
    double t = 0.0;
#pragma unroll 8
    for (unsigned p = p0; p < p1; p++) t += row[(size_t)p * nv + q];
    row[(size_t)(np + blockIdx.x) * nv + q] = t;
  }
}

// Store M chunks of a vector of precision P given in FP64 and leave in q and
// nrm what was stored.  FP16 takes the largest component of the site, which
// lies in kG / M wavefronts of the workgroup (all of a site's wavefronts are in
// one workgroup): mx holds one value per lane of the workgroup.
template <int P, int M>
__device__ __forceinline__ void chunk_store(const SpinorSet<P> &v, int j, const ChunkLane<P, M> &l,
                                            const Cx<double> (&acc)[M][Chunk<P>::kC], u32x4 (&q)[M], float &nrm,
                                            float *mx) {
  using CH = Chunk<P>;
  nrm = 1.0f;
  if constexpr (P == QCD_HIP_F64) {
#pragma unroll
    for (int m = 0; m < M; m++) q[m] = __builtin_bit_cast(u32x4, f64x2{acc[m][0].re, acc[m][0].im});
  } else if constexpr (P == QCD_HIP_F32) {
#pragma unroll
    for (int m = 0; m < M; m++)
      q[m] = __builtin_bit_cast(u32x4, f32x4{(float)acc[m][0].re, (float)acc[m][0].im, (float)acc[m][1].re,
                                             (float)acc[m][1].im});
  } else {
    float x = 0.f;
#pragma unroll
    for (int m = 0; m < M; m++)
#pragma unroll
      for (int i = 0; i < CH::kC; i++) x = fmaxf(x, fmaxf(fabsf((float)acc[m][i].re), fabsf((float)acc[m][i].im)));
    if constexpr (M != CH::kG) {
      constexpr unsigned W = CH::kG / M;   // wavefronts per tile
      const unsigned w0 = (threadIdx.x >> 6) / W * W;
      __syncthreads();   // mx may still be read for the previous vector
      mx[threadIdx.x] = x;
      __syncthreads();
#pragma unroll
      for (unsigned i = 0; i < W; i++) x = fmaxf(x, mx[(w0 + i) * 64u + l.lane]);
    }
    // a site whose largest entry is below the smallest normal float is
    // stored as zero: 1/x would overflow and 0 * inf give NaN
    if (!(x >= FLT_MIN)) x = 0.f;
    const float inv = x > 0.f ? 1.0f / x : 0.f;
    nrm = x;
#pragma unroll
    for (int m = 0; m < M; m++)
#pragma unroll
      for (int i = 0; i < CH::kC; i++)
        q[m][i] = as_u32(__floats2half2_rn((float)acc[m][i].re * inv, (float)acc[m][i].im * inv));
    const unsigned g0 = (l.q0 / 64u) % CH::kG;
    if (l.valid && g0 == 0) __builtin_nontemporal_store(nrm, &v.norm[(size_t)j * v.nstride + l.site()]);
  }
  if (l.valid)
#pragma unroll
    for (int m = 0; m < M; m++) __builtin_nontemporal_store(q[m], CH::at(v, j, l.q0 + 64 * m));
}

// acc[a] += sum of f[a kN + j] times vector j0 + j, j < cnt, J of them in flight
// (and the next J on their way where a lane holds one chunk)
template <int P, int S, int M, int J, bool PRE>
__device__ __forceinline__ void chunk_combine(Cx<double> (&acc)[S][M][Chunk<P>::kC], const SpinorSet<P> &v, int j0,
                                              int cnt, const double2 *f, const ChunkLane<P, M> &l) {
  using CH = Chunk<P>;
  if (!l.valid) return;
  struct Group {
    u32x4 a[J][M];
    float nj[J];
  };
  auto load = [&](Group &g, int i0) {
#pragma unroll
    for (int i = 0; i < J; i++) {
      const int j = j0 + min(i0 + i, cnt - 1);
      g.nj[i] = CH::norm(v, j, l.site());
#pragma unroll
      for (int m = 0; m < M; m++) g.a[i][m] = CH::load(v, j, l.q0 + 64 * m);
    }
  };
  Group next;
  if constexpr (PRE) load(next, 0);
  for (int i0 = 0; i0 < cnt; i0 += J) {
    Group g;
    if constexpr (PRE) {
      g = next;
      if (i0 + J < cnt) load(next, i0 + J);
    } else {
      load(g, i0);
    }
#pragma unroll
    for (int i = 0; i < J; i++)
#pragma unroll
      for (int a = 0; a < S; a++) {
        double2 c = f[a * kN + min(i0 + i, cnt - 1)];
        if (i0 + i >= cnt) c = make_double2(0.0, 0.0);
        if constexpr (P == QCD_HIP_F16) c = make_double2(c.x * (double)g.nj[i], c.y * (double)g.nj[i]);
#pragma unroll
        for (int m = 0; m < M; m++) CH::axpy(acc[a][m], c, g.a[i][m]);
      }
  }
}

// w_{k+a} = v_a + sum_j coef_aj w_j, j < k + a, then res_{k+S} = res_k + sum_a
// step_a w_{k+a} with the stored (rounded) w: one pass over k + S + 1 vectors
// read and S + 1 written.
template <int P, int S, int M, int J, int BLK, bool PRE>
__global__ void __launch_bounds__(BLK) k_gcr_update(SpinorSet<P> W, SpinorSet<P> Rs, int n, int k, double theta,
                                                    const GcrScal *scs, const int *ids, unsigned V) {
  using CH = Chunk<P>;
  __shared__ double2 cf[S * kN], st[S + 1];
  __shared__ float mx[P == QCD_HIP_F16 && M != CH::kG ? BLK : 1];
  const int b = ids[blockIdx.y], k0 = b * n;
  const GcrScal *sc = scs + b;
  for (int i = threadIdx.x; i < S * kN; i += BLK) cf[i] = sc->coef[k * kN + i];
  if (threadIdx.x <= S) st[threadIdx.x] = threadIdx.x < S ? sc->step[threadIdx.x] : sc->take;
  __syncthreads();
  const ChunkLane<P, M> l = ChunkLane<P, M>::of(V);
  auto coef = [](double2 f, float nrm) {
    return P == QCD_HIP_F16 ? scale2((double)nrm, f) : f;
  };
  auto load = [&](u32x4 (&c)[M], float &nrm, const SpinorSet<P> &v, int slot) {
    nrm = l.valid ? CH::norm(v, slot, l.site()) : 0.f;
#pragma unroll
    for (int m = 0; m < M; m++) c[m] = l.valid ? CH::load(v, slot, l.q0 + 64 * m) : u32x4{0, 0, 0, 0};
  };
  auto set = [&](Cx<double> (&x)[M][CH::kC], const u32x4 (&c)[M], float nrm) {
#pragma unroll
    for (int m = 0; m < M; m++)
#pragma unroll
      for (int i = 0; i < CH::kC; i++) {
        const auto y = CH::get(c[m], i);
        x[m][i] = Cx<double>{(double)y.re, (double)y.im};
        if constexpr (P == QCD_HIP_F16) {
          x[m][i].re *= (double)nrm;
          x[m][i].im *= (double)nrm;
        }
      }
  };
  Cx<double> acc[S][M][CH::kC];
  u32x4 r[M], q[S][M];
  float nr, nq[S];
  load(r, nr, Rs, k0 + k);
  {
    u32x4 c[S][M];
    float nc[S];
#pragma unroll
    for (int a = 0; a < S; a++) {
      const GcrD<P, S> v(W, Rs, k0 + k, a + 1);
      load(c[a], nc[a], v.set, v.slot);
    }
#pragma unroll
    for (int a = 0; a < S; a++) {
      set(acc[a], c[a], nc[a]);
#pragma unroll
      for (int m = 0; m < M; m++)
        if (a > 0) CH::axpy(acc[a][m], coef(make_double2(theta, 0.0), nc[a - 1]), c[a - 1][m]);
    }
  }
  if (k > 0) chunk_combine<P, S, M, J, PRE>(acc, W, k0, k, cf, l);
  Cx<double> res[M][CH::kC];
  set(res, r, nr);
#pragma unroll
  for (int m = 0; m < M; m++) CH::axpy(acc[0][m], coef(make_double2(theta, 0.0), nr), r[m]);
  if (st[S].x != 0.0 || st[S].y != 0.0) {
    load(r, nr, W, k0 + k - 1);
#pragma unroll
    for (int m = 0; m < M; m++) CH::axpy(res[m], coef(st[S], nr), r[m]);
  }
#pragma unroll
  for (int a = 0; a < S; a++) {
#pragma unroll
    for (int c = 0; c < a; c++) {
      const double2 f = coef(cf[a * kN + k + c], nq[c]);
#pragma unroll
      for (int m = 0; m < M; m++) CH::axpy(acc[a][m], f, q[c][m]);
    }
    chunk_store<P, M>(W, k0 + k + a, l, acc[a], q[a], nq[a], mx);
    const double2 f = coef(st[a], nq[a]);
#pragma unroll
    for (int m = 0; m < M; m++) CH::axpy(res[m], f, q[a][m]);
  }
  chunk_store<P, M>(Rs, k0 + k + S, l, res, r, nr, mx);
}

// e_b = sum_j beta_j d_j, times |r_b| (the norm the inner source was
// divided by) when scaled
template <int P, int M, int J, int BLK, bool PRE>
__global__ void __launch_bounds__(BLK) k_solution(SpinorSet<P> Rs, int n, const GcrScal *sc, SpinorSet<P> E,
                                                  const int *ids, unsigned V, int scaled) {
  using CH = Chunk<P>;
  __shared__ double2 bt[kN];
  __shared__ float mx[P == QCD_HIP_F16 && M != CH::kG ? BLK : 1];
  const int b = ids[blockIdx.y];
  const double f = scaled ? sc[b].rnorm : 1.0;
  for (int j = threadIdx.x; j < n; j += BLK) bt[j] = make_double2(sc[b].beta[j].x * f, sc[b].beta[j].y * f);
  __syncthreads();
  const ChunkLane<P, M> l = ChunkLane<P, M>::of(V);
  Cx<double> acc[1][M][CH::kC];
#pragma unroll
  for (int m = 0; m < M; m++)
#pragma unroll
    for (int i = 0; i < CH::kC; i++) acc[0][m][i] = Cx<double>{0.0, 0.0};
  chunk_combine<P, 1, M, J, PRE>(acc, Rs, b * n, n, bt, l);
  u32x4 q[M];
  float nrm;
  chunk_store<P, M>(E, b, l, acc[0], q, nrm, mx);
}

// The cycle's solution sum_k (-alpha_k) p_k with p_k = d_k + sum_j coef[k][j]
// p_j (A p_k = w_k) as sum_j beta_j d_j: beta_j = -alpha_j + sum_{k > j} beta_k
// coef[k][j], from the last step down (lane j holds beta_j).  keep_q1 drops the
// first step's -alpha_0 as invert.c:50-53 does.
__global__ void __launch_bounds__(64) k_scal_beta(GcrScal *scs, int n, int keep_q1, const int *ids) {
  GcrScal *sc = scs + ids[blockIdx.x];
  const int j = threadIdx.x;
  double2 b = make_double2(0.0, 0.0);
  if (j < n && !(j == 0 && keep_q1)) b = make_double2(-sc->alpha[j].x, -sc->alpha[j].y);
#pragma unroll 8
  for (int k = n - 1; k > 0; k--) {
    const double2 c = j < k ? sc->coef[k * kN + j] : make_double2(0.0, 0.0);
    const double2 p = cmul2(make_double2(__shfl(b.x, k, 64), __shfl(b.y, k, 64)), c);
    if (j < k) b = make_double2(b.x + p.x, b.y + p.y);
  }
  if (j < n) sc->beta[j] = b;
}

// outer residual norms from the Dslash partials (row x of the launch)
__global__ void __launch_bounds__(1024) k_scal_rnorm(GcrScal *scs, const double *part, unsigned nb, const int *ids,
                                                     double *rn) {
  __shared__ double sums[1];
  const int b = ids[blockIdx.x];
  wave_sums(part + (size_t)blockIdx.x * nb, 1, nb, sums);
  __syncthreads();
  if (threadIdx.x == 0) {
    GcrScal *sc = scs + b;
    sc->rnorm = sqrt(sums[0]);
    sc->rscale = sc->rnorm > 0.0 ? 1.0 / sc->rnorm : 0.0;
    rn[b] = sc->bad ? __builtin_nan("") : sc->rnorm;   // a breakdown reaches the host as NaN
  }
}

// res_0 = r / |r| in the inner precision P (r in precision PI)
template <int PI, int P>
__global__ void __launch_bounds__(kBlock) k_prepare_src(SpinorSet<PI> r, const GcrScal *sc, SpinorSet<P> Rs, int n,
                                                        const int *ids, unsigned V) {
  using R = typename Prec<P>::R;
  using RI = typename Prec<PI>::R;
  const int b = ids[blockIdx.y];
  const unsigned s = blockIdx.x * kBlock + threadIdx.x;
  if (s >= V) return;
  const double f = sc[b].rscale;
  Cx<RI> v[12];
  r.load(b, s, v);
  Cx<R> o[12];
#pragma unroll
  for (int c = 0; c < 12; c++) o[c] = Cx<R>{(R)((double)v[c].re * f), (R)((double)v[c].im * f)};
  Rs.store(b * n, s, o);
}

// x_{x0+b} += |r_b| e_b (FP64 accumulation of the inner correction)
template <int P>
__global__ void __launch_bounds__(kBlock) k_accumulate(SpinorSet<QCD_HIP_F64> X, int x0, SpinorSet<P> E,
                                                       const GcrScal *sc, const int *ids, unsigned V) {
  using R = typename Prec<P>::R;
  const int b = ids[blockIdx.y];
  const unsigned s = blockIdx.x * kBlock + threadIdx.x;
  if (s >= V) return;
  const double f = sc[b].rnorm;
  Cx<double> x[12];
  Cx<R> e[12];
  X.load(x0 + b, s, x);
  E.load(b, s, e);
#pragma unroll
  for (int c = 0; c < 12; c++) x[c] = Cx<double>{x[c].re + f * (double)e[c].re, x[c].im + f * (double)e[c].im};
  X.store(x0 + b, s, x);
}

// system right-hand side of slot b (i g5 b for Q, b for D) and x = 0
__global__ void __launch_bounds__(kBlock) k_start(SpinorSet<QCD_HIP_F64> B, SpinorSet<QCD_HIP_F64> X, int r0,
                                                  SpinorSet<QCD_HIP_F64> Bq, int use_q, unsigned V) {
  const int b = blockIdx.y;
  const unsigned s = blockIdx.x * kBlock + threadIdx.x;
  if (s >= V) return;
  Cx<double> v[12];
  B.load(r0 + b, s, v);
  if (use_q) {
#pragma unroll
    for (int c = 0; c < 6; c++) v[c] = ipow<1>(v[c]);
#pragma unroll
    for (int c = 6; c < 12; c++) v[c] = ipow<3>(v[c]);
  }
  Bq.store(b, s, v);
#pragma unroll
  for (int c = 0; c < 12; c++) v[c] = Cx<double>{0.0, 0.0};
  X.store(r0 + b, s, v);
}

}  // namespace qcdhip

using namespace qcdhip;

// ============================================================ solver object
struct qcd_hip_solver_s {
  qcd_hip_lattice lat;
  qcd_hip_solver_params prm;
  int B = 1;                        // right-hand sides per batch
  hipStream_t stream = nullptr;     // the solver's own stream
  qcd_hip_field g64 = nullptr;      // caller's FP64 gauge field (not owned)
  qcd_hip_field gin = nullptr;      // inner-precision copy (owned unless F64)
  qcd_hip_field Rs = nullptr;       // n*B directions d_j (inner precision)
  qcd_hip_field Ws = nullptr;       // n*B orthogonal vectors w_j (inner precision)
  qcd_hip_field E = nullptr;        // B inner corrections (inner precision)
  qcd_hip_field r64 = nullptr;      // B FP64 residuals (not allocated with split_res)
  // FP16-inner even-odd: the true residual is stored straight into the FP16
  // halves reh, roh and th = M^-1 reh, never as FP64
  bool split_res = false;
  qcd_hip_field bq = nullptr;       // B FP64 right-hand sides of the solved system
  GcrScal *sc = nullptr;            // B coefficient sets
  double *rn = nullptr;             // B residual norms (device)
  double *rn_host = nullptr;        // pinned mirror
  int *ids = nullptr;               // active slots (device)
  int *ids_host = nullptr;          // pinned mirror
  double *part = nullptr;
  size_t part_bytes = 0, rowsz = 0;
  unsigned nb = 0;                   // site-kernel workgroups (full lattice)
  // even-odd preconditioning (prm.eo): the inner GCR runs on the Schur
  // complement D^ over odd-site half vectors
  bool use_q = true;                 // outer system Q x = i g5 b (else D x = b)
  qcd_hip_lattice half = nullptr;    // half lattice of the inner vectors (owned)
  unsigned Vi = 0, nbi = 0;          // inner vector sites and site-kernel workgroups
  qcd_hip_field te = nullptr;        // EO: B inner even temporaries of the matvec
  // EO: B half vectors each for the outer step: even and odd residual halves,
  // M^-1 temporaries, the odd correction; FP64 for an FP64 inner solve, the
  // inner precision otherwise
  qcd_hip_field reh = nullptr, roh = nullptr, th = nullptr, eoh = nullptr;
  bool single = false;               // GCR steps one by one (solve_rhs)
  // the captured GCR cycle (prm.graph) and the launch arguments it was
  // captured with; every buffer it touches belongs to the solver
  hipGraphExec_t cycle = nullptr;
  int cycle_count = 0;
  double cycle_kappa = 0.0, cycle_mu = 0.0;
  void drop_cycle() {
    if (!cycle) return;
    (void)hipStreamSynchronize(stream);   // no replay may still be running
    (void)hipGraphExecDestroy(cycle);
    cycle = nullptr;
  }
};

namespace {

// Work split of the GCR vector kernels: M chunks per lane, J vectors in flight
// (PRE: and the next J on their way), BLK lanes per workgroup.  Chosen by the
// vector length alone, so that a right-hand side gets the same sums alone and in
// any batch.
//   Short FP64 and FP32 vectors: one chunk per lane, so that they still put a few
//     wavefronts on every SIMD.  Solves, ms, Short against long: 8^3x16 even-odd,
//     one FP64 rhs, GCR(32) 1.31 / 1.70, three FP32, GCR(16) 0.98 / 1.05.  9216
//     sites: FP64 1.55 / 1.81, FP32 1.28 / 1.30; 16 128 sites: both 2% slower.
//   FP16 vectors: one chunk per lane at every length; a tile's three wavefronts
//     share a workgroup, which finds the site norms.  Two vectors in flight in the
//     dots; in the kernels without sums too up to 4096 sites, one from there (8^3x16,
//     twelve, GCR(32): k_solution 17.5 against 23.0 us, the solve 2.82 against 2.84 ms;
//     16^3x32 20.45 against 20.14).
//   Long ones: what measured best, us per launch (12 FP16 rhs, GCR(12), 24^3x48;
//     one FP64 rhs, GCR(32), 16^3x32; three FP32, GCR(16), 16^3x24, even-odd).
//     FP16 dots: a third of a site, two vectors 496, one 508, three 618, a whole
//     site 542 (its vectors in FP64 take all registers); they are bound by the FP64
//     arithmetic.  FP16 update: a third of a site, 192 lanes 501 (four
//     wavefronts per SIMD; with six registers more, three, 652), 384 lanes 594,
//     two vectors in flight 519, a whole site (its four FP64 accumulators leave
//     one wavefront per SIMD) 746.  FP64 dots: half a site 71, a whole one 115;
//     update 96 and 97 to 100.  FP32 dots: half a site, one vector, 256 lanes
//     29.4, two vectors 32.9, 512 lanes 37.6; update 37.2 to 38.9.
//   Blocks of 8 hold twice the vectors and accumulators.  FP64 (as above) dots: a
//     quarter of a site, 256 lanes 86, 512 lanes 101, a third of a site 90, a
//     sixth 96; update: a quarter 119.5, a third 119.4, a sixth 125 to 127.  FP32
//     on 16^3x32, Q, GCR(32), dots: a third of a site, PRE 64, without 73, half a
//     site 86, a sixth 83; update: a sixth 66, a third 68, half a site 78.
template <int M_, int J_, int BLK_, bool PRE_>
struct GcrShape {
  static constexpr int M = M_, J = J_, BLK = BLK_;
  static constexpr bool PRE = PRE_;
};
template <int P>
struct GcrShapes;
template <>
struct GcrShapes<QCD_HIP_F16> {
  static constexpr int S = 4;   // steps of a block
  using Dots = GcrShape<1, 2, 192, true>;
  using Update = GcrShape<1, 1, 192, true>;
};
template <>
struct GcrShapes<QCD_HIP_F32> {
  static constexpr int S = 8;
  using Short = GcrShape<1, 4, 256, true>;
  using Dots = GcrShape<3, 1, 256, false>;
  using Update = GcrShape<3, 1, 256, false>;
  using Short8 = GcrShape<1, 2, 256, true>;
  using Dots8 = GcrShape<2, 1, 256, true>;
  using Update8 = GcrShape<1, 2, 256, true>;
};
template <>
struct GcrShapes<QCD_HIP_F64> {
  static constexpr int S = 8;
  using Short = GcrShape<1, 4, 256, true>;
  using Dots = GcrShape<6, 1, 512, false>;
  using Update = GcrShape<6, 1, 256, false>;
  using Short8 = GcrShape<1, 2, 256, true>;
  using Dots8 = GcrShape<3, 1, 256, false>;
  using Update8 = GcrShape<3, 1, 256, false>;
};
template <typename SH>
unsigned gcr_blocks(int prec, long V) {
  const long kG = 12 * (long)spinor_comp_bytes(prec) / 16;
  const long waves = (V + kTile - 1) / kTile * (kG / SH::M);
  return (unsigned)((waves + SH::BLK / 64 - 1) / (SH::BLK / 64));
}
// f(shape, grid) of a launch over count vectors of V sites (DOTS: the dots'
// shape, else that of the kernels without sums) in a block of ST steps
template <int P, int ST, bool DOTS, typename F>
void gcr_launch(long V, int count, F f) {
  using G = GcrShapes<P>;
  auto call = [&](auto sh) { f(sh, dim3(gcr_blocks<decltype(sh)>(P, V), (unsigned)count)); };
  constexpr long kShort = 12288;
  if constexpr (P == QCD_HIP_F16) {
    if (DOTS || V <= 4096) call(typename G::Dots{});
    else call(typename G::Update{});
  } else if constexpr (ST == 8) {
    if (V <= kShort) call(typename G::Short8{});
    else call(std::conditional_t<DOTS, typename G::Dots8, typename G::Update8>{});
  } else {
    if (V <= kShort) call(typename G::Short{});
    else call(std::conditional_t<DOTS, typename G::Dots, typename G::Update>{});
  }
}
// f(block size constant) for the next block of a cycle with left steps to go
template <int P, typename F>
int gcr_next(int left, bool single, F f) {
  constexpr int S = GcrShapes<P>::S;
  if (single) return f(std::integral_constant<int, 1>{});
  if constexpr (S >= 8)
    if (left >= 8) return f(std::integral_constant<int, 8>{});
  if (left >= 4) return f(std::integral_constant<int, 4>{});
  if (left >= 2) return f(std::integral_constant<int, 2>{});
  return f(std::integral_constant<int, 1>{});
}
// More partial sums than kGcrParts are added up in up to kGcrSums groups first.
constexpr unsigned kGcrParts = 256, kGcrSums = 64;

// Steps k .. k + ST - 1 of the cycle (prev: of the block before), the hops of
// matvec(out, out slot, in slot) included
template <int P, int ST, typename F>
int gcr_block(qcd_hip_solver_s *S, int count, int k, int prev, double theta, hipStream_t st, F matvec) {
  const int n = S->prm.n_restart;
  const unsigned V = S->Vi;
  SpinorSet<P> Rs = SpinorSet<P>::of(S->Rs), Ws = SpinorSet<P>::of(S->Ws);
  for (int a = 0; a < ST; a++) {
    const bool last = a == ST - 1;
    QH_TRY(matvec(last ? S->Ws : S->Rs, last ? k + a : k + a + 1, k + a));
  }
  gcr_launch<P, ST, true>(V, count, [&](auto sh, dim3 grid) {
    using SH = decltype(sh);
    k_gcr_dots<P, ST, SH::M, SH::J, SH::BLK, SH::PRE><<<grid, SH::BLK, 0, st>>>(Ws, Rs, n, k, prev, S->ids, V, S->part,
                                                                       S->rowsz);
    unsigned np = grid.x;
    const double *part = S->part;
    if (np > kGcrParts) {
      const unsigned nv = gcr_values<ST>(k), c = std::max(32u, (np + kGcrSums - 1) / kGcrSums), g = (np + c - 1) / c;
      k_gcr_sum<<<dim3(g, (unsigned)count), 256, 0, st>>>(S->part, S->rowsz, np, nv, c);
      part += (size_t)np * nv;
      np = g;
    }
    k_gcr_scal<P, ST><<<count, 1024, 0, st>>>(S->sc, part, S->rowsz, np, k, prev, theta, S->ids);
  });
  if (k + ST < n)   // the last w and the residual after them are not used
    gcr_launch<P, ST, false>(V, count, [&](auto sh, dim3 grid) {
      using SH = decltype(sh);
      k_gcr_update<P, ST, SH::M, SH::J, SH::BLK, SH::PRE><<<grid, SH::BLK, 0, st>>>(Ws, Rs, n, k, theta, S->sc, S->ids, V);
    });
  return 0;
}

template <int P>
int gcr_cycle(qcd_hip_solver_s *S, int count, double kappa, double mu, hipStream_t st) {
  const int n = S->prm.n_restart;
  const unsigned V = S->Vi;
  const int epi = S->use_q ? EPI_Q : EPI_D;
  const double m = 1.0 / (2.0 * kappa) - 4.0;
  SpinorSet<P> Rs = SpinorSet<P>::of(S->Rs), E = SpinorSet<P>::of(S->E);
  // Q, and the local term left out of D and of the Schur complement
  const double theta = S->use_q ? 0.0 : m + 4.0;
  // out = (A - theta) Rs[slot ri]
  auto matvec = [&](qcd_hip_field out, int ro, int ri) -> int {
    if (S->prm.eo) {
      // D^ r = M r - H_oe (M^-1 H_eo r)
      QH_TRY(eo_launch(EO_MINV, false, S->te, 0, 1, S->Rs, ri, n, S->gin, nullptr, 0, 0, S->ids, count, m, mu, 0,
                       nullptr, st, nullptr));
      return eo_launch(EO_SCHUR, false, out, ro, n, S->te, 0, 1, S->gin, S->Rs, ri, n, S->ids, count, m - theta, mu, 1,
                       nullptr, st, nullptr);
    }
    return dslash_launch_batch(epi, false, out, ro, n, S->Rs, ri, n, S->gin, nullptr, 0, 0, S->ids, count, m - theta,
                               mu, nullptr, st, nullptr);
  };
  for (int k = 0, prev = 0; k < n; k += prev)
    QH_TRY(gcr_next<P>(n - k, S->single, [&](auto st_c) -> int {
      constexpr int ST = decltype(st_c)::value;
      QH_TRY((gcr_block<P, ST>(S, count, k, prev, theta, st, matvec)));
      prev = ST;
      return 0;
    }));
  k_scal_beta<<<count, 64, 0, st>>>(S->sc, n, S->prm.keep_q1, S->ids);
  // mixed even-odd solves take the correction scaled by |r^_o| (the outer
  // step adds it as it is); the others scale it where they add it
  const int scaled = S->prm.eo && S->prm.inner_prec != QCD_HIP_F64;
  gcr_launch<P, 1, false>(V, count, [&](auto sh, dim3 grid) {
    using SH = decltype(sh);
    k_solution<P, SH::M, SH::J, SH::BLK, SH::PRE><<<grid, SH::BLK, 0, st>>>(Rs, n, S->sc, E, S->ids, V, scaled);
  });
  QH_CHECK(hipGetLastError());
  return 0;
}

// One GCR cycle on stream st.  With prm.graph the launches of gcr_cycle are
// captured into a graph once per (active rhs count, kappa, mu) and the graph
// is replayed: the kernels read the active-slot list and every coefficient
// from device memory, so a replay is the same work as the eager launches.
// The cycle records no memset or copy nodes.
template <int P>
int run_cycle(qcd_hip_solver_s *S, int count, double kappa, double mu, hipStream_t st) {
  if (!S->prm.graph) return gcr_cycle<P>(S, count, kappa, mu, st);
  if (!S->cycle || S->cycle_count != count || S->cycle_kappa != kappa || S->cycle_mu != mu) {
    S->drop_cycle();
    if (S->prm.eo) {
      // the cycle's first matvec once, eagerly: hop launch shapes seen for the
      // first time are tuned here, which cannot happen under capture (both
      // results are recomputed by the cycle)
      const double m = 1.0 / (2.0 * kappa) - 4.0;
      const int n = S->prm.n_restart;
      QH_TRY(eo_launch(EO_MINV, false, S->te, 0, 1, S->Rs, 0, n, S->gin, nullptr, 0, 0, S->ids, count, m, mu, 0,
                       nullptr, st, nullptr));
      QH_TRY(eo_launch(EO_SCHUR, false, S->Ws, 0, n, S->te, 0, 1, S->gin, S->Rs, 0, n, S->ids, count, m, mu, 1,
                       nullptr, st, nullptr));
    }
    QH_CHECK(hipStreamBeginCapture(st, hipStreamCaptureModeRelaxed));
    const int rc = gcr_cycle<P>(S, count, kappa, mu, st);
    hipGraph_t graph = nullptr;
    const hipError_t e = hipStreamEndCapture(st, &graph);
    if (rc) {
      if (graph) (void)hipGraphDestroy(graph);
      return rc;
    }
    QH_CHECK(e);
    const hipError_t ei = hipGraphInstantiate(&S->cycle, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (ei != hipSuccess) S->cycle = nullptr;
    QH_CHECK(ei);
    S->cycle_count = count;
    S->cycle_kappa = kappa;
    S->cycle_mu = mu;
  }
  QH_CHECK(hipGraphLaunch(S->cycle, st));
  return 0;
}

template <int P>
int outer_step(qcd_hip_solver_s *S, qcd_hip_field x, int x0, int count, double kappa, double mu, hipStream_t st) {
  const dim3 g2(S->nbi, (unsigned)count);
  const unsigned V = S->Vi;
  if (!S->prm.eo) {
    k_prepare_src<QCD_HIP_F64, P><<<g2, kBlock, 0, st>>>(SpinorSet<QCD_HIP_F64>::of(S->r64), S->sc,
                                                         SpinorSet<P>::of(S->Rs), S->prm.n_restart, S->ids, V);
    QH_TRY(run_cycle<P>(S, count, kappa, mu, st));
    k_accumulate<P><<<g2, kBlock, 0, st>>>(SpinorSet<QCD_HIP_F64>::of(x), x0, SpinorSet<P>::of(S->E), S->sc, S->ids,
                                           V);
    QH_CHECK(hipGetLastError());
    return 0;
  }
  // Even-odd: D e = r  <=>  D^ e_o = r_o - H_oe M^-1 r_e,  e_e = M^-1 (r_e - H_eo e_o)
  const double m = 1.0 / (2.0 * kappa) - 4.0;
  const size_t sstride = sizeof(GcrScal) / sizeof(double);
  int grid = 0;
  if constexpr (P == QCD_HIP_F64) {
    QH_TRY(eo_split(S->r64, 0, S->reh, S->roh, S->ids, count, st));
    QH_TRY(eo_minv(S->lat, S->reh, S->th, m, mu, S->ids, count, st));
    QH_TRY(eo_launch(EO_SUB, true, S->eoh, 0, 1, S->th, 0, 1, S->g64, S->roh, 0, 1, S->ids, count, m, mu, 1, S->part,
                     st, &grid));
    k_scal_rnorm<<<count, 1024, 0, st>>>(S->sc, S->part, (unsigned)grid, S->ids, S->rn);   // |r^_o| for the scaling
    k_prepare_src<QCD_HIP_F64, P><<<g2, kBlock, 0, st>>>(SpinorSet<QCD_HIP_F64>::of(S->eoh), S->sc,
                                                         SpinorSet<P>::of(S->Rs), S->prm.n_restart, S->ids, V);
    QH_CHECK(hipGetLastError());
    QH_TRY(run_cycle<P>(S, count, kappa, mu, st));
    QH_TRY(eo_scale64(S->lat, S->E, S->eoh, &S->sc[0].rnorm, sstride, S->ids, count, st));
    QH_TRY(eo_launch(EO_SUB_MINV, false, S->th, 0, 1, S->eoh, 0, 1, S->g64, S->reh, 0, 1, S->ids, count, m, mu, 0,
                     nullptr, st, nullptr));
    QH_TRY(eo_accumulate(x, x0, S->th, S->eoh, S->ids, count, st));
    return 0;
  }
  // Mixed precision: only the true residual, the accumulation into x and the
  // reductions are FP64.  The halves of the residual (reh, roh and th =
  // M^-1 reh; FP16: written by the true residual itself), the inner source
  // r^_o and the even correction e_e are in the inner precision, with the
  // inner-precision links: their rounding only perturbs the correction of this
  // outer step, which the next FP64 true residual measures.
  if (!S->split_res) QH_TRY(eo_split_minv(S->r64, 0, S->reh, S->roh, S->th, m, mu, S->ids, count, st));
  QH_TRY(eo_launch(EO_SUB, true, S->eoh, 0, 1, S->th, 0, 1, S->gin, S->roh, 0, 1, S->ids, count, m, mu, 1, S->part,
                   st, &grid));
  k_scal_rnorm<<<count, 1024, 0, st>>>(S->sc, S->part, (unsigned)grid, S->ids, S->rn);   // |r^_o| for the scaling
  k_prepare_src<P, P><<<g2, kBlock, 0, st>>>(SpinorSet<P>::of(S->eoh), S->sc, SpinorSet<P>::of(S->Rs),
                                             S->prm.n_restart, S->ids, V);
  QH_CHECK(hipGetLastError());
  QH_TRY(run_cycle<P>(S, count, kappa, mu, st));
  QH_TRY(eo_launch(EO_SUB_MINV, false, S->th, 0, 1, S->E, 0, 1, S->gin, S->reh, 0, 1, S->ids, count, m, mu, 0,
                   nullptr, st, nullptr));
  QH_TRY(eo_accumulate_p(x, x0, S->th, S->E, S->ids, count, st));
  return 0;
}

// r_b = bq_b - A x_{x0+b} for the active slots; residual norms to rn_host
int true_residual(qcd_hip_solver_s *S, qcd_hip_field x, int x0, int count, double kappa, double mu, hipStream_t st) {
  const int epi = S->use_q ? EPI_RES_Q : EPI_RES_D;
  const double m = 1.0 / (2.0 * kappa) - 4.0;
  int grid = 0;
  if (S->split_res)
    QH_TRY(dslash_residual_eo_split(x, x0, 1, S->g64, S->bq, 0, 1, S->ids, count, m, mu, S->reh, S->roh, S->th,
                                    S->part, st, &grid));
  else
    QH_TRY(dslash_launch_batch(epi, true, S->r64, 0, 1, x, x0, 1, S->g64, S->bq, 0, 1, S->ids, count, m, mu, S->part,
                               st, &grid));
  k_scal_rnorm<<<count, 1024, 0, st>>>(S->sc, S->part, (unsigned)grid, S->ids, S->rn);
  QH_CHECK(hipGetLastError());
  QH_CHECK(hipMemcpyAsync(S->rn_host, S->rn, sizeof(double) * S->B, hipMemcpyDeviceToHost, st));
  QH_CHECK(hipStreamSynchronize(st));
  return 0;
}

int upload_ids(qcd_hip_solver_s *S, const std::vector<int> &ids, hipStream_t st) {
  for (size_t i = 0; i < ids.size(); i++) S->ids_host[i] = ids[i];
  QH_CHECK(hipMemcpyAsync(S->ids, S->ids_host, sizeof(int) * ids.size(), hipMemcpyHostToDevice, st));
  QH_CHECK(hipStreamSynchronize(st));   // the pinned mirror is reused next step
  return 0;
}

// Solve rhs [x0, x0 + cnt) of b into x; *broke: a breakdown ended it.
int solve_batch(qcd_hip_solver_s *S, qcd_hip_field x, qcd_hip_field b, int x0, int cnt, double kappa, double mu,
                hipStream_t st, qcd_hip_solver_stats *tot, int *worst, bool *broke) {
  const unsigned V = (unsigned)S->lat->V;
  k_start<<<dim3(S->nb, (unsigned)cnt), kBlock, 0, st>>>(SpinorSet<QCD_HIP_F64>::of(b), SpinorSet<QCD_HIP_F64>::of(x),
                                                         x0, SpinorSet<QCD_HIP_F64>::of(S->bq), S->use_q, V);
  QH_CHECK(hipGetLastError());
  QH_CHECK(hipMemsetAsync(S->sc, 0, sizeof(GcrScal) * S->B, st));
  std::vector<int> act(cnt);
  for (int i = 0; i < cnt; i++) act[i] = i;
  QH_TRY(upload_ids(S, act, st));
  QH_TRY(true_residual(S, x, x0, cnt, kappa, mu, st));
  std::vector<double> bnorm(cnt), rel(cnt);
  std::vector<int> outer(cnt, 0);
  for (int i = 0; i < cnt; i++) {
    bnorm[i] = S->rn_host[i];
    rel[i] = bnorm[i] > 0.0 ? 1.0 : 0.0;
  }
  int bad = 0;
  std::vector<int> uploaded = act;   // the list the device holds
  for (int it = 0; it < S->prm.max_outer; it++) {
    act.clear();
    for (int i = 0; i < cnt; i++)
      if (rel[i] > S->prm.tol) act.push_back(i);
    if (act.empty()) break;
    if (act != uploaded) {   // most outer steps keep every rhs active: no upload, no host round trip
      QH_TRY(upload_ids(S, act, st));
      uploaded = act;
    }
    const int na = (int)act.size();
    switch (S->prm.inner_prec) {
      case QCD_HIP_F64: QH_TRY(outer_step<QCD_HIP_F64>(S, x, x0, na, kappa, mu, st)); break;
      case QCD_HIP_F32: QH_TRY(outer_step<QCD_HIP_F32>(S, x, x0, na, kappa, mu, st)); break;
      default: QH_TRY(outer_step<QCD_HIP_F16>(S, x, x0, na, kappa, mu, st)); break;
    }
    QH_TRY(true_residual(S, x, x0, na, kappa, mu, st));
    for (int i : act) {
      outer[i]++;
      rel[i] = S->rn_host[i] / bnorm[i];
      if (!(rel[i] == rel[i])) bad = 1;
    }
    if (bad) break;
  }
  for (int i = 0; i < cnt; i++) {
    tot->outer += outer[i];
    tot->inner_iters += outer[i] * S->prm.n_restart;
    tot->relres = std::max(tot->relres, rel[i]);
    if (!bad && rel[i] > S->prm.tol) *worst = std::max(*worst, 6);
  }
  *broke = bad;
  return 0;
}

// solve_batch, and after a breakdown once more with single GCR steps.  A block
// applies the operator up to eight times without a normalisation: eight powers
// of a norm of 6e4 (kappa 1e-5, Q) or single ones of links far from SU(3) leave
// the range of FP32, which a step at a time stays in.
int solve_rhs(qcd_hip_solver_s *S, qcd_hip_field x, qcd_hip_field b, int x0, int cnt, double kappa, double mu,
              hipStream_t st, qcd_hip_solver_stats *tot, int *worst) {
  const qcd_hip_solver_stats before = *tot;
  const int worst0 = *worst;
  bool broke = false;
  QH_TRY(solve_batch(S, x, b, x0, cnt, kappa, mu, st, tot, worst, &broke));
  if (broke) {
    *tot = before;
    *worst = worst0;
    S->drop_cycle();
    S->single = true;
    const int rc = solve_batch(S, x, b, x0, cnt, kappa, mu, st, tot, worst, &broke);
    S->drop_cycle();
    S->single = false;
    QH_TRY(rc);
  }
  if (broke) *worst = 5;
  return 0;
}

}  // namespace

extern "C" {

void qcd_hip_solver_default_params(qcd_hip_solver_params *p) {
  std::memset(p, 0, sizeof(*p));
  p->n_restart = 32;
  p->max_outer = 10000;
  p->tol = 1e-10;
  p->inner_prec = QCD_HIP_F64;
  p->op = QCD_HIP_OP_Q;
  p->keep_q1 = 0;
  p->batch = 1;
  p->eo = 0;
  p->graph = 1;
}

}  // extern "C"

namespace qcdhip {
// Partial sums of one batch row: the dots of the last GCR step, or one sum per Dslash or hop workgroup (at most one per 256
// sites, and the z-march grids).
static size_t solver_row(qcd_hip_lattice lat, long Vi, const qcd_hip_solver_params *prm) {
  const int n = prm->n_restart;
  size_t dots = 0;
  auto blocks = [&](auto p) {
    constexpr int P = decltype(p)::value;
    for (bool single : {false, true})
      for (int k = 0; k < n;)
        k += gcr_next<P>(n - k, single, [&](auto st) -> int {
          constexpr int ST = decltype(st)::value;
          gcr_launch<P, ST, true>(Vi, 1, [&](auto, dim3 grid) {
            dots = std::max(dots, (size_t)(grid.x + kGcrSums) * gcr_values<ST>(k));
          });
          return ST;
        });
  };
  if (prm->inner_prec == QCD_HIP_F64) blocks(std::integral_constant<int, QCD_HIP_F64>{});
  else if (prm->inner_prec == QCD_HIP_F32) blocks(std::integral_constant<int, QCD_HIP_F32>{});
  else blocks(std::integral_constant<int, QCD_HIP_F16>{});
  return std::max(dots, std::max((size_t)grid_for(lat->V) + 64, (size_t)dslash_grid_bound(lat)));
}

// Device bytes qcd_hip_solver_create and qcd_hip_solver_set_gauge allocate
// for a lattice of extents L with parameters prm: the same field shapes and
// reduction rows, without allocating anything.
size_t solver_device_bytes(const int L[4], const qcd_hip_solver_params *prm) {
  qcd_hip_lattice_s lat{};
  for (int d = 0; d < 4; d++) lat.L[d] = L[d];
  lat.V = (long)L[0] * L[1] * L[2] * L[3];
  lat.stride = round_up(lat.V, kTile);
  auto field = [](long stride, int prec, int nrhs) {
    return (size_t)12 * nrhs * stride * spinor_comp_bytes(prec) + (prec == QCD_HIP_F16 ? (size_t)4 * nrhs * stride : 0);
  };
  const int n = prm->n_restart, B = prm->batch, ip = prm->inner_prec;
  const long V = lat.V;
  const long Vi = prm->eo ? V / 2 : V;
  const long sti = round_up(Vi, kTile);
  size_t b = 0;
  b += 2 * field(sti, ip, n * B) + field(sti, ip, B);                  // Rs, Ws, E
  if (prm->eo) b += 5 * field(sti, ip, B);                             // te, reh, roh, th, eoh
  const bool split = prm->eo && ip == QCD_HIP_F16;                     // no r64 (split residual)
  b += (split ? 1 : 2) * field(lat.stride, QCD_HIP_F64, B);            // r64, bq
  b += sizeof(GcrScal) * B + sizeof(double) * B + sizeof(int) * B;      // sc, rn, ids
  b += sizeof(double) * solver_row(&lat, Vi, prm) * B;                 // partials
  if (ip != QCD_HIP_F64) b += (size_t)36 * lat.stride * spinor_comp_bytes(ip);   // inner-precision links
  if (ip == QCD_HIP_F16) b += (size_t)8 * 36 * lat.V;                            // matrix-core hop links
  return b;
}
}  // namespace qcdhip

extern "C" {

size_t qcd_hip_solver_bytes(const int L[4], const qcd_hip_solver_params *prm) {
  if (!L || !prm || prm->n_restart < 1 || prm->batch < 1 || L[0] < 1 || L[1] < 1 || L[2] < 1 || L[3] < 1) return 0;
  return solver_device_bytes(L, prm);
}

int qcd_hip_solver_create(qcd_hip_solver *out, qcd_hip_lattice lat, const qcd_hip_solver_params *prm) {
  *out = nullptr;
  QH_TRY(ensure_init());
  if (!lat || !prm || prm->n_restart < 1 || prm->n_restart > kN || prm->tol <= 0.0 || prm->max_outer < 1 ||
      prm->inner_prec < QCD_HIP_F64 || prm->inner_prec > QCD_HIP_F16 || prm->batch < 1 || prm->batch > 1024 ||
      (prm->op != QCD_HIP_OP_Q && prm->op != QCD_HIP_OP_D) || (prm->eo != 0 && prm->eo != 1) ||
      (prm->graph != 0 && prm->graph != 1)) {
    set_error("solver_create: bad parameters (n_restart 1..%d, tol > 0, max_outer >= 1, batch 1..1024, eo 0/1, "
              "graph 0/1)", kN);
    return 1;
  }
  if (prm->eo && !eo_supported(lat)) {
    set_error("solver_create: even-odd preconditioning needs every lattice extent even");
    return 1;
  }
  auto *S = new qcd_hip_solver_s();
  S->lat = lat;
  S->prm = *prm;
  if (hipStreamCreateWithFlags(&S->stream, hipStreamNonBlocking) != hipSuccess) {
    delete S;
    set_error("solver_create: cannot create a stream");
    return 2;
  }
  S->B = prm->batch;
  S->nb = (unsigned)grid_for(lat->V);
  S->use_q = prm->op == QCD_HIP_OP_Q && !prm->eo;   // the EO inner system is D's Schur complement
  qcd_hip_lattice ilat = lat;
  if (prm->eo) ilat = S->half = eo_half_lattice(lat);
  S->Vi = (unsigned)ilat->V;
  S->nbi = (unsigned)grid_for(ilat->V);
  const int n = prm->n_restart, B = S->B;
  int rc = qcd_hip_spinor_create(&S->Rs, ilat, prm->inner_prec, n * B);
  if (!rc) rc = qcd_hip_spinor_create(&S->Ws, ilat, prm->inner_prec, n * B);
  if (!rc) rc = qcd_hip_spinor_create(&S->E, ilat, prm->inner_prec, B);
  if (!rc && prm->eo) rc = qcd_hip_spinor_create(&S->te, ilat, prm->inner_prec, B);
  for (qcd_hip_field *f : {&S->reh, &S->roh, &S->th, &S->eoh})
    if (!rc && prm->eo) rc = qcd_hip_spinor_create(f, ilat, prm->inner_prec, B);
  S->split_res = prm->eo && prm->inner_prec == QCD_HIP_F16;
  if (!rc && !S->split_res) rc = qcd_hip_spinor_create(&S->r64, lat, QCD_HIP_F64, B);
  if (!rc) rc = qcd_hip_spinor_create(&S->bq, lat, QCD_HIP_F64, B);
  if (!rc) rc = dev_alloc((void **)&S->sc, sizeof(GcrScal) * B);
  if (!rc) rc = dev_alloc((void **)&S->rn, sizeof(double) * B);
  if (!rc) rc = dev_alloc((void **)&S->ids, sizeof(int) * B);
  if (!rc && hipHostMalloc((void **)&S->rn_host, sizeof(double) * B, hipHostMallocDefault) != hipSuccess) rc = 4;
  if (!rc && hipHostMalloc((void **)&S->ids_host, sizeof(int) * B, hipHostMallocDefault) != hipSuccess) rc = 4;
  S->rowsz = solver_row(lat, (long)S->Vi, prm);
  S->part_bytes = sizeof(double) * S->rowsz * B;
  if (!rc) rc = dev_alloc((void **)&S->part, S->part_bytes);
  if (rc) {
    if (rc == 4) set_error("solver_create: out of memory for %d rhs x %d Krylov vectors", B, n);
    qcd_hip_solver_destroy(S);
    return rc;
  }
  *out = S;
  return 0;
}

void qcd_hip_solver_destroy(qcd_hip_solver S) {
  if (!S) return;
  S->drop_cycle();
  qcd_hip_field_destroy(S->Rs);
  qcd_hip_field_destroy(S->Ws);
  qcd_hip_field_destroy(S->E);
  qcd_hip_field_destroy(S->r64);
  qcd_hip_field_destroy(S->bq);
  for (qcd_hip_field f : {S->te, S->reh, S->roh, S->th, S->eoh}) qcd_hip_field_destroy(f);
  if (S->gin && S->gin != S->g64) qcd_hip_field_destroy(S->gin);
  if (S->stream) {
    (void)hipStreamSynchronize(S->stream);
    (void)hipStreamDestroy(S->stream);
  }
  dev_free(S->sc, sizeof(GcrScal) * S->B);
  dev_free(S->rn, sizeof(double) * S->B);
  dev_free(S->ids, sizeof(int) * S->B);
  dev_free(S->part, S->part_bytes);
  if (S->rn_host) (void)hipHostFree(S->rn_host);
  if (S->ids_host) (void)hipHostFree(S->ids_host);
  delete S->half;
  delete S;
}

int qcd_hip_solver_set_gauge(qcd_hip_solver S, qcd_hip_field g64) {
  QH_TRY(ensure_init());
  if (!S || !g64 || g64->kind != QCD_HIP_GAUGE || g64->prec != QCD_HIP_F64 || g64->lat->V != S->lat->V) {
    set_error("solver_set_gauge: need an FP64 gauge field on the solver's lattice");
    return 1;
  }
  S->g64 = g64;
  S->drop_cycle();   // the captured cycle holds the previous field's pointers
  if (S->prm.inner_prec == QCD_HIP_F64) {
    if (S->gin && S->gin != g64) qcd_hip_field_destroy(S->gin);
    S->gin = g64;
    return 0;
  }
  if (!S->gin || S->gin == g64) {
    S->gin = nullptr;
    QH_TRY(qcd_hip_gauge_create(&S->gin, S->lat, S->prm.inner_prec));
  }
  QH_TRY(qcd_hip_field_convert(S->gin, g64));
  if (S->prm.inner_prec == QCD_HIP_F16) {
    // the matrix-core hops read phased links prepared once per gauge field
    QH_TRY(mma_prepare(S->gin, S->lat, ctx()->stream));
    QH_CHECK(hipStreamSynchronize(ctx()->stream));
  }
  return 0;
}

int qcd_hip_solver_solve(qcd_hip_solver S, qcd_hip_field x, qcd_hip_field b, double kappa, double mu,
                         qcd_hip_solver_stats *stats) {
  QH_TRY(ensure_init());
  if (!S || !S->g64) {
    set_error("solver_solve: no gauge field set (qcd_hip_solver_set_gauge)");
    return 1;
  }
  if (!x || !b || x->kind != QCD_HIP_SPINOR || b->kind != QCD_HIP_SPINOR || x->prec != QCD_HIP_F64 ||
      b->prec != QCD_HIP_F64 || x->nrhs != b->nrhs || x->lat->V != S->lat->V || b->lat->V != S->lat->V) {
    set_error("solver_solve: x and b must be FP64 spinors with equal rhs counts on the solver's lattice");
    return 1;
  }
  if (x == b) {
    set_error("solver_solve: x must not alias b");
    return 1;
  }
  if (kappa <= 0.0) {
    set_error("solver_solve: kappa must be positive");
    return 1;
  }
  hipStream_t st = S->stream;
  const auto t0 = std::chrono::steady_clock::now();
  // Tune the inner and outer operators before the first timed use.
  if (!S->prm.eo) QH_TRY(dslash_prepare(S->Ws, S->Rs, S->gin));
  // (scratch output of the tuning launches: r64, or bq, which each batch
  // fills afterwards)
  QH_TRY(dslash_prepare(S->r64 ? S->r64 : S->bq, x, S->g64));
  qcd_hip_solver_stats tot;
  std::memset(&tot, 0, sizeof(tot));
  int worst = 0;
  for (int r0 = 0; r0 < b->nrhs && worst != 5; r0 += S->B) {
    const int cnt = std::min(S->B, b->nrhs - r0);
    QH_TRY(solve_rhs(S, x, b, r0, cnt, kappa, mu, st, &tot, &worst));
  }
  tot.seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  if (stats) *stats = tot;
  if (worst == 5) set_error("solver: Krylov space breakdown (NaN or zero norm)");
  if (worst == 6) set_error("solver: not converged to %g within %d outer iterations (reached %g)", S->prm.tol,
                            S->prm.max_outer, tot.relres);
  return worst;
}

// ||D x - b|| / ||b|| in FP64 with m = 1/(2 kappa) - 4 (b_minus_Dx.c:152-167)
int qcd_hip_b_minus_Dx(qcd_hip_field x, int rx, qcd_hip_field b, int rb, qcd_hip_field g, double kappa, double mu,
                       double *rel) {
  std::lock_guard<std::recursive_mutex> lock(state_mutex());   // shared scratch field and stream
  QH_TRY(ensure_init());
  if (!x || !b || !g || x->prec != QCD_HIP_F64 || b->prec != QCD_HIP_F64 || g->prec != QCD_HIP_F64 || !rel ||
      rx < 0 || rx >= x->nrhs || rb < 0 || rb >= b->nrhs) {
    set_error("b_minus_Dx: needs FP64 x, b and gauge field");
    return 1;
  }
  QH_TRY(dslash_check(x, b, g));
  qcd_hip_field r = nullptr;
  QH_TRY(scratch_spinor(1, x->lat, QCD_HIP_F64, 1, &r));
  hipStream_t st = ctx()->stream;
  QH_TRY(dslash_prepare(r, x, g));
  int grid = 0;
  Context *c = ctx();
  const size_t need = sizeof(double) * (size_t)(dslash_grid(x, g) + 64);
  double *part = nullptr;
  QH_TRY(dev_alloc((void **)&part, need));
  int rc = dslash_launch(EPI_RES_D, true, r, 0, x, rx, g, b, rb, 1.0 / (2.0 * kappa) - 4.0, mu, part, st, &grid);
  if (!rc) rc = finalize(part, grid, 1, c->scalars, st);
  double num = 0.0, den = 0.0;
  if (!rc) rc = hipMemcpyAsync(&num, c->scalars, sizeof(double), hipMemcpyDeviceToHost, st) ? 2 : 0;
  if (!rc) rc = hipStreamSynchronize(st) ? 2 : 0;
  dev_free(part, need);
  QH_TRY(rc);
  QH_TRY(qcd_hip_norm2(b, rb, &den));
  *rel = std::sqrt(num) / std::sqrt(den);
  return 0;
}

}  // extern "C"

// ------------------------------------------------------------ allocation-free residual
// qcd_hip_b_minus_Dx_noalloc keeps its workgroup partial sums and the two
// finished sums in this array instead of library allocations: at most
// kNoAllocParts Dslash workgroups (every launch configuration of a 2^24-site
// lattice fits), kMaxReduceBlocks norm partials and 2 results, 2.0 MiB per
// GPU, held until the process ends.  In host code `scratch` only names the
// symbol; kernels get its device address from noalloc_scratch().
namespace {
constexpr size_t kNoAllocParts = (size_t)1 << 18;
constexpr size_t kNoAllocNorm = kNoAllocParts;                      // offset of the norm partials
constexpr size_t kNoAllocOut = kNoAllocParts + kMaxReduceBlocks;    // offset of the two sums
constexpr size_t kNoAllocDoubles = kNoAllocOut + 2;
__device__ __align__(256) double scratch[kNoAllocDoubles];
constexpr int kMaxDevices = 64;
double *g_scratch_ptr[kMaxDevices];

// device address of `scratch` on the current device (looked up once per device)
int noalloc_scratch(double **out) {
  int dev = 0;
  QH_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) {
    set_error("b_minus_Dx_noalloc: device %d out of range", dev);
    return 1;
  }
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    QH_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch_ptr[dev] = (double *)p;
  }
  *out = g_scratch_ptr[dev];
  return 0;
}
}  // namespace

extern "C" {

int qcd_hip_b_minus_Dx_noalloc(qcd_hip_field x, int rx, qcd_hip_field b, int rb, qcd_hip_field g, double kappa,
                               double mu, qcd_hip_field r, int rr, double *rel) {
  std::lock_guard<std::recursive_mutex> lock(state_mutex());   // the library stream
  if (!ctx()->stream) {
    set_error("b_minus_Dx_noalloc: the library is not initialised (create the fields first)");
    return 1;
  }
  if (!x || !b || !g || !r || x->prec != QCD_HIP_F64 || b->prec != QCD_HIP_F64 || g->prec != QCD_HIP_F64 ||
      r->prec != QCD_HIP_F64 || r->kind != QCD_HIP_SPINOR || !rel || rx < 0 || rx >= x->nrhs || rb < 0 ||
      rb >= b->nrhs || rr < 0 || rr >= r->nrhs) {
    set_error("b_minus_Dx_noalloc: needs FP64 x, b, r and gauge field and valid rhs indices");
    return 1;
  }
  QH_TRY(dslash_check(r, x, g));
  QH_TRY(dslash_check(x, b, g));
  const int grid = dslash_grid(x, g);
  if (grid < 1 || (size_t)grid > kNoAllocParts) {
    set_error("b_minus_Dx_noalloc: %d Dslash workgroups exceed the %zu partial sums of the static scratch", grid,
              kNoAllocParts);
    return 1;
  }
  double *sp = nullptr;
  QH_TRY(noalloc_scratch(&sp));
  hipStream_t st = ctx()->stream;
  int used = 0, nb = 0;
  // r = b - D x with |r|^2 workgroup partials (every workgroup writes its slot)
  QH_TRY(dslash_launch(EPI_RES_D, true, r, rr, x, rx, g, b, rb, 1.0 / (2.0 * kappa) - 4.0, mu, sp, st, &used));
  if (used != grid) {
    set_error("b_minus_Dx_noalloc: launch used %d workgroups, expected %d", used, grid);
    return 1;
  }
  QH_TRY(norm2_launch(b, rb, sp + kNoAllocNorm, &nb, st));
  QH_TRY(finalize(sp, used, 1, sp + kNoAllocOut, st));
  QH_TRY(finalize(sp + kNoAllocNorm, nb, 1, sp + kNoAllocOut + 1, st));
  double h[2] = {0.0, 0.0};
  QH_CHECK(hipMemcpyAsync(h, sp + kNoAllocOut, sizeof(h), hipMemcpyDeviceToHost, st));
  QH_CHECK(hipStreamSynchronize(st));
  *rel = std::sqrt(h[0]) / std::sqrt(h[1]);
  return 0;
}

// One-shot convenience: create a solver, solve every rhs of b, destroy it.
int qcd_hip_invert(qcd_hip_field x, qcd_hip_field b, qcd_hip_field g64, double kappa, double mu,
                   const qcd_hip_solver_params *prm, qcd_hip_solver_stats *stats) {
  qcd_hip_solver S = nullptr;
  qcd_hip_solver_params def;
  if (!prm) {
    qcd_hip_solver_default_params(&def);
    prm = &def;
  }
  if (!b) {
    set_error("invert: null right-hand side");
    return 1;
  }
  QH_TRY(qcd_hip_solver_create(&S, b->lat, prm));
  int rc = qcd_hip_solver_set_gauge(S, g64);
  if (!rc) rc = qcd_hip_solver_solve(S, x, b, kappa, mu, stats);
  qcd_hip_solver_destroy(S);
  return rc;
}

}  // extern "C"
