// split.hip -- the full and even-odd hopping kernels for launches of few sites:
// one wavefront per hop.
//
// A workgroup of 8 wavefronts owns 64 sites of one batch row.  Wavefront i
// forms hop i of every site (the colour-multiplied, phased half spinor) and
// leaves it in LDS; after one barrier the half spinors are added up in the order
// of the one-site kernels, so the results have the same bits.  The marching
// and one-site kernels walk a site's eight hops one after another in one lane,
// about 1 us each when nothing else runs on the SIMD: on 8^3x16 they put 32
// workgroups of 256 lanes on 256 CUs.  Here a site's loads are all in flight at
// once and every hop is its own wavefront.
#include "eo_common.h"

namespace qcdhip {

constexpr int kSplitBlock = 512;

// Hop i in summation order: D starts with the z hops, backward first (as
// k_dslash_zm); the even-odd hops go t, x, y, z, forward first (as k_eo_hop).
template <bool EO, int I>
struct SplitHop {
  static constexpr int mu = EO ? I / 2 : I < 2 ? 3 : (I - 2) / 2;
  static constexpr int s = EO ? (I % 2 ? +1 : -1) : I == 0 ? +1 : I == 1 ? -1 : (I % 2 ? +1 : -1);
};

template <typename R>
struct SplitLds {
  Cx<R> h[8][6][64];   // [hop][2 spins x 3 colours][site]
};

template <bool EO, int I, int PS, int PG, typename R>
__device__ __forceinline__ void split_hop(SplitLds<R> &l, const DslashArgs &a, const Site &st, const SpinorIn<PS> &in,
                                          const GaugeIn<PG> &U) {
  constexpr int MU = SplitHop<EO, I>::mu, S = SplitHop<EO, I>::s;
  const unsigned n = S < 0 ? neighbour<MU, +1>(st, a) : neighbour<MU, -1>(st, a);
  const Cx<R> ph{(R)a.ph_re[MU], S < 0 ? (R)a.ph_im[MU] : -(R)a.ph_im[MU]};
  Cx<R> g0[3], g1[3];
  hop_half_at<MU, S, (S > 0)>(g0, g1, in, EO ? n >> 1 : n, U, S < 0 ? st.s : n, ph);
  const unsigned lane = threadIdx.x & 63u;
#pragma unroll
  for (int c = 0; c < 3; c++) {
    l.h[I][c][lane] = g0[c];
    l.h[I][3 + c][lane] = g1[c];
  }
}

template <bool EO, int PS, int PG, typename R>
__device__ __forceinline__ void split_hops(SplitLds<R> &l, unsigned wave, const DslashArgs &a, const Site &st,
                                           const SpinorIn<PS> &in, const GaugeIn<PG> &U) {
  switch (wave) {
    case 0: split_hop<EO, 0>(l, a, st, in, U); break;
    case 1: split_hop<EO, 1>(l, a, st, in, U); break;
    case 2: split_hop<EO, 2>(l, a, st, in, U); break;
    case 3: split_hop<EO, 3>(l, a, st, in, U); break;
    case 4: split_hop<EO, 4>(l, a, st, in, U); break;
    case 5: split_hop<EO, 5>(l, a, st, in, U); break;
    case 6: split_hop<EO, 6>(l, a, st, in, U); break;
    default: split_hop<EO, 7>(l, a, st, in, U); break;
  }
}

// the four spins of colour c: acc += hop I (rebuild_add of one colour)
template <bool EO, int I, typename R>
__device__ __forceinline__ void split_add(Cx<R> acc[4], const SplitLds<R> &l, int c) {
  using PJ = Proj<SplitHop<EO, I>::mu>;
  constexpr int sp = SplitHop<EO, I>::s > 0 ? 0 : 2;
  const unsigned lane = threadIdx.x & 63u;
  const Cx<R> g0 = l.h[I][c][lane], g1 = l.h[I][3 + c][lane];
  acc[0] = cadd(acc[0], g0);
  acc[1] = cadd(acc[1], g1);
  acc[2] = cadd(acc[2], ipow<PJ::C + sp>(PJ::R == 0 ? g0 : g1));
  acc[3] = cadd(acc[3], ipow<PJ::D + sp>(PJ::W == 0 ? g0 : g1));
}
template <bool EO, typename R>
__device__ __forceinline__ void split_sum(Cx<R> acc[4], const SplitLds<R> &l, int c) {
  split_add<EO, 0>(acc, l, c);
  split_add<EO, 1>(acc, l, c);
  split_add<EO, 2>(acc, l, c);
  split_add<EO, 3>(acc, l, c);
  split_add<EO, 4>(acc, l, c);
  split_add<EO, 5>(acc, l, c);
  split_add<EO, 6>(acc, l, c);
  split_add<EO, 7>(acc, l, c);
}

// D or Q (epilogues without reduction) of 64 sites per workgroup; batch rows in
// groups of 4, the row fastest within a group (block_row).  FP64 sums colour c in wavefront c; the grouped
// FP32 and FP16 layouts (and the FP16 site norm) take whole sites, in wavefront
// 0.
template <int PS, int PG, int EPI>
__global__ void __launch_bounds__(kSplitBlock) k_dslash_split(DslashArgs a, SpinorIn<PS> in_all, GaugeIn<PG> U,
                                                              SpinorOut<PS> out_all) {
  using R = typename Prec<PS>::R;
  __shared__ SplitLds<R> l;
  const BlockRow br = block_row(a);
  const RhsView<PS> v = rhs_view(a, in_all, out_all, in_all, br.row);
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned s = br.blk * 64u + (threadIdx.x & 63u);
  const bool ok = s < a.V;
  const Site st = site_coords(ok ? s : 0, a);
  constexpr bool kColour = PS == QCD_HIP_F64;
  typename Prec<PS>::T r[12];
  float n = 0.f;
  if (ok) {
    if constexpr (kColour) {
      if (wave < 3)
#pragma unroll
        for (int q = 0; q < 4; q++) r[q] = v.in.p[0][(size_t)(s / kTile) * 12 * kTile + (3 * q + wave) * kTile + s % kTile];
    } else {
      if (wave == 0) v.in.load_raw(s, r, n);
    }
    split_hops<false>(l, wave, a, st, v.in, U);
  }
  __syncthreads();
  if (!ok || wave >= (kColour ? 3u : 1u)) return;
  const R mp4 = R(a.mp4), tm = R(a.tm);
  auto colour = [&](Cx<R> o[4], const Cx<R> psi[4], int c) {
#pragma unroll
    for (int q = 0; q < 4; q++) o[q] = diag_term(psi[q], mp4, q < 2 ? tm : -tm);
    split_sum<false>(o, l, c);
#pragma unroll
    for (int q = 0; q < 4; q++) {
      o[q] = Cx<R>{R(-0.5) * o[q].re, R(-0.5) * o[q].im};
      if constexpr (EPI == EPI_Q) o[q] = q < 2 ? ipow<1>(o[q]) : ipow<3>(o[q]);
    }
  };
  if constexpr (kColour) {
    Cx<R> psi[4], o[4];
#pragma unroll
    for (int q = 0; q < 4; q++) psi[q] = to_cx<R>(r[q]);
    colour(o, psi, (int)wave);
#pragma unroll
    for (int q = 0; q < 4; q++)
      v.out.p[0][(size_t)(s / kTile) * 12 * kTile + (3 * q + wave) * kTile + s % kTile] =
          from_cx<typename Prec<PS>::T>(o[q]);
  } else {
    Cx<R> psi[12], o[12];
    SpinorIn<PS>::convert(r, n, psi);
#pragma unroll
    for (int c = 0; c < 3; c++) {
      Cx<R> p[4] = {psi[c], psi[3 + c], psi[6 + c], psi[9 + c]}, x[4];
      colour(x, p, c);
#pragma unroll
      for (int q = 0; q < 4; q++) o[3 * q + c] = x[q];
    }
    v.out.store(s, o);
  }
}

// the even-odd hop with epilogue EPI, as k_eo_hop without reduction
template <int PS, int PG, int EPI>
__global__ void __launch_bounds__(kSplitBlock) k_eo_split_hop(EoArgs e, SpinorIn<PS> in_all, GaugeIn<PG> U,
                                                              SpinorOut<PS> out_all, SpinorIn<PS> b_all) {
  using R = typename Prec<PS>::R;
  __shared__ SplitLds<R> l;
  const DslashArgs &a = e.d;
  const BlockRow br = block_row(a);
  const RhsView<PS> v = rhs_view(a, in_all, out_all, b_all, br.row);
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned h = br.blk * 64u + (threadIdx.x & 63u);
  const bool ok = h < e.Vh;
  if (ok) split_hops<true>(l, wave, a, eo_site(h, e.par, a), v.in, U);
  __syncthreads();
  if (!ok || wave > 0) return;
  Cx<R> acc[4][3];
#pragma unroll
  for (int c = 0; c < 3; c++) {
    Cx<R> x[4];
#pragma unroll
    for (int q = 0; q < 4; q++) x[q] = Cx<R>{R(0), R(0)};
    split_sum<true>(x, l, c);
#pragma unroll
    for (int q = 0; q < 4; q++) acc[q][c] = x[q];
  }
  Cx<R> o[12];
  eo_epilogue<EPI>(o, acc, e, v.b, h);
  v.out.store(h, o);
}

template <int PS, int PG>
static int dslash_split_pp(int epi, const DslashArgs &a, dim3 gr, qcd_hip_field out, int ro, qcd_hip_field in, int ri,
                           qcd_hip_field g, hipStream_t st) {
  const SpinorIn<PS> si = SpinorIn<PS>::of(in, ri);
  const SpinorOut<PS> so = SpinorOut<PS>::of(out, ro);
  const GaugeIn<PG> gu = GaugeIn<PG>::of(g);
  if (epi == EPI_D) k_dslash_split<PS, PG, EPI_D><<<gr, kSplitBlock, 0, st>>>(a, si, gu, so);
  else k_dslash_split<PS, PG, EPI_Q><<<gr, kSplitBlock, 0, st>>>(a, si, gu, so);
  QH_CHECK(hipGetLastError());
  return 0;
}

int dslash_split_launch(int epi, DslashArgs a, qcd_hip_field out, int ro, qcd_hip_field in, int ri,
                        qcd_hip_field g, hipStream_t st) {
  a.nblk = (a.V + 63) / 64;
  a.rgroup = 4;
  const dim3 gr(a.nblk * a.count);
  const int ps = in->prec, pg = g->prec;
  if (epi == EPI_D || epi == EPI_Q) {
    if (ps == QCD_HIP_F64 && pg == QCD_HIP_F64)
      return dslash_split_pp<QCD_HIP_F64, QCD_HIP_F64>(epi, a, gr, out, ro, in, ri, g, st);
    if (ps == QCD_HIP_F32 && pg == QCD_HIP_F32)
      return dslash_split_pp<QCD_HIP_F32, QCD_HIP_F32>(epi, a, gr, out, ro, in, ri, g, st);
    if (ps == QCD_HIP_F16 && pg == QCD_HIP_F16)
      return dslash_split_pp<QCD_HIP_F16, QCD_HIP_F16>(epi, a, gr, out, ro, in, ri, g, st);
  }
  set_error("dslash: the split kernel takes D and Q of equal precisions (epilogue %d, spinor %d, gauge %d)", epi, ps, pg);
  return 1;
}

template <int PS>
static int eo_split_pp(int epi, EoArgs e, qcd_hip_field out, int ro, qcd_hip_field in, int ri, qcd_hip_field g,
                       qcd_hip_field b, int rb, hipStream_t st) {
  const SpinorIn<PS> si = SpinorIn<PS>::of(in, ri), sb = b ? SpinorIn<PS>::of(b, rb) : si;
  const SpinorOut<PS> so = SpinorOut<PS>::of(out, ro);
  const GaugeIn<PS> gu = GaugeIn<PS>::of(g);
  e.d.nblk = (e.Vh + 63) / 64;
  e.d.rgroup = 4;
  const dim3 gr(e.d.nblk * e.d.count);
  switch (epi) {
    case EO_MINV: k_eo_split_hop<PS, PS, EO_MINV><<<gr, kSplitBlock, 0, st>>>(e, si, gu, so, sb); break;
    case EO_SCHUR: k_eo_split_hop<PS, PS, EO_SCHUR><<<gr, kSplitBlock, 0, st>>>(e, si, gu, so, sb); break;
    case EO_SUB: k_eo_split_hop<PS, PS, EO_SUB><<<gr, kSplitBlock, 0, st>>>(e, si, gu, so, sb); break;
    case EO_SUB_MINV: k_eo_split_hop<PS, PS, EO_SUB_MINV><<<gr, kSplitBlock, 0, st>>>(e, si, gu, so, sb); break;
    default: set_error("eo: unsupported epilogue %d", epi); return 1;
  }
  QH_CHECK(hipGetLastError());
  return 0;
}

int eo_split_launch(int epi, const EoArgs &e, qcd_hip_field out, int ro, qcd_hip_field in, int ri, qcd_hip_field g,
                    qcd_hip_field b, int rb, hipStream_t st) {
  if (in->prec == QCD_HIP_F64) return eo_split_pp<QCD_HIP_F64>(epi, e, out, ro, in, ri, g, b, rb, st);
  if (in->prec == QCD_HIP_F32) return eo_split_pp<QCD_HIP_F32>(epi, e, out, ro, in, ri, g, b, rb, st);
  return eo_split_pp<QCD_HIP_F16>(epi, e, out, ro, in, ri, g, b, rb, st);
}

}  // namespace qcdhip
