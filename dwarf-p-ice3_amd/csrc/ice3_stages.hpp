// ice3_stages.hpp -- the stages of the ice_adjust / rain_ice path as per-thread
// device functions:
//   adjust_at     one point of ICE_ADJUST;
//   sedim_column  one column, levels walked top-down: the statistical
//                 sedimentation flux recurrence (fluxes stay in registers) and
//                 the surface precipitation;
//   adjust_sedim_column  ICE_ADJUST and the sedimentation of one column in one walk;
//   micro_at      one point: RAIN_ICE sections 1, 4, 5 and 8 (nucleation
//                 outside the microphysics mask, the ICE4 time splitting, the
//                 total tendencies and the negativity correction).
// The kernels in ice3_kernels.hip launch one thread per column / per point on
// these functions.  Everything here is force-inlined and every array index is a
// compile-time constant after unrolling, so the state lives in registers.
#pragma once
#include "../../include/ice3.h"
#include "ice3_physics.hpp"

namespace ice3 {

// The wavefront's issue priority on its SIMD (0 to 3); nothing in a CPU build of the stages.
template <int N> __device__ __forceinline__ void wave_priority() {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_s_setprio(N);
#endif
}

struct AdjustArgs {
  int ncol, nlev, ld;
  double dt;
  ice3_ice_adjust_in in;
  ice3_ice_adjust_out out;  // t, rv_out, rc_out, ri_out, cph, lv, ls, ris, srcs may be NULL
  double *ris_copy;         // optional second copy of the adjusted ris
  const double *rh;         // hail mixing ratio at t (KRR=7 only)
};

// The OCND2 branch's extra inputs and outputs (include/ice3.h: ice3_ocnd2_in/_out).
struct Ocnd2Args {
  ice3_ocnd2_in in;
  ice3_ocnd2_out out;
  const double *tiwmx;  // ESTABW then ESTABI, ICE3_TIWMX_N entries each
};

// The fields ICE_ADJUST reads at a point.
struct AdjustPoint {
  double sigqsat, pabs, sigs, th, exn, exn_ref, rho_dry_ref, rv, rc, ri, rr, rs, rg, cf_mf, rc_mf, ri_mf, rvs,
      rcs, ris, ths, rh;
};
template <bool HAIL = false>
__device__ __forceinline__ AdjustPoint adjust_load(const AdjustArgs &a, double sigqsat, size_t j) {
  const ice3_ice_adjust_in &in = a.in;
  return AdjustPoint{sigqsat, in.pabs[j], in.sigs[j], in.th[j], in.exn[j], in.exn_ref[j], in.rho_dry_ref[j],
                     in.rv[j], in.rc[j], in.ri[j], in.rr[j], in.rs[j], in.rg[j], in.cf_mf[j], in.rc_mf[j],
                     in.ri_mf[j], in.rvs[j], in.rcs[j], in.ris[j], in.ths[j], HAIL ? a.rh[j] : 0.};
}

// ICE_ADJUST at point j (level k) of column i (micro/ice_adjust.F90:257-472) on the fields p; returns the
// adjusted ris.  With OCND2 the branch's extra fields come from x: the layer thickness is
// ZDZ(k) = PZZ(kp) - PZZ(kp-1), kp = min(k+1, nlev-1) (condensation.F90:366,376-378).
// HAIL (KRR=7): a.rh enters the heat capacity.
// c0 is the offset of the column's lowest level, a.ld the step to the next one.
template <bool OCND2 = false, bool HAIL = false>
__device__ __forceinline__ double adjust_at(const AdjustArgs &a, int i, size_t j, int k,
                                            const Ocnd2Args *x, unsigned *br, size_t c0,
                                            const AdjustPoint &p) {
  double rvs = p.rvs, rcs = p.rcs, ris = p.ris, ths = p.ths;
  AdjustOut o;
  Ocnd2Point xp;
  if constexpr (OCND2) {
    const int kp = k + 1 < a.nlev - 1 ? k + 1 : a.nlev - 1;
    const double *zz = x->in.zz;
    xp.tiwmx = x->tiwmx;
    xp.z = zz[j];
    xp.dz = zz[(size_t)kp * a.ld + c0] - zz[(size_t)(kp - 1) * a.ld + c0];
    xp.cld_wgt = x->in.ice_cld_wgt[i];
    xp.bottom = k == 0;
  }
  ice_adjust_point<OCND2, HAIL>(a.dt, p.sigqsat, p.pabs, p.sigs, p.th, p.exn, p.exn_ref, p.rho_dry_ref, p.rv,
                                p.rc, p.ri, p.rr, p.rs, p.rg, p.cf_mf, p.rc_mf, p.ri_mf, rvs, rcs, ris, ths, o,
                                &xp, p.rh, br);
  if constexpr (OCND2) {
    x->out.icldfr[j] = xp.icldfr;
    x->out.wcldfr[j] = xp.wcldfr;
    x->out.ssio[j] = xp.ssio;
    x->out.ssiu[j] = xp.ssiu;
    x->out.ifr[j] = 10.;  // PIFR(:,:) = 10. (condensation.F90:260)
  }
  const ice3_ice_adjust_out &out = a.out;
  if (out.t) out.t[j] = o.t;
  if (out.rv_out) out.rv_out[j] = o.rv;
  if (out.rc_out) out.rc_out[j] = o.rc;
  if (out.ri_out) out.ri_out[j] = o.ri;
  out.cldfr[j] = o.cldfr;
  out.hlc_hrc[j] = o.hlc_hrc;
  out.hlc_hcf[j] = o.hlc_hcf;
  out.hli_hri[j] = o.hli_hri;
  out.hli_hcf[j] = o.hli_hcf;
  if (out.cph) out.cph[j] = o.cph;
  if (out.lv) out.lv[j] = o.lv;
  if (out.ls) out.ls[j] = o.ls;
  out.rvs[j] = rvs;
  out.rcs[j] = rcs;
  if (out.ris) out.ris[j] = ris;
  out.ths[j] = ths;
  if (out.srcs) out.srcs[j] = o.srcs;
  if (a.ris_copy) a.ris_copy[j] = ris;
  return ris;
}

template <bool OCND2 = false, bool HAIL = false>
__device__ __forceinline__ double adjust_at(const AdjustArgs &a, int i, size_t j, int k,
                                            const Ocnd2Args *x, unsigned *br, size_t c0) {
  return adjust_at<OCND2, HAIL>(a, i, j, k, x, br, c0, adjust_load<HAIL>(a, a.in.sigqsat[i], j));
}

// Fields (nlev, ld): the lowest level of column i at offset i.
template <bool OCND2 = false, bool HAIL = false>
__device__ __forceinline__ double adjust_at(const AdjustArgs &a, int i, size_t j, int k = 0,
                                            const Ocnd2Args *x = nullptr, unsigned *br = nullptr) {
  return adjust_at<OCND2, HAIL>(a, i, j, k, x, br, (size_t)i);
}

// Sedimentation stage arguments.  src_* are the sources entering RAIN_ICE,
// dst_* receive them after sedimentation (dst may alias src).
struct SedimArgs {
  int ncol, nlev, ld;
  double dt;
  const double *rhodref, *dzz;
  const double *src_rr, *src_ri, *src_rs, *src_rg;
  double *dst_rr, *dst_ri, *dst_rs, *dst_rg;
  double *inprc, *inprr, *inpri, *inprs, *inprg;
  double *zzz;  // OCND2 branch: receives the model level height ZZZZ (micro/rain_ice.F90:387-395)
  const double *src_rh;  // hail (KRR=7): source in, source out, surface rate
  double *dst_rh, *inprh;
};

// Columns per compute unit from which the statistical sedimentation walks a column with one thread
// (k_sedim_walk, or k_adjust_sedim with ICE_ADJUST), below which k_sedim takes 64 columns with a
// wavefront per species and half.  Few levels leave k_sedim's pipeline of three levels a step
// unfilled and its prologue unpaid; few columns leave the walk's chain of levels, 2 us each, uncovered.
// The walk steps up whenever another wavefront a SIMD is needed (every 256 columns a compute unit).
// 256 compute units, us of the walk / k_sedim; the form taken changes at each line's middle pair:
//   FP64   2 levels:   8,192 columns 6/7,     16,384 6/7,      65,536 8/15
//          5 levels:  32,768 15/13,           49,152 15/17,    65,536 15/23
//         12 levels:  49,152 31/27,           65,536 32/35,    98,304 46/48
//         20 levels:  65,536 54/52, 98,304 74/72,  110,000 76/82, 262,144 135/175
//         90 levels:  98,304 308/252, 110,000 309/290, 131,072 319/320, 262,144 559/640
//   hail   5 levels:  32,768 19/15,           49,152 19/21,    65,536 19/32
//         20 levels:  49,152 65/50,           65,536 72/79,    98,304 93/112
//         90 levels:  81,920 395/360,         98,304 398/411, 262,144 694/1019
//   mixed  5 levels:  32,768 10/8,            49,152 10/10,    65,536 10/13
//         90 levels:  65,536 140/97,         110,000 167/160
//   fused, k_adjust_sedim / ICE_ADJUST and k_sedim: 2 levels 64 columns 11/14, 16,384 12/14;
//          4 levels:  32,768 26/20,           49,152 27/24,    65,536 28/31;
//          5 levels and more: from 432 columns a compute unit on (launch_adjust_sedim)
// k_sedim never has 2^28 columns, at ten threads a column, in one launch: they are walked.
enum SedimForm { SEDIM_FP64, SEDIM_HAIL, SEDIM_MIXED, SEDIM_FUSED };
inline int sedim_walk_cols(SedimForm form, int nlev) {
  if (form == SEDIM_FUSED) return nlev <= 2 ? 0 : nlev <= 4 ? 72 * (nlev - 1) : 432;
  const int few = 48 * (nlev - 1);
  const int many = form == SEDIM_MIXED  ? 432
                   : form == SEDIM_HAIL ? (nlev < 51 ? 180 + 4 * nlev : 384)
                   : nlev <= 12         ? 216
                                        : (nlev < 76 ? 360 + 2 * nlev : 512);
  return few < many ? few : many;
}

// ICE4_SEDIMENTATION with CSEDIM='SPLI' (micro/mode_ice4_sedimentation.F90:196-219): the
// split sedimentation of rain, pristine ice, snow, graupel (and hail) on the state at t, then
// ICE4_CORRECT_NEGATIVITIES of every source.  FP64 whatever the precision of the call.
struct SplitArgs {
  int ncol, nlev, ld;
  double dt, tscale, maxcfl;
  const double *rhodref, *dzz, *exn;
  const double *t[8];    // state at t (times tscale): th, rv, rc, rr, ri, rs, rg, rh
  const double *src[8];  // sources read
  double *dst[8];        // sources written (may alias src)
  double *inprc, *inprr, *inpri, *inprs, *inprg, *inprh;
  double *zzz;           // OCND2 branch: receives the model level height ZZZZ
  unsigned long long *capped;  // columns whose species hit the sub-step cap
  double *keep[3];       // optional: receive t[0..2] as read (th, rv, rc at t, unscaled)
};

// ICE4_SEDIMENTATION_STAT (micro/mode_ice4_sedimentation_stat.F90:143-229) for column i,
// followed by the surface precipitation of RAIN_ICE (PINPRS += PINPRI, PINPRC = 0 with
// LSEDIC=F).  With ZZZ the walk also writes RAIN_ICE's model level height ZZZZ into a.zzz:
// PDZZ accumulated from the top level down, minus half the level's own (rain_ice.F90:387-395,
// JK = IKTE..IKTB with level 1 the lowest).  HAIL: hail sediments too (species 7,
// micro/mode_ice4_sedimentation_stat.F90:184-188,208-210,220-222).
template <class R, bool ZZZ = false, bool HAIL = false>
__device__ __forceinline__ void sedim_column(const SedimArgs &a, int i) {
  const double dt = a.dt;
  double fr = 0., fi = 0., fs = 0., fg = 0., fh = 0., zzsum = 0.;
  for (int k = a.nlev - 1; k >= 0; --k) {
    const size_t j = (size_t)k * a.ld + i;
    const double rho = a.rhodref[j], dz = a.dzz[j];
    if constexpr (ZZZ) {
      zzsum = zzsum + dz;
      a.zzz[j] = zzsum - dz * 0.5;
    }
    const R lnrho = rlog<R>((R)rho);
    double rrs = a.src_rr[j], ris = a.src_ri[j], rss = a.src_rs[j], rgs = a.src_rg[j];
    sediment_species<R>(IRR, dt, rho, lnrho, dz, rrs, fr);
    sediment_species<R>(IRI, dt, rho, lnrho, dz, ris, fi);
    sediment_species<R>(IRS, dt, rho, lnrho, dz, rss, fs);
    sediment_species<R>(IRG, dt, rho, lnrho, dz, rgs, fg);
    a.dst_rr[j] = rrs; a.dst_ri[j] = ris; a.dst_rs[j] = rss; a.dst_rg[j] = rgs;
    if constexpr (HAIL) {
      double rhs = a.src_rh[j];
      sediment_species<R>(IRH, dt, rho, lnrho, dz, rhs, fh);
      a.dst_rh[j] = rhs;
    }
  }
  a.inprc[i] = 0.;
  a.inprr[i] = fr / by(P.XRHOLW);
  a.inpri[i] = fi / by(P.XRHOLW);
  a.inprs[i] = fs / by(P.XRHOLW) + fi / by(P.XRHOLW);
  a.inprg[i] = fg / by(P.XRHOLW);
  if constexpr (HAIL) a.inprh[i] = fh / by(P.XRHOLW);
}

// ICE_ADJUST and the sedimentation of column i in one top-down walk (the FP64 fused step):
// at each level the point is adjusted, then its precipitating species sediment, ri from the
// adjusted source held in a register.  The sedimentation of a level needs only that level
// and the flux from above, so the results are those of adjust_at over all points followed
// by sedim_column.  HAIL: ICE_ADJUST with the hail heat capacity, and hail sediments.
// A wavefront's priority falls with each quarter of its column, so that those behind catch up: a SIMD
// favours its oldest, and the last ran on alone (262,144 columns 1.47 -> 1.43 ms, 150,000 0.98 ->
// 0.91; hail 1.60 -> 1.54, 1.10 -> 1.01).
// A level's inputs are all named before the first store, which the compiler would not move
// a load across: 1.43 ms at 262,144 columns of 90 levels (6.8 GB, 4.8 TB/s, the VALU 86 % busy),
// 0.03 more with the sedimentation's loads after the adjustment's stores.
template <class R, bool HAIL = false>
__device__ __forceinline__ void adjust_sedim_column(const AdjustArgs &aa, const SedimArgs &a, int i) {
  const double dt = a.dt;
  double fr = 0., fi = 0., fs = 0., fg = 0., fh = 0.;
  const double sigqsat = aa.in.sigqsat[i];
  wave_priority<3>();
  for (int k = a.nlev - 1; k >= 0; --k) {
    const size_t j = (size_t)k * a.ld + i;
    if (k == 3 * a.nlev / 4) wave_priority<2>();
    if (k == a.nlev / 2) wave_priority<1>();
    if (k == a.nlev / 4) wave_priority<0>();
    const AdjustPoint p = adjust_load<HAIL>(aa, sigqsat, j);
    const double rho = a.rhodref[j], dz = a.dzz[j];
    double rrs = a.src_rr[j], rss = a.src_rs[j], rgs = a.src_rg[j], rhs = 0.;
    if constexpr (HAIL) rhs = a.src_rh[j];
    double ris = adjust_at<false, HAIL>(aa, i, j, 0, nullptr, nullptr, (size_t)i, p);
    const R lnrho = rlog<R>((R)rho);
    sediment_species<R>(IRR, dt, rho, lnrho, dz, rrs, fr);
    sediment_species<R>(IRI, dt, rho, lnrho, dz, ris, fi);
    sediment_species<R>(IRS, dt, rho, lnrho, dz, rss, fs);
    sediment_species<R>(IRG, dt, rho, lnrho, dz, rgs, fg);
    a.dst_rr[j] = rrs; a.dst_ri[j] = ris; a.dst_rs[j] = rss; a.dst_rg[j] = rgs;
    if constexpr (HAIL) {
      sediment_species<R>(IRH, dt, rho, lnrho, dz, rhs, fh);
      a.dst_rh[j] = rhs;
    }
  }
  a.inprc[i] = 0.;
  a.inprr[i] = fr / by(P.XRHOLW);
  a.inpri[i] = fi / by(P.XRHOLW);
  a.inprs[i] = fs / by(P.XRHOLW) + fi / by(P.XRHOLW);
  a.inprg[i] = fg / by(P.XRHOLW);
  if constexpr (HAIL) a.inprh[i] = fh / by(P.XRHOLW);
}

// Microphysics stage arguments.  The t-state of species v is t[v][j] * tscale
// (tscale = 1 when the caller hands the t-state over, dt when it is the adjusted
// sources); src[v] are the sources after sedimentation, dst[v] the results (may
// alias src).  Species order: th, rv, rc, rr, ri, rs, rg, and hail (entry 7, read by the
// KRR=7 kernels only).
struct MicroArgs {
  int ncol, nlev, ld;
  double dt, tscale;
  const double *tab;
  const double *exn, *rhodref, *exn_ref, *pabs, *cldfr, *sigs;
  const double *t[8];
  const double *src[8];
  const double *src_ci;
  double *dst[8];
  double *ci, *evap3d, *rainfr;
  int *calls;
  unsigned long long *counters;  // [0] tendency calls, [1] capped points, [2] micro points
  int max_calls;                 // sub-step cap per point
  unsigned long long *capped;    // context counter of capped points (always counted)
  // OCND2 branch only: ICE_ADJUST's OCND2 outputs, the TIWMX tables, and the model level
  // height ZZZZ, which the sedimentation writes into rainfr before the
  // microphysics reads it and writes the rain fraction over it
  const double *icldfr, *ssio, *ssiu, *ifr, *tiwmx;
  unsigned *branches;  // test hook only (ice3_rain_ice_branches): per point, ICE3_BR_* bits
};

// ICE4_CORRECT_NEGATIVITIES (micro/mode_ice4_correct_negativities.F90:51-171) on one
// point's sources: negative condensate goes back to vapour with its latent heat, then
// vapour below XRTMIN(1) is restored from cloud + ice, rain, snow and graupel; with HAIL,
// hail takes part in both steps after graupel (:115-120,165-170).
template <bool HAIL = false>
__device__ __forceinline__ void correct_negativities(double &ths, double &rvs, double &rcs,
                                                     double &rrs, double &ris, double &rss,
                                                     double &rgs, double lvfact, double lsfact,
                                                     double *rhs = nullptr) {
  double zw;
  zw = rcs - dmax(rcs, 0.); rvs = rvs + zw; ths = ths - zw * lvfact; rcs = rcs - zw;
  zw = rrs - dmax(rrs, 0.); rvs = rvs + zw; ths = ths - zw * lvfact; rrs = rrs - zw;
  zw = ris - dmax(ris, 0.); rvs = rvs + zw; ths = ths - zw * lsfact; ris = ris - zw;
  zw = rss - dmax(rss, 0.); rvs = rvs + zw; ths = ths - zw * lsfact; rss = rss - zw;
  zw = rgs - dmax(rgs, 0.); rvs = rvs + zw; ths = ths - zw * lsfact; rgs = rgs - zw;
  if constexpr (HAIL) {
    zw = *rhs - dmax(*rhs, 0.); rvs = rvs + zw; ths = ths - zw * lsfact; *rhs = *rhs - zw;
  }
  zw = dmin(1., dmax(P.XRTMIN[1] - rvs, 0.) / by(dmax(rcs + ris, 1.E-20)));
  ths = ths - zw * (rcs * lvfact + ris * lsfact);
  rvs = rvs + zw * (rcs + ris);
  rcs = (1. - zw) * rcs;
  ris = (1. - zw) * ris;
  zw = dmin(dmax(rrs, 0.), dmax(P.XRTMIN[1] - rvs, 0.));
  rvs = rvs + zw; rrs = rrs - zw; ths = ths - zw * lvfact;
  zw = dmin(dmax(rss, 0.), dmax(P.XRTMIN[1] - rvs, 0.));
  rvs = rvs + zw; rss = rss - zw; ths = ths - zw * lsfact;
  zw = dmin(dmax(rgs, 0.), dmax(P.XRTMIN[1] - rvs, 0.));
  rvs = rvs + zw; rgs = rgs - zw; ths = ths - zw * lsfact;
  if constexpr (HAIL) {
    zw = dmin(dmax(*rhs, 0.), dmax(P.XRTMIN[1] - rvs, 0.));
    rvs = rvs + zw; *rhs = *rhs - zw; ths = ths - zw * lsfact;
  }
}

// t-state (times tscale) and sources of the first NV variables at point j (7, or 8 with hail).
template <int NV = 7>
__device__ __forceinline__ void micro_load(const MicroArgs &a, size_t j, double *t, double *s) {
  const double ts = a.tscale;
#pragma unroll
  for (int v = 0; v < NV; ++v) t[v] = a.t[v][j] * ts;
#pragma unroll
  for (int v = 0; v < NV; ++v) s[v] = a.src[v][j];
}

// RAIN_ICE's latent heat factors L / cph (micro/rain_ice.F90:334-347) from the t-state t;
// with HAIL the ice mixing ratio includes hail (:337-338).
template <bool HAIL = false>
__device__ __forceinline__ void rain_ice_factors(const double *t, double exn, double &lsfact,
                                                 double &lvfact) {
  double zrice = t[IRI] + t[IRS] + t[IRG];
  if constexpr (HAIL) zrice = zrice + t[IRH];
  const double zdevide = P.XCPD + P.XCPV * t[IRV] + P.XCL * (t[IRC] + t[IRR]) + P.XCI * zrice;
  const double zt = t[ITH] * exn;
  lsfact = (P.XLSTT + (P.XCPV - P.XCI) * (zt - P.XTT)) / by(zdevide);
  lvfact = (P.XLVTT + (P.XCPV - P.XCL) * (zt - P.XTT)) / by(zdevide);
}

// RAIN_ICE's microphysics mask (micro/rain_ice.F90:365-381): a hydrometeor above XRTMIN;
// with OCND2 (:348-364), ice supersaturation in the ice cloud above XFRMIN(12) or a
// hydrometeor above XFRMIN(13).  HAIL: hail above XRTMIN(7) too (:366-372).
template <bool OCND2 = false, bool HAIL = false>
__device__ __forceinline__ bool micro_mask(const double *t, const MicroArgs &a, size_t j) {
  if constexpr (OCND2)
    return a.ssio[j] > P.XFRMIN[12] || t[IRC] > P.XFRMIN[13] || t[IRR] > P.XFRMIN[13] ||
           t[IRI] > P.XFRMIN[13] || t[IRS] > P.XFRMIN[13] || t[IRG] > P.XFRMIN[13];
  if constexpr (HAIL)
    return t[IRC] > P.XRTMIN[2] || t[IRR] > P.XRTMIN[3] || t[IRI] > P.XRTMIN[4] ||
           t[IRS] > P.XRTMIN[5] || t[IRG] > P.XRTMIN[6] || t[IRH] > P.XRTMIN[7];
  return t[IRC] > P.XRTMIN[2] || t[IRR] > P.XRTMIN[3] || t[IRI] > P.XRTMIN[4] ||
         t[IRS] > P.XRTMIN[5] || t[IRG] > P.XRTMIN[6];
}

// The OCND2 inputs of point j (the model level height is staged in rainfr).
__device__ __forceinline__ MicroOcnd2 ocnd2_point(const MicroArgs &a, size_t j) {
  return MicroOcnd2{a.tiwmx, a.icldfr[j], a.ssio[j], a.ssiu[j], a.ifr[j], a.rainfr[j]};
}

// Nucleation outside the microphysics mask (micro/rain_ice.F90:505-540) at point j with
// t-state t: cit is reset and updated, rvheni receives the nucleated vapour.
template <class R, bool OCND2 = false, bool HAIL = false>
__device__ __forceinline__ void micro_nucleation(const MicroArgs &a, size_t j, const double *t,
                                                 double &cit, double &rvheni) {
  const double exn = a.exn[j];
  double lsfact, lvfact;
  rain_ice_factors<HAIL>(t, exn, lsfact, lvfact);
  cit = 0.;
  MicroOcnd2 x;
  if constexpr (OCND2) x = ocnd2_point(a, j);
  nucleation<R, OCND2>(true, t[ITH], a.pabs[j], a.rhodref[j], P.XTT / by(exn), lsfact / by(exn), t[ITH] * exn,
                       t[IRV], cit, rvheni, &x);
}

// RAIN_ICE section 8 at point j (micro/rain_ice.F90:612-652 and the reinstated 754-823):
// total tendencies from the end state wr of the time splitting, ICE4_CORRECT_NEGATIVITIES,
// and the stores.  The t-state and sources are read again from memory (they are not
// written before this point's stores).  rvheni: vapour nucleated outside the mask.  HAIL:
// wr has hail last, and the hail source takes its tendency and negativity correction.
template <bool HAIL = false>
__device__ __forceinline__ void micro_finish(const MicroArgs &a, size_t j, const double *t,
                                             const double *s, double exn, const double *wr,
                                             double cit, double evap3d, double rvheni, int calls,
                                             double exnref) {
  constexpr int NV = HAIL ? 8 : 7;
  const double dt = a.dt, zinv = 1. / by(dt);
  double lsfact, lvfact;
  rain_ice_factors<HAIL>(t, exn, lsfact, lvfact);
  rvheni = dmin(s[IRV], rvheni / by(dt));
  // 8.1 total tendencies
  lsfact = lsfact / by(exnref);
  lvfact = lvfact / by(exnref);
  const double wrv = (wr[IRV] - t[IRV]) * zinv, wrc = (wr[IRC] - t[IRC]) * zinv;
  const double wrr = (wr[IRR] - t[IRR]) * zinv, wri = (wr[IRI] - t[IRI]) * zinv;
  const double wrs = (wr[IRS] - t[IRS]) * zinv, wrg = (wr[IRG] - t[IRG]) * zinv;
  const double wrh = HAIL ? (wr[NV - 1] - t[NV - 1]) * zinv : 0.;
  const double wth = (wrc + wrr) * lvfact + (wri + wrs + wrg + wrh) * lsfact;
  double ths = s[ITH] + wth + rvheni * lsfact;
  double rvs = s[IRV] + wrv - rvheni;
  double rcs = s[IRC] + wrc;
  double rrs = s[IRR] + wrr;
  double ris = s[IRI] + wri + rvheni;
  double rss = s[IRS] + wrs;
  double rgs = s[IRG] + wrg;
  double rhs = HAIL ? s[NV - 1] + wrh : 0.;
  // 8.2 ICE4_CORRECT_NEGATIVITIES
  correct_negativities<HAIL>(ths, rvs, rcs, rrs, ris, rss, rgs, lvfact, lsfact, &rhs);
  a.dst[ITH][j] = ths; a.dst[IRV][j] = rvs; a.dst[IRC][j] = rcs; a.dst[IRR][j] = rrs;
  a.dst[IRI][j] = ris; a.dst[IRS][j] = rss; a.dst[IRG][j] = rgs;
  if constexpr (HAIL) a.dst[NV - 1][j] = rhs;
  a.ci[j] = cit;
  a.evap3d[j] = evap3d;
  a.rainfr[j] = 1.;
  if (a.calls) a.calls[j] = calls;
}

// RAIN_ICE sections 1, 4, 5, 8 (micro/rain_ice.F90:334-384, 505-540, 612-652 and the
// reinstated 754-823) for point j, all in one thread.  Returns the number of tendency
// calls, negative if the sub-step cap was hit.  HAIL: KRR=7, hail the eighth variable.
template <class R, bool OCND2 = false, bool HAIL = false, class TB>
__device__ __forceinline__ int micro_at(const MicroArgs &a, size_t j, const TB *__restrict__ tab,
                                        unsigned *br = nullptr) {
  constexpr int NV = HAIL ? 8 : 7;
  double wr[NV], s[NV];
  micro_load<NV>(a, j, wr, s);
  double cit = a.src_ci[j], rvheni = 0., evap3d = 0.;
  int calls = 0;
  if (micro_mask<OCND2, HAIL>(wr, a, j)) {
    MicroOcnd2 x;
    if constexpr (OCND2) x = ocnd2_point(a, j);
    calls = stepping_point<R, OCND2, HAIL>(a.dt, a.exn[j], a.rhodref[j], a.pabs[j], a.cldfr[j],
                                           a.sigs[j], cit, wr, s, evap3d, a.max_calls, tab, &x,
                                           HAIL ? a.tab + ICE3_T_ICE3 : nullptr, br);
  } else {
    micro_nucleation<R, OCND2, HAIL>(a, j, wr, cit, rvheni);
  }
  double t[NV];
  micro_load<NV>(a, j, t, s);
  micro_finish<HAIL>(a, j, t, s, a.exn[j], wr, cit, evap3d, rvheni, calls, a.exn_ref[j]);
  return calls;
}

// Input features of the surrogate at point j (the microphysics inputs of micro_at):
// T, ln p, rhodref, ln(r + 1e-9) of the six water species of the t-state, ln(1 + ci),
// sigma_s, exner, dt, cloud fraction, and asinh(1e6 * dt * e) of the external tendency
// e = source - t-state/dt of rr, ri, rs, rg (the sedimentation, which the time
// splitting integrates beside the processes).  Returns false where RAIN_ICE would not
// run the ICE4 microphysics (no hydrometeor above XRTMIN), as micro_at decides it.
__device__ __forceinline__ bool surrogate_features(const MicroArgs &a, size_t j, float *f) {
  const double ts = a.tscale, exn = a.exn[j];
  double r[7];
#pragma unroll
  for (int v = 0; v < 7; ++v) r[v] = a.t[v][j] * ts;
  f[0] = (float)(r[ITH] * exn);
  f[1] = logf((float)a.pabs[j]);
  f[2] = (float)a.rhodref[j];
#pragma unroll
  for (int v = 1; v < 7; ++v) f[2 + v] = logf((float)fmax(r[v], 0.) + 1e-9f);
  f[9] = logf(1.f + (float)fmax(a.src_ci[j], 0.));
  f[10] = (float)a.sigs[j];
  f[11] = (float)exn;
  f[12] = (float)a.dt;
  f[13] = (float)a.cldfr[j];
#pragma unroll
  for (int v = IRR; v <= IRG; ++v)
    f[14 + v - IRR] = asinhf((float)(1e6 * (a.src[v][j] * a.dt - r[v])));
  return r[IRC] > P.XRTMIN[2] || r[IRR] > P.XRTMIN[3] || r[IRI] > P.XRTMIN[4] ||
         r[IRS] > P.XRTMIN[5] || r[IRG] > P.XRTMIN[6];
}

// Latent heat factors L/(cph * exnref) of the total tendencies at point j (t-state), as
// micro_at computes them (micro/rain_ice.F90:334-347 divided by PEXNREF).
__device__ __forceinline__ void latent_factors(const MicroArgs &a, size_t j, double &lvfact,
                                               double &lsfact) {
  double t[7], s[7];
  micro_load(a, j, t, s);
  rain_ice_factors(t, a.exn[j], lsfact, lvfact);
  lsfact = lsfact / by(a.exn_ref[j]);
  lvfact = lvfact / by(a.exn_ref[j]);
}

// ---------------------------------------------------------------- argument set-up
// Host-side wiring of the C-ABI structs into the stage arguments, shared by the
// kernel launchers and by CPU builds of the stages.

// rain_ice: sedimentation updates the precipitating sources in place, then the
// microphysics reads the handed-over t-state and updates all sources in place.
// The split sedimentation's arguments for the stages whose sedimentation is described by sa
// and whose microphysics (the state at t, th/rv/rc sources) by m.
inline SplitArgs split_args(const SedimArgs &sa, const MicroArgs &m, double maxcfl,
                            unsigned long long *capped) {
  SplitArgs a = SplitArgs{};
  a.ncol = sa.ncol; a.nlev = sa.nlev; a.ld = sa.ld; a.dt = sa.dt; a.tscale = m.tscale;
  a.maxcfl = maxcfl;
  a.rhodref = sa.rhodref; a.dzz = sa.dzz; a.exn = m.exn;
  for (int q = 0; q < 8; ++q) a.t[q] = m.t[q];
  for (int q = 0; q < 3; ++q) { a.src[q] = m.src[q]; a.dst[q] = m.dst[q]; }
  a.src[3] = sa.src_rr; a.src[4] = sa.src_ri; a.src[5] = sa.src_rs; a.src[6] = sa.src_rg;
  a.src[7] = sa.src_rh;
  a.dst[3] = sa.dst_rr; a.dst[4] = sa.dst_ri; a.dst[5] = sa.dst_rs; a.dst[6] = sa.dst_rg;
  a.dst[7] = sa.dst_rh;
  a.inprc = sa.inprc; a.inprr = sa.inprr; a.inpri = sa.inpri; a.inprs = sa.inprs;
  a.inprg = sa.inprg; a.inprh = sa.inprh;
  a.zzz = sa.zzz;
  a.capped = capped;
  return a;
}

inline void rain_ice_args(int ncol, int nlev, int ld, double dt, const double *tab,
                          const ice3_rain_ice_in *in, const ice3_rain_ice_inout *io,
                          const ice3_rain_ice_out *out, const ice3_stats *stats,
                          SedimArgs &sa, MicroArgs &m) {
  sa = SedimArgs{};
  sa.ncol = ncol; sa.nlev = nlev; sa.ld = ld; sa.dt = dt;
  sa.rhodref = in->rhodref; sa.dzz = in->dzz;
  sa.src_rr = sa.dst_rr = io->rrs; sa.src_ri = sa.dst_ri = io->ris;
  sa.src_rs = sa.dst_rs = io->rss; sa.src_rg = sa.dst_rg = io->rgs;
  sa.inprc = out->inprc; sa.inprr = out->inprr; sa.inpri = out->inpri; sa.inprs = out->inprs;
  sa.inprg = out->inprg;
  m = MicroArgs{};
  m.ncol = ncol; m.nlev = nlev; m.ld = ld; m.dt = dt; m.tscale = 1.; m.tab = tab;
  m.max_calls = DEFAULT_MAX_CALLS;
  m.exn = in->exn; m.rhodref = in->rhodref; m.exn_ref = in->exn_ref; m.pabs = in->pabs;
  m.cldfr = in->cldfr; m.sigs = in->sigs;
  const double *t[7] = {in->tht, in->rvt, in->rct, in->rrt, in->rit, in->rst, in->rgt};
  double *v[7] = {io->ths, io->rvs, io->rcs, io->rrs, io->ris, io->rss, io->rgs};
  for (int q = 0; q < 7; ++q) { m.t[q] = t[q]; m.src[q] = v[q]; m.dst[q] = v[q]; }
  m.src_ci = m.ci = io->ci;
  m.evap3d = out->evap3d; m.rainfr = out->rainfr;
  if (stats) { m.calls = stats->calls; m.counters = stats->counters; }
}

// The fused time step.
// 1. ICE_ADJUST writes the adjusted th, rv, rc, ri sources into the outputs and
//    stages a copy of the adjusted ris in out->evap3d (the microphysics reads it
//    there as the ri t-state, then overwrites it with the evaporation).
// 2. Sedimentation of rr, rs, rg (input sources) and ri (adjusted) into the outputs.
// 3. Microphysics with the t-state = adjusted sources x dt.
inline void pipeline_args(int ncol, int nlev, int ld, double dt, const double *tab,
                          const ice3_pipeline_in *in, const ice3_pipeline_out *out,
                          const ice3_stats *stats, AdjustArgs &aa, SedimArgs &sa, MicroArgs &m) {
  aa = AdjustArgs{};
  aa.ncol = ncol; aa.nlev = nlev; aa.ld = ld; aa.dt = dt;
  aa.in.pabs = in->pabs; aa.in.sigs = in->sigs; aa.in.th = in->th; aa.in.exn = in->exn;
  aa.in.exn_ref = in->exn_ref; aa.in.rho_dry_ref = in->rhodref; aa.in.rv = in->rv;
  aa.in.rc = in->rc; aa.in.ri = in->ri; aa.in.rr = in->rr; aa.in.rs = in->rs; aa.in.rg = in->rg;
  aa.in.cf_mf = in->cf_mf; aa.in.rc_mf = in->rc_mf; aa.in.ri_mf = in->ri_mf;
  aa.in.rvs = in->rvs; aa.in.rcs = in->rcs; aa.in.ris = in->ris; aa.in.ths = in->ths;
  aa.in.sigqsat = in->sigqsat;
  aa.out.cldfr = out->cldfr; aa.out.hlc_hrc = out->hlc_hrc; aa.out.hlc_hcf = out->hlc_hcf;
  aa.out.hli_hri = out->hli_hri; aa.out.hli_hcf = out->hli_hcf;
  aa.out.rvs = out->rvs; aa.out.rcs = out->rcs; aa.out.ris = out->ris; aa.out.ths = out->ths;
  aa.ris_copy = out->evap3d;
  sa = SedimArgs{};
  sa.ncol = ncol; sa.nlev = nlev; sa.ld = ld; sa.dt = dt;
  sa.rhodref = in->rhodref; sa.dzz = in->dzz;
  sa.src_rr = in->rrs; sa.src_ri = out->ris; sa.src_rs = in->rss; sa.src_rg = in->rgs;
  sa.dst_rr = out->rrs; sa.dst_ri = out->ris; sa.dst_rs = out->rss; sa.dst_rg = out->rgs;
  sa.inprc = out->inprc; sa.inprr = out->inprr; sa.inpri = out->inpri; sa.inprs = out->inprs;
  sa.inprg = out->inprg;
  m = MicroArgs{};
  m.ncol = ncol; m.nlev = nlev; m.ld = ld; m.dt = dt; m.tscale = dt; m.tab = tab;
  m.max_calls = DEFAULT_MAX_CALLS;
  m.exn = in->exn; m.rhodref = in->rhodref; m.exn_ref = in->exn_ref; m.pabs = in->pabs;
  m.cldfr = out->cldfr; m.sigs = in->sigs;
  const double *t[7] = {out->ths, out->rvs, out->rcs, in->rrs, out->evap3d, in->rss, in->rgs};
  double *v[7] = {out->ths, out->rvs, out->rcs, out->rrs, out->ris, out->rss, out->rgs};
  for (int q = 0; q < 7; ++q) { m.t[q] = t[q]; m.src[q] = v[q]; m.dst[q] = v[q]; }
  m.src_ci = in->ci; m.ci = out->ci;
  m.evap3d = out->evap3d; m.rainfr = out->rainfr;
  if (stats) { m.calls = stats->calls; m.counters = stats->counters; }
}

// For a call that runs the sedimentation after ICE_ADJUST: ICE_ADJUST's ris goes to the copy that
// is the microphysics' state at t only, and the sedimentation, which writes every level of
// out->ris, reads it there (8 of the 232 bytes a point that ICE_ADJUST moves; at 262,144 columns
// of 90 levels k_ice_adjust 1.01 -> 0.98 ms, k_adjust_sedim 1.49 -> 1.45).
inline void hand_ris_over(AdjustArgs &aa, SedimArgs &sa) {
  aa.out.ris = nullptr;
  sa.src_ri = aa.ris_copy;
}

}  // namespace ice3
