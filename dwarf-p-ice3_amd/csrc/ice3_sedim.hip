// ice3_sedim.hip -- the statistical sedimentation as a kernel of its own (the fused FP64 step
// over many columns runs it in k_adjust_sedim's column walk instead).
#include <hip/hip_runtime.h>

#define ICE3_SCALAR_COEF  // bound by the VALU issue rate
#include "ice3_sedim.hpp"

namespace ice3 {

// ---- k_sedim: ICE4_SEDIMENTATION_STAT, a wavefront per 64 columns, species and half.
//
// The flux recurrence of a species runs down its column (a logarithm, an exponential and a
// division a level, each waiting for the level above), but the species are independent and so
// is the flux that a level's own content sends down.  A workgroup takes 64 columns and NS
// species (rain, ice, snow, graupel, hail): wavefront w < NS evaluates the own-content fluxes
// of species w, wavefront NS + w runs its recurrence, and they hand values over in LDS, SG
// levels (a group) a step:
//   step t: wavefront w < SG takes level w of group t + 1: its density, thickness, the
//           logarithm and powers of the density that every species needs;
//           wavefronts w < NS: own-content fluxes of group t;
//           wavefronts NS + w: the recurrence over group t - 1, and its stores;
// with one barrier a step, the level values in three buffers and the fluxes in two.  Every
// load is issued a step before its use.
//
// Few columns: bound by the recurrence (pristine ice's two logarithms and exponential, about
// 0.7 us a level).  1,024 columns of 90 levels take 59 us (one thread per column, four species
// after one another: 186 us; four wavefronts without the own-content half split off: 104 us).
// More columns: bound by the VALU (76 % busy).  65,536 columns: 179 us (223); from the counts of
// sedim_walk_cols on one thread per column is the better form.  Groups of three levels keep four workgroups' LDS on a compute unit; four levels took
// 206 us at 65,536 columns.  The Horner coefficients as scalars, hoisted out of the loop by
// machine LICM, are worth 9 us at 1,024 columns and 20 us at 65,536 against vector ones.
constexpr int SG = 3;  // levels of a group

template <class R, bool ZZZ = false, bool HAIL = false>
__global__ void __launch_bounds__(128 * (HAIL ? 5 : 4)) k_sedim(SedimArgs a) {
  constexpr int NS = HAIL ? 5 : 4;
  __shared__ double sRho[3][SG][64], sDz[3][SG][64], sTs[3][SG][64], sF1[2][NS][SG][64], sFi[64], sZz[64];
  __shared__ R sLn[3][SG][64], sRhoc[3][SG][64];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool own = w < NS;             // this wavefront's half
  const int sp = own ? w : w - NS;     // and its species
  const int c = blockIdx.x * 64 + lane;
  const bool in = c < a.ncol;
  const int i = in ? c : a.ncol - 1;  // lanes past the last column repeat it and store nothing
  const double *src = sp == 0 ? a.src_rr : sp == 1 ? a.src_ri : sp == 2 ? a.src_rs : sp == 3 ? a.src_rg : a.src_rh;
  double *dst = sp == 0 ? a.dst_rr : sp == 1 ? a.dst_ri : sp == 2 ? a.dst_rs : sp == 3 ? a.dst_rg : a.dst_rh;
  const FallLaw<R> law = sp == 0   ? fall_law<R>(3)
                         : sp == 1 ? fall_law<R>(4)
                         : sp == 2 ? fall_law<R>(5)
                         : sp == 3 ? fall_law<R>(6)
                                   : fall_law<R>(7);
  const double dt = a.dt, zinv = 1. / by(dt);
  const int top = a.nlev - 1, ng = (a.nlev + SG - 1) / SG;
  // levels below the ground are read as level 0 and not used
  auto at = [&](int k) { return (size_t)(k > 0 ? k : 0) * a.ld + i; };
  double s[SG], rho = 0., dz = 0.;
  auto load_src = [&](int g) {
#pragma unroll
    for (int u = 0; u < SG; ++u) s[u] = src[at(top - SG * g - u)];
  };
  auto load_level = [&](int g) {
    rho = a.rhodref[at(top - SG * g - w)];
    dz = a.dzz[at(top - SG * g - w)];
  };
  auto put_level = [&](int b) {
    const R ln = rlog<R>((R)rho);
    sRho[b][w][lane] = rho;
    sDz[b][w][lane] = dz;
    sLn[b][w][lane] = ln;
    sRhoc[b][w][lane] = fall_rhoc<R>(ln);
    sTs[b][w][lane] = dt / by(rho * dz);
  };
  if (ZZZ && w == 3) sZz[lane] = 0.;  // read by this wavefront only
  load_src(0);
  if (w < SG) {
    load_level(0);
    put_level(0);
    load_level(1);
  }
  __syncthreads();
  // the recurrences, pristine ice's first of all, before the own-content halves that they wait for
  // least: 1,024 columns 61 -> 58 us (float 39.8 -> 35.4), 1 % at 65,536
  if (!own) {
    if (sp == 1) wave_priority<3>();
    else wave_priority<1>();
  }
  double flux = 0.;
  for (int t = 0, b = 0, f = 0; t <= ng; ++t, f ^= 1) {
    const int bn = b == 2 ? 0 : b + 1, bp = b == 0 ? 2 : b - 1;  // buffers of groups t + 1, t - 1
    if (own) {
      double x[SG];
      bool any = false;
#pragma unroll
      for (int u = 0; u < SG; ++u) {
        x[u] = s[u] * dt;
        any = any || x[u] > law.thr;
      }
      load_src(t + 1);
      if (w < SG) {
        put_level(bn);
        load_level(t + 2);
      }
      if constexpr (ZZZ) {  // RAIN_ICE's model level height (rain_ice.F90:387-395)
        if (w == 3) {
          double sum = sZz[lane];
#pragma unroll
          for (int u = 0; u < SG; ++u) {
            const int k = top - SG * t - u;
            sum = sum + sDz[b][u][lane];
            if (in && k >= 0) a.zzz[(size_t)k * a.ld + i] = sum - sDz[b][u][lane] * 0.5;
          }
          sZz[lane] = sum;
        }
      }
      double w1[SG] = {};
      if (__any(any)) {
#pragma unroll
        for (int u = 0; u < SG; ++u) {
          const double v = (double)fall_speed_above<R>(law, x[u], sLn[b][u][lane], sRhoc[b][u][lane]);
          w1[u] = x[u] > law.thr ? v : 0.;
        }
      }
#pragma unroll
      for (int u = 0; u < SG; ++u)
        sF1[f][sp][u][lane] = sediment_own(zinv, sRho[b][u][lane], sDz[b][u][lane], x[u], w1[u]);
    } else if (t > 0) {
      double r[SG];
#pragma unroll
      for (int u = 0; u < SG; ++u) r[u] = s[u];
      load_src(t);
#pragma unroll
      for (int u = 0; u < SG; ++u) {
        const int k = top - SG * (t - 1) - u;
        if (k < 0) break;  // uniform
        sediment_through<R>(law, dt, zinv, sLn[bp][u][lane], sRhoc[bp][u][lane], sDz[bp][u][lane],
                            sTs[bp][u][lane], sF1[f ^ 1][sp][u][lane], r[u], flux);
        if (in) dst[(size_t)k * a.ld + i] = r[u];
      }
    }
    __syncthreads();
    b = bn;
  }
  const double rate = flux / by(P.XRHOLW);
  if (!own && sp == 1) sFi[lane] = rate;
  __syncthreads();
  if (!in || own) return;
  if (sp == 0) {
    a.inprc[i] = 0.;
    a.inprr[i] = rate;
  } else if (sp == 1) {
    a.inpri[i] = rate;
  } else if (sp == 2) {
    a.inprs[i] = rate + sFi[lane];
  } else if (sp == 3) {
    a.inprg[i] = rate;
  } else if constexpr (HAIL) {
    a.inprh[i] = rate;
  }
}

// One thread per column, walking it: few levels, which leave k_sedim's pipeline unfilled, and many
// columns, which hide a column's latency without k_sedim's own-content wavefronts, LDS and barriers.
// 262,144 columns of 90 levels: 559 us, k_sedim 640 (hail 694 and 1019, OCND2 587 and 698); 4 million
// columns of one level: 0.10 ms and 0.60.  The scalar coefficients are worth 10 % here too (616 us without).
template <class R, bool ZZZ = false, bool HAIL = false>
__global__ void __launch_bounds__(256) k_sedim_walk(SedimArgs a) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.ncol) return;
  sedim_column<R, ZZZ, HAIL>(a, i);
}

template <class R, bool ZZZ, bool HAIL>
static hipError_t sedim_launch_as(const SedimArgs &sa, SedimForm form, int ncu, hipStream_t s) {
  if (sa.ncol >= (long long)sedim_walk_cols(form, sa.nlev) * ncu)
    hipLaunchKernelGGL((k_sedim_walk<R, ZZZ, HAIL>), dim3((sa.ncol - 1) / 256 + 1), dim3(256), 0, s, sa);
  else
    hipLaunchKernelGGL((k_sedim<R, ZZZ, HAIL>), dim3((sa.ncol - 1) / 64 + 1), dim3(HAIL ? 640 : 512), 0, s, sa);
  return hipGetLastError();
}

template <> hipError_t sedim_launch<double>(const SedimArgs &sa, int ncu, hipStream_t s) {
  if (sa.src_rh) return sedim_launch_as<double, false, true>(sa, SEDIM_HAIL, ncu, s);
  if (sa.zzz) return sedim_launch_as<double, true, false>(sa, SEDIM_FP64, ncu, s);
  return sedim_launch_as<double, false, false>(sa, SEDIM_FP64, ncu, s);
}

template <> hipError_t sedim_launch<float>(const SedimArgs &sa, int ncu, hipStream_t s) {
  return sedim_launch_as<float, false, false>(sa, SEDIM_MIXED, ncu, s);
}

}  // namespace ice3
