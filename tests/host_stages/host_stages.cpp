// CPU build of the device stages of libice3_hip (dwarf-p-ice3_amd/csrc/ice3_stages.hpp),
// for tests only: the adjust_at / sedim_column / micro_at code that the one-thread kernels
// run (k_ice_adjust, k_sedim_walk, k_adjust_sedim, k_micro_points), executed point by point in
// their launch order (all ICE_ADJUST points, then every column's sedimentation, then every
// microphysics point), so that the kernel source can be checked against the oracle and under
// sanitizers without a GPU.  k_sedim, k_sedim_split and k_micro arrange the same point
// functions over wavefronts in code of their own, which GPU tests alone cover.
// Entry points mirror include/ice3.h with host arrays and no context or stream.
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "ice3_stages.hpp"

using namespace ice3;

static double *g_tab = nullptr;
static double *g_tiwmx = nullptr;  // TIWMX tables of the OCND2 branch
static int g_max_calls = DEFAULT_MAX_CALLS;  // sub-step cap (ice3_ctx_set_substep_cap)

extern "C" int hst_set_substep_cap(int max_calls) {
  if (max_calls < 1) return -1;
  g_max_calls = max_calls;
  return 0;
}

extern "C" int hst_init(void) {
  if (!g_tab || !g_tiwmx) {
    double *tab = (double *)malloc(sizeof(double) * ICE3_T_TOTAL);
    double *tiwmx = (double *)malloc(sizeof(double) * ICE3_TW_NTAB * ICE3_TIWMX_N);
    ice3_params p;
    if (tab && tiwmx) {
      ice3_build_params(&p, tab);
      ice3_build_tiwmx(&p, tiwmx);
    }
    if (!tab || !tiwmx || memcmp(&p, &P, sizeof p) != 0) {  // no memory, or stale constants
      free(tab);
      free(tiwmx);
      return tab && tiwmx ? -2 : -1;
    }
    g_tab = tab;
    g_tiwmx = tiwmx;
  }
  return 0;
}

// The TIWMX tables the kernels read (ice3_tiwmx_tables order), copied into out
// (ICE3_TW_NTAB * ICE3_TIWMX_N doubles).
extern "C" int hst_tiwmx(double *out) {
  if (hst_init()) return -1;
  memcpy(out, g_tiwmx, sizeof(double) * ICE3_TW_NTAB * ICE3_TIWMX_N);
  return ICE3_TW_NTAB;
}

template <class R, bool OCND2 = false>
static void run_rain_ice(const SedimArgs &sa, const MicroArgs &m) {
  for (int i = 0; i < sa.ncol; ++i) sedim_column<R, OCND2>(sa, i);
  unsigned long long n = 0, c = 0, p = 0;
  for (int k = 0; k < m.nlev; ++k)
    for (int i = 0; i < m.ncol; ++i) {
      const int calls = micro_at<R, OCND2>(m, (size_t)k * m.ld + i, m.tab);
      n += calls < 0 ? -calls : calls;
      c += calls < 0;
      p += calls != 0;
    }
  if (m.counters) { m.counters[0] += n; m.counters[1] += c; m.counters[2] += p; }
}

extern "C" int hst_ice_adjust(int ncol, int nlev, int ld, double dt, const ice3_ice_adjust_in *in,
                              const ice3_ice_adjust_out *out) {
  if (hst_init()) return -1;
  AdjustArgs a = AdjustArgs{};
  a.ncol = ncol; a.nlev = nlev; a.ld = ld; a.dt = dt; a.in = *in; a.out = *out;
  for (int k = 0; k < nlev; ++k)
    for (int i = 0; i < ncol; ++i) adjust_at(a, i, (size_t)k * ld + i);
  return 0;
}

extern "C" int hst_ice_adjust_ocnd2(int ncol, int nlev, int ld, double dt,
                                    const ice3_ice_adjust_in *in, const ice3_ocnd2_in *in2,
                                    const ice3_ice_adjust_out *out, const ice3_ocnd2_out *out2) {
  if (hst_init()) return -1;
  AdjustArgs a = AdjustArgs{};
  a.ncol = ncol; a.nlev = nlev; a.ld = ld; a.dt = dt; a.in = *in; a.out = *out;
  const Ocnd2Args x{*in2, *out2, g_tiwmx};
  for (int k = 0; k < nlev; ++k)
    for (int i = 0; i < ncol; ++i) adjust_at<true>(a, i, (size_t)k * ld + i, k, &x);
  return 0;
}

extern "C" int hst_rain_ice(int prec, int ncol, int nlev, int ld, double dt,
                            const ice3_rain_ice_in *in, const ice3_rain_ice_inout *io,
                            const ice3_rain_ice_out *out, const ice3_stats *stats) {
  if (hst_init()) return -1;
  SedimArgs sa;
  MicroArgs m;
  rain_ice_args(ncol, nlev, ld, dt, g_tab, in, io, out, stats, sa, m);
  m.max_calls = g_max_calls;
  if (prec == ICE3_PREC_FP64) run_rain_ice<double>(sa, m);
  else run_rain_ice<float>(sa, m);
  return 0;
}

extern "C" int hst_adjust_rain_ice(int prec, int ncol, int nlev, int ld, double dt,
                                   const ice3_pipeline_in *in, const ice3_pipeline_out *out,
                                   const ice3_stats *stats) {
  if (hst_init()) return -1;
  AdjustArgs aa;
  SedimArgs sa;
  MicroArgs m;
  pipeline_args(ncol, nlev, ld, dt, g_tab, in, out, stats, aa, sa, m);
  m.max_calls = g_max_calls;
  for (int k = 0; k < nlev; ++k)
    for (int i = 0; i < ncol; ++i) adjust_at(aa, i, (size_t)k * ld + i);
  if (prec == ICE3_PREC_FP64) run_rain_ice<double>(sa, m);
  else run_rain_ice<float>(sa, m);
  return 0;
}

extern "C" int hst_rain_ice_ocnd2(int ncol, int nlev, int ld, double dt, const ice3_rain_ice_in *in,
                                  const ice3_rain_ocnd2_in *in2, const ice3_rain_ice_inout *io,
                                  const ice3_rain_ice_out *out, const ice3_stats *stats) {
  if (hst_init()) return -1;
  SedimArgs sa;
  MicroArgs m;
  rain_ice_args(ncol, nlev, ld, dt, g_tab, in, io, out, stats, sa, m);
  m.max_calls = g_max_calls;
  m.icldfr = in2->icldfr; m.ssio = in2->ssio; m.ssiu = in2->ssiu; m.ifr = in2->ifr;
  m.tiwmx = g_tiwmx;
  sa.zzz = out->rainfr;
  run_rain_ice<double, true>(sa, m);
  return 0;
}

extern "C" int hst_adjust_rain_ice_ocnd2(int ncol, int nlev, int ld, double dt,
                                         const ice3_pipeline_in *in, const ice3_ocnd2_in *in2,
                                         const ice3_pipeline_out *out, const ice3_ocnd2_out *out2,
                                         const ice3_stats *stats) {
  if (hst_init()) return -1;
  AdjustArgs aa;
  SedimArgs sa;
  MicroArgs m;
  pipeline_args(ncol, nlev, ld, dt, g_tab, in, out, stats, aa, sa, m);
  m.max_calls = g_max_calls;
  m.icldfr = out2->icldfr; m.ssio = out2->ssio; m.ssiu = out2->ssiu; m.ifr = out2->ifr;
  m.tiwmx = g_tiwmx;
  sa.zzz = out->rainfr;
  const Ocnd2Args x{*in2, *out2, g_tiwmx};
  for (int k = 0; k < nlev; ++k)
    for (int i = 0; i < ncol; ++i) adjust_at<true>(aa, i, (size_t)k * ld + i, k, &x);
  run_rain_ice<double, true>(sa, m);
  return 0;
}

// ---- hail (KRR=7): the kernels' order (all columns' sedimentation, then every point's
// microphysics), with the hail stage functions.
static void run_rain_ice_hail(const SedimArgs &sa, const MicroArgs &m) {
  for (int i = 0; i < sa.ncol; ++i) sedim_column<double, false, true>(sa, i);
  unsigned long long n = 0, c = 0, p = 0;
  for (int k = 0; k < m.nlev; ++k)
    for (int i = 0; i < m.ncol; ++i) {
      const int calls = micro_at<double, false, true>(m, (size_t)k * m.ld + i, m.tab);
      n += calls < 0 ? -calls : calls;
      c += calls < 0;
      p += calls != 0;
    }
  if (m.counters) { m.counters[0] += n; m.counters[1] += c; m.counters[2] += p; }
}

extern "C" int hst_ice_adjust_hail(int ncol, int nlev, int ld, double dt,
                                   const ice3_ice_adjust_in *in, const double *rh,
                                   const ice3_ice_adjust_out *out) {
  if (hst_init()) return -1;
  AdjustArgs a = AdjustArgs{};
  a.ncol = ncol; a.nlev = nlev; a.ld = ld; a.dt = dt; a.in = *in; a.out = *out; a.rh = rh;
  for (int k = 0; k < nlev; ++k)
    for (int i = 0; i < ncol; ++i) adjust_at<false, true>(a, i, (size_t)k * ld + i);
  return 0;
}

extern "C" int hst_rain_ice_hail(int ncol, int nlev, int ld, double dt, const ice3_rain_ice_in *in,
                                 const ice3_rain_ice_inout *io, const ice3_rain_ice_out *out,
                                 const ice3_hail *hail, const ice3_stats *stats) {
  if (hst_init()) return -1;
  SedimArgs sa;
  MicroArgs m;
  rain_ice_args(ncol, nlev, ld, dt, g_tab, in, io, out, stats, sa, m);
  m.max_calls = g_max_calls;
  sa.src_rh = hail->rhs; sa.dst_rh = hail->rhs; sa.inprh = hail->inprh;
  m.t[IRH] = hail->rht; m.src[IRH] = hail->rhs; m.dst[IRH] = hail->rhs;
  run_rain_ice_hail(sa, m);
  return 0;
}

extern "C" int hst_adjust_rain_ice_hail(int ncol, int nlev, int ld, double dt,
                                        const ice3_pipeline_in *in, const ice3_pipeline_out *out,
                                        const ice3_pipeline_hail *hail, const ice3_stats *stats) {
  if (hst_init()) return -1;
  AdjustArgs aa;
  SedimArgs sa;
  MicroArgs m;
  pipeline_args(ncol, nlev, ld, dt, g_tab, in, out, stats, aa, sa, m);
  m.max_calls = g_max_calls;
  aa.rh = hail->rh;
  sa.src_rh = hail->rhs; sa.dst_rh = hail->rhs_out; sa.inprh = hail->inprh;
  m.t[IRH] = hail->rhs; m.src[IRH] = hail->rhs_out; m.dst[IRH] = hail->rhs_out;
  for (int i = 0; i < ncol; ++i) adjust_sedim_column<double, true>(aa, sa, i);
  for (int k = 0; k < m.nlev; ++k)
    for (int i = 0; i < m.ncol; ++i) {
      const int calls = micro_at<double, false, true>(m, (size_t)k * m.ld + i, m.tab);
      if (stats && stats->counters) {
        stats->counters[0] += calls < 0 ? -calls : calls;
        stats->counters[1] += calls < 0;
        stats->counters[2] += calls != 0;
      }
    }
  return 0;
}

#ifdef HST_MAIN
// Sanitizer driver: host_stages_san <dir> <ncol> <nlev> <dt> <prec> reads
// <dir>/<field>.bin (float64, (nlev, ncol), sigqsat (ncol)) for every
// ice3_pipeline_in field, runs the fused step with exact-size heap buffers and
// writes <dir>/out_<field>.bin.
static double *load(const char *dir, const char *name, size_t n) {
  char path[1024];
  snprintf(path, sizeof path, "%s/%s.bin", dir, name);
  FILE *f = fopen(path, "rb");
  if (!f) { fprintf(stderr, "missing %s\n", path); exit(2); }
  double *v = (double *)malloc(n * sizeof(double));
  if (fread(v, sizeof(double), n, f) != n) { fprintf(stderr, "short %s\n", path); exit(2); }
  fclose(f);
  return v;
}

static void save(const char *dir, const char *name, const void *v, size_t bytes) {
  char path[1024];
  snprintf(path, sizeof path, "%s/out_%s.bin", dir, name);
  FILE *f = fopen(path, "wb");
  if (!f) exit(2);
  fwrite(v, 1, bytes, f);
  fclose(f);
}

int main(int argc, char **argv) {
  if (argc != 6) return 2;
  const char *dir = argv[1];
  const int ncol = atoi(argv[2]), nlev = atoi(argv[3]), prec = atoi(argv[5]);
  const double dt = atof(argv[4]);
  const size_t n = (size_t)ncol * nlev;
  static const char *IN[] = {"pabs", "sigs", "th", "exn", "exn_ref", "rhodref", "rhodj", "dzz",
                             "rv", "rc", "ri", "rr", "rs", "rg", "ci", "cf_mf", "rc_mf", "ri_mf",
                             "ths", "rvs", "rcs", "rrs", "ris", "rss", "rgs", "sigqsat"};
  static const char *OUT[] = {"ths", "rvs", "rcs", "rrs", "ris", "rss", "rgs", "cldfr",
                              "hlc_hrc", "hlc_hcf", "hli_hri", "hli_hcf", "ci", "evap3d",
                              "rainfr", "inprc", "inprr", "inpri", "inprs", "inprg"};
  const double *inp[26];
  for (int q = 0; q < 26; ++q) inp[q] = load(dir, IN[q], q == 25 ? (size_t)ncol : n);
  double *outp[20];
  for (int q = 0; q < 20; ++q) outp[q] = (double *)malloc((q >= 15 ? (size_t)ncol : n) * 8);
  ice3_pipeline_in pin;
  ice3_pipeline_out pout;
  static_assert(sizeof pin == 26 * sizeof(void *), "ice3_pipeline_in layout");
  static_assert(sizeof pout == 20 * sizeof(void *), "ice3_pipeline_out layout");
  memcpy(&pin, inp, sizeof pin);
  memcpy(&pout, outp, sizeof pout);
  int *calls = (int *)malloc(n * sizeof(int));
  unsigned long long counters[3] = {0, 0, 0};
  ice3_stats st = {calls, counters};
  if (hst_adjust_rain_ice(prec, ncol, nlev, ncol, dt, &pin, &pout, &st)) return 3;
  for (int q = 0; q < 20; ++q) save(dir, OUT[q], outp[q], (q >= 15 ? (size_t)ncol : n) * 8);
  save(dir, "calls", calls, n * sizeof(int));
  printf("calls %llu capped %llu micro_points %llu\n", counters[0], counters[1], counters[2]);
  for (int q = 0; q < 26; ++q) free((void *)inp[q]);
  for (int q = 0; q < 20; ++q) free(outp[q]);
  free(calls);
  free(g_tab);
  return 0;
}
#endif

// The FP64 exp and log of the physics kernels (ice3_physics.hpp), elementwise.
extern "C" void hst_exp_f64(const double *x, double *y, long n) {
  for (long q = 0; q < n; ++q) y[q] = exp_f64(x[q]);
}
extern "C" void hst_log_f64(const double *x, double *y, long n) {
  for (long q = 0; q < n; ++q) y[q] = log_f64(x[q]);
}

// From how many columns a compute unit the sedimentation walks (ice3_stages.hpp: sedim_walk_cols).
extern "C" int hst_sedim_walk_cols(int form, int nlev) { return sedim_walk_cols((SedimForm)form, nlev); }

// The OCND2 tables' index of a temperature, and their length (ice3_physics.hpp: tiwmx_index).
extern "C" int hst_tiwmx_index(double t) { return tiwmx_index(t); }
extern "C" int hst_tiwmx_n(void) { return ICE3_TIWMX_N; }

// The kernels' FP64 quotients a / b from given approximate reciprocals r0 (ice3_physics.hpp: by_from,
// corrected_quotient); fma is the C library's.
extern "C" void hst_quotients(const double *a, const double *b, const double *r0, double *q, long n) {
  for (long e = 0; e < n; ++e) q[e] = corrected_quotient(a[e], by_from(b[e], r0[e]));
}
