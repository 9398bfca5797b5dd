// p3_kernel.hpp -- p3_main_init, part 1 and part 2 of a P3 step in one kernel
// (sedimentation and part 3 are in p3_sed.hpp).
//
// Both parts are pointwise in the level, so p3_front_kernel runs them with one
// thread per (level, column).  The reference's early exits are column-wide, but
// nothing a point computes depends on them (front_level says why); the column
// status words are kept only where a caller reads them or needs the exchange
// fields untouched (KParams::track).
//
// The step follows components/eamxx/src/physics/p3/impl/p3_main_impl.hpp:74-260.
#pragma once

#include "p3_part2.hpp"

namespace p3d {

// Scratch fields (ncol x nlev doubles each, in the layout of the column set):
// per-level results of part 1 for sedimentation and part 3 (T, rhofacr,
// rhofaci, acn), and the marks of part 2's pending levels (SC_PEND, only
// without exch_zero).
// SC_WET and SC_ORDER hold the words and the lists of p3_order_kernel.
enum Scr { SC_T = 0, SC_RHOFACR, SC_RHOFACI, SC_ACN, SC_PEND, SC_WET, SC_ORDER, SC_COUNT };

// The P3Microphysics pre- and post-amble (eamxx_p3_process_interface.hpp:63-261),
// fused into part 1 and part 3 when `on`.  The prognostic pointers then hold the
// field manager's wet mixing ratios: part 1 reads them wet and writes them dry,
// part 3 writes them wet again; th is the process's own array.
struct Amble {
  int on;
  const double *p_mid, *dp_wet, *cldfrac_tot;  // p_mid, pseudo_density, cldfrac_tot
  double *T_mid, *T_prev;                      // T_mid (in, out), T_prev_micro_step (out)
  double* qv_prev;                             // qv_prev_micro_step: wet in, dry in p3_main, wet out
  double *dz, *inv_exner, *cld_frac_l, *cld_frac_i, *rainfrac;  // P3 inputs part 1 writes
  double *precip_liq_mass, *precip_ice_mass;   // per column, accumulated
  double *vapor_flux, *water_flux, *ice_flux, *heat_flux;  // per column; NULL = off
};

struct KParams {
  // P3PrognosticState (in/out)
  double *qc, *nc, *qr, *nr, *qi, *qm, *ni, *bm, *qv, *th;
  // P3DiagnosticInputs
  const double *nc_nuceat_tend, *nccn, *ni_activated, *inv_qc_relvar, *cld_frac_i, *cld_frac_l,
      *cld_frac_r, *pres, *dz, *dpres, *inv_exner, *qv_prev, *t_prev;
  // P3DiagnosticOutputs
  double *qv2qi_depos_tend, *precip_liq_surf, *precip_ice_surf, *diag_eff_radius_qc,
      *diag_eff_radius_qi, *diag_eff_radius_qr, *rho_qi, *precip_liq_flux, *precip_ice_flux,
      *precip_total_tend, *nevapr;
  // P3HistoryOnly (in/out unless exch_zero)
  double *liq_ice_exchange, *vap_liq_exchange, *vap_ice_exchange;
  double* scratch;      // SC_COUNT fields of sfs doubles
  int* colstat;         // per column: 0 skipped after part 1, 1 after part 2, 3 full step (if track())
  unsigned* err;        // error word, in device or in pinned host memory
  int *dbg_status, *dbg_substeps, *dbg_ice_idx;
  int* dbg_check;       // per column: check_values flags (NULL = the check is off)
  Tables tab;
  Runtime rt;
  RainGamma rg, rgf;    // of the FP64 and of the mixed form
  int ncol, nlev;
  // Layout.  Element (column i, level k) of a level field is at i*cs + k*ks, of
  // an interface field (nlev + 1 levels) at i*fcs + k*fks: level-major
  // (cs = fcs = 1, ks = fks = the row stride) or column-major, the reference's
  // (column, level) LayoutRight views (ks = fks = 1, cs and fcs the column
  // strides).  Scratch field f holds (i, k) at f*sfs + i*scs + k*sks, dense, in
  // the same order.
  int cs, ks, fcs, fks;
  int scs, sks;
  size_t sfs;
  int colmajor;         // 1: column-major; the pointwise kernels then map lanes to levels
  int dbg_stride;       // species stride of dbg_substeps (>= ncol)
  double dt;
  int predictNc, prescribedCCN, exch_zero;
  int keep_order;       // sedimentation takes the columns as they come (order())
  double e_melt;        // saturation vapour pressure over liquid at Tmelt (qv_sat_dry(Tmelt, p) numerator)
  Amble amble;

  // The step keeps the column status words: for the status array, for
  // check_values (fully stepped columns only), or for exchange fields that a
  // skipped column leaves as they were.
  __host__ __device__ __forceinline__ bool track() const { return dbg_status || dbg_check || !exch_zero; }
  // Sedimentation with several columns per wavefront takes them in the order of
  // p3_order_kernel.  Not with the status words: the lists would hold there too (a
  // column that the reference skips has none of the species), but the gain is measured
  // without them.  And only where the words and lists fit their scratch fields and
  // the counts their 21 bits each.
  __host__ __device__ __forceinline__ bool ordered() const {
    return !keep_order && !track() && ncol >= 64 && ncol < 1 << 21 && nlev >= 16;
  }
  // The words: a bit per column, 8 bytes per 64 columns, a row per level, for
  // cloud, rain and ice.
  __host__ __device__ __forceinline__ int wet_words() const { return (ncol + 63) / 64; }
  __device__ __forceinline__ unsigned long long* wet(int species) const {
    return (unsigned long long*)(scratch + SC_WET * sfs) + (size_t)species * nlev * wet_words();
  }
  // The counts of the blocks that have appended so far (21 bits each: columns, of
  // them with cloud or rain, with ice), and each group's list.
  __device__ __forceinline__ unsigned long long* order_count() const {
    return (unsigned long long*)(scratch + SC_ORDER * sfs);
  }
  __device__ __forceinline__ uint2* order(int group) const { return (uint2*)(order_count() + 1) + (size_t)group * ncol; }
  __host__ __device__ __forceinline__ size_t at(int i, int k) const { return (size_t)i * cs + (size_t)k * ks; }
  __host__ __device__ __forceinline__ size_t atf(int i, int k) const { return (size_t)i * fcs + (size_t)k * fks; }
  __host__ __device__ __forceinline__ double& sc(int f, int i, int k) const {
    return scratch[(size_t)f * sfs + (size_t)i * scs + (size_t)k * sks];
  }
};

__host__ __device__ __forceinline__ double exner_function(double pres) {  // PhysicsFunctions, p^(Rd/cp)
  return p3m_pow(p3m_div(pres, P0), Rair * INV_CP);
}

// Air density of a layer (dpres / dz / g), as every kernel forms it.
__device__ __forceinline__ double air_density(double dpres, double dz) {
  return p3m_div(p3m_div_inf(dpres, dz), gravit);
}

// q * num / den of several q, with one reciprocal; both factors are scaled by a power
// of two where den is too small for that, which changes no bit of a quotient.
struct Ratio {
  double num, den, rden;
  __device__ __forceinline__ Ratio(double n, double d) {
    const double s = m_fabs(d) < 0x1p-1000 ? 0x1p100 : 1.0;
    num = n * s;
    den = d * s;
    rden = p3m_recip(den);
  }
  __device__ __forceinline__ double of(double q) const { return p3m_div_y_inf(q * num, den, rden); }
};

constexpr int kMaxSubsteps = 100000;
// Column status bits: part 1 found work, part 2 left hydrometeors.
constexpr int kStatusPart1 = 1, kStatusPart2 = 2, kStatusFull = 3;
// What front_level leaves to sediment at its level: cloud, and the next bits rain and ice.
constexpr int kWet = 4;
// Species groups of the sedimentation and of its lists of columns.
enum SedGroup { SED_LIQ = 0, SED_ICE = 1 };

template <class R> struct RainOf {
  static __device__ __forceinline__ const RainGamma& get(const KParams& p) { return sizeof(R) == 8 ? p.rg : p.rgf; }
};

// p3_main_init, part 1 (P3I/p3_main_impl_part1.hpp:18-185) and part 2
// (P3I/p3_main_impl_part2.hpp:113-524) of level k of column i.
//
// The reference skips a column after part 1 unless some level of it has
// hydrometeors or may nucleate ice (P3I/p3_main_impl.hpp:222-230), and after
// part 2 unless some level has hydrometeors (:255-260).  A point needs neither:
//  * a level with hydrometeors or possible nucleation (its own flag is set)
//    makes its column run, so part 2 runs exactly there (unless skip_all);
//  * a level without, in a column that runs because of other levels, is either
//    skip_all or warm and clear; part 2 changes nothing at the latter (every
//    tendency is zero) but zeroes its exchange fields.  Where those are not
//    zeroed on entry, the level is marked pending in scratch and part 3, which
//    knows the column's status, zeroes them;
//  * sedimentation runs for a species that is present, and a level that has
//    hydrometeors after part 2 makes its column run.
//
// What part 2 needs later than it is computed stays in LDS (s), not in
// registers: 28 doubles per point in FP64, 26 in the mixed form.  Without that part 2
// alone spilled at two wavefronts per SIMD in FP64 and could not run at three in the
// mixed form.
//
// Bound by the latency of its loads and table gathers at two and three wavefronts per
// SIMD: the VALU is busy 52 % of the time in FP64, 74 % in the mixed form.  As kernels of
// their own, part 1 (at the HBM rate) wrote seven scratch fields and part 2
// (43 % busy, waiting on loads) read them and the state again.  Together, at
// 21600 x 72 FP64 48 + 187 -> 225 us, at 16384 x 128 mixed 67 + 189 -> 195 us,
// and a launch (two with the status words' clear) fewer.  One logarithm of T for
// the saturation values, T^1.5 and T^1.81, one viscosity for both parts, the rain
// gammas from outside (RainGamma) and polynomial coefficients in scalar registers
// then made it 203 and 187 us.
template <class R>
__device__ __forceinline__ void front_level(const KParams& p, int k, int i, const Pt s, int& stat, unsigned& err) {
  const double dt = p.dt;
  const double latvap = LatVap, latice = LatIce, inv_cp = INV_CP;
  const Runtime& rt = p.rt;
  const size_t x = p.at(i, k);
  int flags = 0;  // bit 0 nucleationPossible, bit 1 hydrometeorsPresent
  double inv_exner, th, qv, qc, nc, qr, nr, qi, ni, qm, bm, dz;
  double cfl = 1.0, cfr = 1.0, cfi = 1.0, qv_prev = 0, t_prev = 0, ni_act = 0;
  if (p.amble.on) {
    // p3_preamble, eamxx_p3_process_interface.hpp:63-124
    const Amble& a = p.amble;
    const double pmid = a.p_mid[x], T = a.T_mid[x], cft = a.cldfrac_tot[x];
    const double dp = a.dp_wet[x], dp_dry = p.dpres[x];
    const double c1 = -1.0 + 1.0 / ep_2;  // calculate_dz with the wet qv's virtual temperature
    const double T_virtual = T * (1.0 + c1 * p.qv[x]);
    dz = p3m_div_inf((Rair / gravit) * dp * T_virtual, pmid);
    a.dz[x] = dz;
    // wet -> dry mixing ratios (calculate_drymmr_from_wetmmr_dp_based)
    const Ratio dry(dp, dp_dry);
    auto to_dry = [&](double q) { return dry.of(q); };
    qc = to_dry(p.qc[x]); nc = to_dry(p.nc[x]); qr = to_dry(p.qr[x]);
    nr = to_dry(p.nr[x]); qi = to_dry(p.qi[x]); ni = to_dry(p.ni[x]);
    qm = to_dry(p.qm[x]); bm = to_dry(p.bm[x]);
    qv = to_dry(p.qv[x]);
    qv_prev = to_dry(a.qv_prev[x]);
    a.qv_prev[x] = qv_prev;
    const double ex = exner_function(pmid), rex = p3m_recip(ex);
    inv_exner = p3m_div_y(1.0, ex, rex);
    a.inv_exner[x] = inv_exner;
    th = p3m_div_y(T, ex, rex);
    // cloud fractions with the 1e-4 floor and the maximum-overlap rain fraction
    cfl = cft > 0.0001 ? cft : 0.0001;
    cfi = cfl;
    a.cld_frac_l[x] = cfl;
    a.cld_frac_i[x] = cfl;
    cfr = cfl;
    if (k != 0) {
      const double above = a.cldfrac_tot[x - p.ks];
      cfr = above > cfr ? above : cfr;
    }
    a.rainfrac[x] = cfr;
  } else {
    inv_exner = p.inv_exner[x];
    th = p.th[x];
    qv = p.qv[x];
    qc = p.qc[x]; nc = p.nc[x]; qr = p.qr[x]; nr = p.nr[x];
    qi = p.qi[x]; ni = p.ni[x]; qm = p.qm[x]; bm = p.bm[x];
    dz = p.dz[x];
    if (p.prescribedCCN) cfl = p.cld_frac_l[x];
  }
  const double pres = p.pres[x], dpres = p.dpres[x];
  // What only part 2 reads is requested as soon as the point is known to need
  // it, and arrives while part 1 computes.
  auto load_late = [&] {
    if (!p.amble.on) {
      cfl = p.cld_frac_l[x];
      cfr = p.cld_frac_r[x];
      cfi = p.cld_frac_i[x];
      qv_prev = p.qv_prev[x];
    }
    t_prev = p.t_prev[x];
    ni_act = p.ni_activated[x];
  };
  const bool wet = qc >= QSMALL || qr >= QSMALL || qi >= QSMALL;
  if (wet) load_late();

  // the state as it is in memory: a field left bit for bit unchanged is not
  // stored again (with the pre-amble every field changes to dry)
  const double in[10] = {qc, nc, qr, nr, qi, ni, qm, bm, qv, th};
  qv = vmax(qv, 0.0);
  const double exner = p3m_div_inf(1.0, inv_exner);
  double T_atm = th * exner;
  // The mixed form refuses an inverse Exner function of 0 (an array never filled), as it
  // did when its divisions made T NaN of it; in FP64 T is infinite, which passes.
  if (sizeof(R) == 4 && !(m_fabs(exner) < p3m_inf())) err |= ERR_BAD_TEMPERATURE;
  const double rho = air_density(dpres, dz);
  const double inv_rho = p3m_div_inf(1.0, rho);
  const double T_first = T_atm;
  double lh, ll;
  log_temperature(T_atm, lh, ll);
  double qv_sat_l, qv_sat_i;
  qv_sat_dry_both(T_atm, lh + ll, pres, qv_sat_l, qv_sat_i, err);
  const double qv_supersat_i = p3m_div_inf(qv, qv_sat_i) - 1;
  double rhofacr, rhofaci, acn;
  R mu;
  {
    const R ir = R(inv_rho), Tr = R(T_atm);
    rhofacr = double(m_pow(R(RHO_1000MB) * ir, R(.54)));
    rhofaci = double(m_pow(R(RHO_600MB) * ir, R(.54)));
    mu = viscosity(Tr, pow_of_log(Tr, lh, ll, R(1.5)));
    acn = double(m_div(R(gravit) * R(RHO_H2O), R(18) * mu));
  }
  if (T_atm < T_zerodegc && qv_supersat_i >= -0.05) flags |= 1;

  if (qc < QSMALL) {
    qv = qv + qc;
    th = th - inv_exner * qc * latvap * inv_cp;
    qc = 0; nc = 0;
  } else {
    flags |= 2;
    if (p.prescribedCCN) nc = vmax(nc, rt.spa_ccn_to_nc_factor * p.nccn[x] / (1 / cfl));
    else if (p.predictNc) nc = vmax(nc + p.nc_nuceat_tend[x] * dt, 0.0);
    else nc = NCCNST * inv_rho;
  }
  if (qr < QSMALL) {
    qv = qv + qr;
    th = th - inv_exner * qr * latvap * inv_cp;
    qr = 0; nr = 0;
  } else {
    flags |= 2;
  }
  if (qi < QSMALL || (qi < 1.e-8 && qv_supersat_i < -0.1)) {
    qv = qv + qi;
    th = th - inv_exner * qi * (latvap + latice) * inv_cp;
    qi = 0; ni = 0; qm = 0; bm = 0;
  } else {
    flags |= 2;
  }
  if (qi >= QSMALL && qi < 1.e-8 && T_atm >= T_zerodegc) {
    qr = qr + qi;
    th = th - inv_exner * qi * latice * inv_cp;
    qi = 0; ni = 0; qm = 0; bm = 0;
  }
  T_atm = th * exner;

  p.sc(SC_T, i, k) = T_atm;
  p.sc(SC_RHOFACR, i, k) = rhofacr;
  p.sc(SC_RHOFACI, i, k) = rhofaci;
  p.sc(SC_ACN, i, k) = acn;

  // state fields to store: bit q for field q of f
  unsigned chg = p.amble.on ? 0x3ffu : 0u;
  double st[10] = {qc, nc, qr, nr, qi, ni, qm, bm, qv, th};
#pragma unroll
  for (int q = 0; q < 10; ++q)
    if (__double_as_longlong(st[q]) != __double_as_longlong(in[q])) chg |= 1u << q;

  const bool skip_all = qc < QSMALL && qr < QSMALL && qi < QSMALL && T_atm < T_zerodegc && qv_supersat_i < -0.05;
  const bool done = flags && !skip_all;
  if (p.track()) {
    stat = flags ? kStatusPart1 : 0;
    if (!p.exch_zero) p.sc(SC_PEND, i, k) = !flags && !skip_all ? 1.0 : 0.0;
  }
  if (done) {
    if (!wet) load_late();
#pragma unroll
    for (int q = 0; q < 10; ++q) s[S_QC + q] = st[q];
    s[S_T] = T_atm; s[S_PRES] = pres; s[S_RHO] = rho; s[S_INV_RHO] = inv_rho;
    s[S_QVSL] = qv_sat_l; s[S_QVSI] = qv_sat_i; s[S_SUPI] = qv_supersat_i;
    s[S_RHOFACI] = rhofaci;
    s[S_CFL] = cfl; s[S_CFR] = cfr; s[S_CFI] = cfi;
    s[S_INV_EXNER] = inv_exner; s[S_QV_PREV] = qv_prev; s[S_T_PREV] = t_prev; s[S_NI_ACT] = ni_act;
    // T and so its logarithm and viscosity are part 1's unless it clipped a trace
    if (T_atm != T_first) {
      if constexpr (sizeof(R) == 8) log_temperature(T_atm, lh, ll);
      mu = viscosity(R(T_atm), pow_of_log(R(T_atm), lh, ll, R(1.5)));
    }
    if constexpr (sizeof(R) == 8) {
      s[S_MU] = mu;
      s[S_ACN] = acn;
      s[S_T181] = p3m_pow_log(lh, ll, 1.81);
    } else {
      s.pair(S_MU) = make_float2(mu, float(acn));  // acn was formed in FP32
    }
    lds_fence();
    P2Out o;
    // hydrometeorsPresent after part 2 (P3I/p3_main_impl.hpp:255-260): a column flag
    if (part2_level<R>(rt, RainOf<R>::get(p), p.tab, dt, p.predictNc, p.prescribedCCN, p.e_melt,
                       s, st, chg, o, err))
      stat |= kStatusPart2;
    p.qv2qi_depos_tend[x] = o.qv2qi_depos_tend;
    p.precip_total_tend[x] = o.precip_total_tend;
    p.nevapr[x] = o.nevapr;
    p.vap_ice_exchange[x] = o.vap_ice_exchange;
    p.vap_liq_exchange[x] = o.vap_liq_exchange;
    p.liq_ice_exchange[x] = o.liq_ice_exchange;
  } else {
    p.qv2qi_depos_tend[x] = 0;
    p.precip_total_tend[x] = 0;
    p.nevapr[x] = 0;
    if (p.exch_zero) {
      p.vap_ice_exchange[x] = 0;
      p.vap_liq_exchange[x] = 0;
      p.liq_ice_exchange[x] = 0;
    }
  }
  double* const f[10] = {p.qc, p.nc, p.qr, p.nr, p.qi, p.ni, p.qm, p.bm, p.qv, p.th};
#pragma unroll
  for (int q = 0; q < 10; ++q)
    if (chg >> q & 1) f[q][x] = st[q];
#pragma unroll
  for (int sp = 0; sp < 3; ++sp)
    if (st[2 * sp] >= QSMALL) stat |= kWet << sp;
}

// Tiles of the pointwise kernels (part 1, part 2, part 3): 256 threads, one
// (level, column) point each, arranged so that a wavefront's loads coalesce:
//  * level-major: 64 consecutive columns x 4 levels, one level per wavefront,
//    columns fastest, so a wavefront reads 64 consecutive doubles of a row
//    (and holds points of one level, whose work is alike);
//  * column-major, two arrangements:
//    - PW_RUNS (part 3, memory-bound): 256 consecutive points of the
//      column-by-column order, so a wavefront reads 512 contiguous bytes;
//    - PW_BLOCKS (parts 1 and 2): a wavefront holds 8 columns x 8 consecutive levels
//      (levels fastest, 8 runs of 64 bytes per load), a block 32 columns x 8
//      levels, so that a wavefront's points are of nearby levels: the upper
//      levels are mostly dry and skip part 2's processes, and a wavefront
//      spanning a whole column would run them for its few wet lanes (part 2
//      330 -> 270 us at 21600 x 72 against PW_RUNS).
//    Both take the same grid (the larger of their tile counts); tiles past an
//    arrangement's end hold no points.
constexpr int kPart2Cols = 64, kPart2Levels = 4;
static_assert(kTileThreads == kPart2Cols * kPart2Levels, "one point per thread");
constexpr int kBlkCols = 32, kBlkLevels = 8;
enum PwMap { PW_RUNS = 0, PW_BLOCKS = 1 };
__host__ __device__ __forceinline__ int part2_tiles(int ncol, int nlev) {
  return ((ncol + kPart2Cols - 1) / kPart2Cols) * ((nlev + kPart2Levels - 1) / kPart2Levels);
}
__host__ __device__ __forceinline__ int pw_tiles(const KParams& p) {
  if (p.colmajor) {
    const int runs = (int)(((long long)p.ncol * p.nlev + kTileThreads - 1) / kTileThreads);
    const int blocks = ((p.ncol + kBlkCols - 1) / kBlkCols) * ((p.nlev + kBlkLevels - 1) / kBlkLevels);
    return runs > blocks ? runs : blocks;
  }
  return part2_tiles(p.ncol, p.nlev);
}
// The point of this thread in tile `tile`; false past the end of the set.
// (Column-major point counts are below 2^31: the host refuses larger sets.)
template <int MAP>
__device__ __forceinline__ bool pw_point(const KParams& p, int tile, int& i, int& k) {
  if (p.colmajor) {
    if constexpr (MAP == PW_RUNS) {
      const unsigned e = (unsigned)tile * kTileThreads + threadIdx.x;
      const unsigned nl = (unsigned)p.nlev;
      i = (int)(e / nl);
      k = (int)(e - (unsigned)i * nl);
      return i < p.ncol;
    } else {
      const int ntc = (p.ncol + kBlkCols - 1) / kBlkCols;
      const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
      i = (tile % ntc) * kBlkCols + w * 8 + (l >> 3);
      k = (tile / ntc) * kBlkLevels + (l & 7);
      return i < p.ncol && k < p.nlev;
    }
  }
  const int ntc = (p.ncol + kPart2Cols - 1) / kPart2Cols;
  i = (tile % ntc) * kPart2Cols + (threadIdx.x & 63);
  k = (tile / ntc) * kPart2Levels + (threadIdx.x >> 6);
  return i < p.ncol && k < p.nlev;
}

// ORs `bit` into the status word of column i for every lane whose `set` is
// true, one atomic per column and wavefront, on the points of pw_point<PW_BLOCKS>.
// Level-major lanes hold distinct columns; column-major the aligned groups of 8
// lanes hold one column's levels, and the lowest lane of a group with `set` makes
// the atomic.  Every lane of the wavefront that is still running must call this.
__device__ __forceinline__ void colstat_or(const KParams& p, int i, bool set, int bit) {
  if (!p.colmajor) {
    if (set) atomicOr(&p.colstat[i], bit);
    return;
  }
  const unsigned long long m = __ballot(set);
  const int l = threadIdx.x & 63;
  const unsigned long long below = (0xFFull << (l & ~7)) & ((1ull << l) - 1);
  if (set && !(m & below)) atomicOr(&p.colstat[i], bit);
}

// Stores where the points of pw_point<PW_BLOCKS> hold species sp, from the ballot
// m of the wavefront's lanes; (i, k) is this lane's point.
__device__ __forceinline__ void put_wet(const KParams& p, int sp, int i, int k, unsigned long long m) {
  unsigned long long* const w = p.wet(sp);
  const int lane = threadIdx.x & 63;
  if (!p.colmajor) {
    if (lane == 0) w[(size_t)k * p.wet_words() + i / 64] = m;
    return;
  }
  // a byte per column, a bit per level: transposed, and a byte per level from the
  // first column's lanes
  unsigned long long t = (m ^ m >> 7) & 0x00aa00aa00aa00aaull;
  m ^= t ^ t << 7;
  t = (m ^ m >> 14) & 0x0000cccc0000ccccull;
  m ^= t ^ t << 14;
  t = (m ^ m >> 28) & 0x00000000f0f0f0f0ull;
  m ^= t ^ t << 28;
  if (lane < 8) ((unsigned char*)w)[(size_t)k * p.wet_words() * 8 + i / 8] = (unsigned char)(m >> 8 * lane);
}

// Orders the columns of a step for each sedimentation group, those with the
// group's species first and the others behind them, and finds the top levels of
// their species: entry {column, top levels of the group's first and second species
// in 16 bits each (nlev: none)}.  A wavefront that sediments several columns lasts
// as long as its longest; with clear columns spread among the wet ones nearly every
// wavefront carries idle lanes.  The blocks append in the order in which they
// arrive: the lists differ from run to run, the results do not.
//
// Bound by latency (one round of loads, one atomic): block blk of the set takes the
// columns [blk * kOrderCols, + kOrderCols), stages kOrderRows levels of their words
// in LDS at a time and searches them in groups of 8 levels, then within the group.
// With a loop over the levels' words in global memory instead it took 16 and 26 us
// at 21600 x 72 and 16384 x 128, now 6 and 6.  Sedimentation itself, which no longer
// searches for the top levels: 21600 x 72 mixed dt 1800, a third of the columns clear,
// 267 -> 208 us; 16384 x 128 mixed dt 100, none clear, 158 -> 138.
constexpr int kOrderCols = 512, kOrderRows = 128, kOrderThreads = 1024;
__device__ __forceinline__ void order_block(const KParams& p, int blk) {
  constexpr int kWords = kOrderCols / 64, kGroups = kOrderRows / 8;
  static_assert(kWords * kOrderRows == kOrderThreads && 3 * kGroups * kWords <= kOrderThreads, "one word per thread");
  __shared__ unsigned long long s_row[3][kOrderRows][kWords], s_grp[3][kGroups][kWords];
  __shared__ int s_n[2][kWords];
  __shared__ unsigned long long s_at;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nw = p.wet_words(), nlev = p.nlev;
  const bool lists = threadIdx.x < kOrderCols;  // whole wavefronts, one thread per column
  const int i = blk * kOrderCols + threadIdx.x;
  int top[3] = {nlev, nlev, nlev};
  for (int k0 = 0; k0 < nlev; k0 += kOrderRows) {
    const int row = threadIdx.x / kWords, q = threadIdx.x % kWords, w = blk * kWords + q, k = k0 + row;
#pragma unroll
    for (int sp = 0; sp < 3; ++sp) s_row[sp][row][q] = k < nlev && w < nw ? p.wet(sp)[(size_t)k * nw + w] : 0;
    __syncthreads();
    if (threadIdx.x < 3 * kGroups * kWords) {
      const int sp = threadIdx.x / (kGroups * kWords), g = threadIdx.x / kWords % kGroups;
      unsigned long long any = 0;
#pragma unroll
      for (int r = 0; r < 8; ++r) any |= s_row[sp][g * 8 + r][q];
      s_grp[sp][g][q] = any;
    }
    __syncthreads();
    if (lists) {
      const unsigned bit = 1u << (lane & 31);
      const int h = wave * 2 + (lane >> 5);  // the 32-bit half word of this column
#pragma unroll
      for (int sp = 0; sp < 3; ++sp) {
        int g = kGroups;
#pragma unroll
        for (int n = kGroups - 1; n >= 0; --n)
          if (((const unsigned*)s_grp[sp][n])[h] & bit) g = n;
        if (top[sp] == nlev && g < kGroups) {
          int r = 0;
#pragma unroll
          for (int n = 7; n >= 0; --n)
            if (((const unsigned*)s_row[sp][g * 8 + n])[h] & bit) r = n;
          top[sp] = k0 + g * 8 + r;
        }
      }
    }
    __syncthreads();
  }
  bool wet[2] = {false, false};
  unsigned before[2] = {0, 0};
  if (lists) {
    // (past the last column the words may hold anything)
    const bool col = i < p.ncol;
    wet[SED_LIQ] = col && (top[0] < nlev || top[1] < nlev);
    wet[SED_ICE] = col && top[2] < nlev;
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const unsigned long long m = __ballot(wet[g]);
      before[g] = (unsigned)__popcll(m & ((1ull << lane) - 1));
      if (lane == 0) s_n[g][wave] = __popcll(m);
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const int left = p.ncol - blk * kOrderCols;
    unsigned long long n = (unsigned long long)(left < kOrderCols ? left : kOrderCols);
    for (int v = 0; v < kWords; ++v)
      n += (unsigned long long)s_n[SED_LIQ][v] << 21 | (unsigned long long)s_n[SED_ICE][v] << 42;
    s_at = atomicAdd(p.order_count(), n);
  }
  __syncthreads();
  if (lists && i < p.ncol) {
    const unsigned mask = (1u << 21) - 1;
    const unsigned cols = (unsigned)s_at & mask;  // columns of the blocks before
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const unsigned base = (unsigned)(s_at >> 21 * (g + 1)) & mask;  // of them wet
      for (int v = 0; v < wave; ++v) before[g] += (unsigned)s_n[g][v];
      const unsigned at =
          wet[g] ? base + before[g] : (unsigned)p.ncol - 1 - (cols - base + threadIdx.x - before[g]);
      p.order(g)[at] = make_uint2((unsigned)i, g == SED_ICE ? (unsigned)top[2] : (unsigned)(top[0] | top[1] << 16));
    }
  }
}

template <class R>
__global__ __launch_bounds__(kOrderThreads) void p3_order_kernel(const KParams p) {
  order_block(p, blockIdx.x);
}

// Zeroes the column status words before p3_front_kernel (templated only so
// that each precision's translation unit has its own copy).
template <class R>
__global__ __launch_bounds__(256) void p3_colstat_clear_kernel(int* colstat, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) colstat[i] = 0;
}

// Parts 1 and 2 on the pointwise tiles; s_lds holds kSlots<R> * kTileThreads doubles.
template <class R>
__device__ __forceinline__ void front_tile(const KParams& p, int tile, double* s_lds) {
  int i, k;
  if (!pw_point<PW_BLOCKS>(p, tile, i, k)) return;
  unsigned err = 0;
  int stat = 0;
  front_level<R>(p, k, i, Pt{s_lds + threadIdx.x}, stat, err);
  if (p.track()) {
    colstat_or(p, i, (stat & kStatusPart1) != 0, kStatusPart1);
    colstat_or(p, i, (stat & kStatusPart2) != 0, kStatusPart2);
    if (k == 0 && p.dbg_check) p.dbg_check[i] = 0;  // part 3 ORs the column's check_values flags
  }
  if (p.ordered()) {
#pragma unroll
    for (int sp = 0; sp < 3; ++sp) put_wet(p, sp, i, k, __ballot((stat & kWet << sp) != 0));
    if (tile == 0 && threadIdx.x == 0) *p.order_count() = 0;
  }
  if (err) report_errors(p.err, err);
}

// Wavefronts per SIMD the front kernel is compiled for.  Two in FP64 (246
// VGPRs; at three it spilled 89 of them: 276 against 225 us at 21600 x 72), three
// in the mixed form (164 VGPRs).  A block of four wavefronts holds 52 KB of LDS slots
// in the mixed form, of which three blocks fit a CU, and 56 KB in FP64, of which two.
template <class R> constexpr int kFrontWaves = sizeof(R) == 8 ? 2 : 3;

template <class R>
__global__ __launch_bounds__(kTileThreads, kFrontWaves<R>) void p3_front_kernel(const KParams p) {
  __shared__ double s_lds[kSlots<R> * kTileThreads];
  front_tile<R>(p, blockIdx.x, s_lds);
}

}  // namespace p3d
